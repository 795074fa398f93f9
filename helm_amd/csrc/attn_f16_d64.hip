// Matrix-core attention kernels with f16 KV pages of head dim 64.
#define HELM_TKV helm::f16_t
#define HELM_DIM 64
#define HELM_LAUNCH_NAME launch_attn_f16_d64
#include "attn_dim.h"
