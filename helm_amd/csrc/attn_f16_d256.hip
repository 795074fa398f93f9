// Matrix-core attention kernels with f16 KV pages of head dim 256.
#define HELM_TKV helm::f16_t
#define HELM_DIM 256
#define HELM_LAUNCH_NAME launch_attn_f16_d256
#include "attn_dim.h"
