// Matrix-core attention kernels with bf16 KV pages of head dim 256.
#define HELM_TKV helm::bf16_t
#define HELM_DIM 256
#define HELM_LAUNCH_NAME launch_attn_bf16_d256
#include "attn_dim.h"
