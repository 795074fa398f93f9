// The matrix-core kernels at head dims 64 and 256: instantiation and dispatch
// for one 16-bit KV element type.  Each including file defines HELM_TKV (the
// element type), HELM_DIM (the head dim) and HELM_LAUNCH_NAME, so that the
// instantiations compile in parallel per type and head dim.
#pragma once

#include "attn_kernel.h"
#include "attn_mfma.h"
#include "attn_chunk32.h"
#include "attn_launch.h"

namespace helm {
namespace {

template <typename T, class Src, int FEAT, int D>
hipError_t launch_dim_feat(const LaunchSpec& s, const Src& src, hipStream_t st) {
  if (s.p.row_waves && s.nw == 4)
    HELM_ATTN_LAUNCH((chunk32_mfma_dim_kernel<T, Src, FEAT, 4, D>), s.grid, dim3(256), s.p, src);
  else if (!s.p.row_waves && s.nw == 4)
    HELM_ATTN_LAUNCH((decode_mfma_dim_kernel<T, Src, FEAT, D>), s.grid, dim3(256), s.p, src);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <typename T, class Src, int D>
hipError_t launch_dim_src(const LaunchSpec& s, const Src& src, hipStream_t st) {
  switch (s.feat) {
    case 0: return launch_dim_feat<T, Src, 0, D>(s, src, st);
    case 1: return launch_dim_feat<T, Src, 1, D>(s, src, st);
    case 2: return launch_dim_feat<T, Src, 2, D>(s, src, st);
    case 3: return launch_dim_feat<T, Src, 3, D>(s, src, st);
    case 4: return launch_dim_feat<T, Src, 4, D>(s, src, st);
    case 5: return launch_dim_feat<T, Src, 5, D>(s, src, st);
    case 6: return launch_dim_feat<T, Src, 6, D>(s, src, st);
    case 7: return launch_dim_feat<T, Src, 7, D>(s, src, st);
    case 9: return launch_dim_feat<T, Src, 9, D>(s, src, st);
    case 11: return launch_dim_feat<T, Src, 11, D>(s, src, st);
    case 13: return launch_dim_feat<T, Src, 13, D>(s, src, st);
    case 15: return launch_dim_feat<T, Src, 15, D>(s, src, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t HELM_LAUNCH_NAME(const LaunchSpec& s, hipStream_t st) {
  if (s.mode == 0) return launch_dim_src<HELM_TKV, PoolSrc, HELM_DIM>(s, s.pool, st);
  return launch_dim_src<HELM_TKV, DescSrc, HELM_DIM>(s, s.desc, st);
}

}  // namespace helm
