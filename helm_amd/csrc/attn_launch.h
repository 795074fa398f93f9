// The launch macro of the attention kernels' dispatch files.
#pragma once

#include <hip/hip_ext.h>

// A launch timed by helm_profile_split_kernels goes through
// hipExtLaunchKernelGGL with the spec's start / stop events, which then carry
// the kernel's own start and end; every other launch is a plain launch.
#define HELM_ATTN_LAUNCH(KERNEL, GRID, BLOCK, ...)                                       \
  do {                                                                                   \
    if (s.ev_start)                                                                      \
      hipExtLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, st, s.ev_start, s.ev_stop, 0,        \
                            __VA_ARGS__);                                                \
    else                                                                                 \
      hipLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, st, __VA_ARGS__);                       \
  } while (0)
