// Kernel launches of the numeric phase (device translation units).
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "gdx_internal.h"

// Launch of a numeric phase's kernel.  The phase's events ride on the kernels'
// own packets: an event record of its own costs a barrier and a cache flush,
// about 5 us of the stream each.
#define GDX_LAUNCH(p, kernel, grid, block, st, ...)                                                              \
  do {                                                                                                           \
    if ((p)->launch_ev[0] || (p)->launch_ev[1])                                                                  \
      hipExtLaunchKernelGGL(kernel, grid, block, 0, st, (p)->launch_ev[0], (p)->launch_ev[1], 0, __VA_ARGS__);   \
    else                                                                                                         \
      hipLaunchKernelGGL(kernel, grid, block, 0, st, __VA_ARGS__);                                               \
  } while (0)
