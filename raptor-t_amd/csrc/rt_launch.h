// Kernel launch of the library's device code: an ordinary launch, or, when the calling thread has left a pair
// of events with rt_time_next_launch, a launch that writes the dispatch's own start and end timestamps into
// them (what a profiler reports as the kernel's duration; a pair of hipEventRecord calls around a launch also
// counts the gaps to the neighbouring kernels, several microseconds on this part).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "rt_common.h"

namespace rt {
// Cache policy of stores whose data the next kernel reads: on to memory at once (SC1), the line stays in the L2.  Each XCD has an
// L2 of its own, so a kernel that leaves dirty lines behind ends with writing them back, while nothing else runs; written
// through they are on their way while the kernel works.  What that saves grows with the share of a launch that its end
// has, so it is nothing for launches of many rounds (those of the large products are non-temporal, which is the
// same to them: 16 x 512-4096 tokens 7.95 ms with either).  Encoder of 12 layers, operands in rotation (us, plain stores / 16-bit
// products and their fp32 slices written through / K and V^T tiles too / attention / LayerNorms):
//   1 x 512       589 / 583 / 583 / 581 / 579        4 x 256-1024   1135 / 1104 / 1095 / 1090 / 1087
//   1 x 4096     1445 / 1437 / 1432 / 1424 / 1418     the model on a padded batch of 8 x 150-1700   2020 / 1974 / 1974 / 1957 / 1930
// Non-temporal stores make the same products 10-20 % faster by themselves (512 x 3072 x 768 + GELU 8.8 -> 7.0) but the kernels
// behind them slower: 1 x 512 586, 4 x 256-1024 1089, with K and V^T tiles 598 and 1120.
constexpr int WRITE_THROUGH = 16;
}  // namespace rt

#define RT_LAUNCH(kernel, grid, block, shmem, stream, ...)                                              \
  do {                                                                                                  \
    const rt::LaunchEvents rt_ev_ = rt::take_launch_events();                                           \
    if (rt_ev_.start || rt_ev_.stop)                                                                    \
      hipExtLaunchKernelGGL(kernel, grid, block, shmem, stream, static_cast<hipEvent_t>(rt_ev_.start),  \
                            static_cast<hipEvent_t>(rt_ev_.stop), 0, __VA_ARGS__);                      \
    else                                                                                                \
      hipLaunchKernelGGL(kernel, grid, block, shmem, stream, __VA_ARGS__);                              \
  } while (0)
