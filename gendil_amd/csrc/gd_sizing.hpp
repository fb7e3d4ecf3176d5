// Elements per block where a mesh is too small to fill every CU with full blocks.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace gd {

constexpr int kCus = 256;
constexpr size_t kLdsPerCu = 160 * 1024;

// Blocks of `threads` threads that the kernel's registers let a CU hold.
template <typename Kernel>
int blocks_per_cu(Kernel kern, int threads)
{
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(kern), threads, 0) != hipSuccess)
    (void)hipGetLastError();
  return std::max(n, 1);
}

// Elements per block, up to `most`: halved, down to `least`, until there are two
// blocks for every CU; then, if these are more blocks than are resident at once
// (`per` bytes of LDS an element), the next number with which all are: a second
// round of blocks costs a small mesh as much as the first (FP64 plane advection,
// n = 5, q = 6, 1,728 elements: 576 blocks of 3 on 512 slots 42 us, 432 of 4
// 21 us).  Fewer elements than that where more blocks would fit is no gain
// (n = q = 2, 4,096 elements: 8.2 us with 8, 9.9 with 4).
inline int elements_per_block(int64_t E, int least, int most, size_t per, int resident)
{
  int epb = most;
  while (epb > least && (int64_t)epb * 2 * kCus > E) epb = (epb + 1) / 2;
  for (int n = epb; n < most; ++n) {
    const int64_t slots = (int64_t)kCus * std::min<int64_t>(resident, (int64_t)(kLdsPerCu / (n * per)));
    if ((E + n - 1) / n <= slots) return n;
  }
  return most;
}

}  // namespace gd
