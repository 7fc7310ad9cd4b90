// ox_xcd.hpp -- which tile a workgroup takes: launches of any length, and the deal
// over the XCDs.
#pragma once

#include <hip/hip_runtime.h>

namespace ox {

// The grid of a launch of n workgroups of up to 512 lanes, and a workgroup's number
// in it (not below n in the last row: nothing to do).  HIP refuses 2^32 or more work
// items in one dimension, which the tiles of thin grids and of long batches reach
// (8 x 2^27 points in 2-D: 19 million tiles), so longer launches are folded.
constexpr int LAUNCH_ROW = 1 << 22;
__host__ inline dim3 launch_grid(long long n) {
  return n <= LAUNCH_ROW ? dim3((unsigned)n) : dim3(LAUNCH_ROW, (unsigned)((n + LAUNCH_ROW - 1) / LAUNCH_ROW));
}
__device__ __forceinline__ unsigned launch_block() { return blockIdx.x + gridDim.x * blockIdx.y; }

// Workgroups are dispatched round-robin over the eight XCDs, and each XCD has
// its own L2.  Of every 8 * XCD_CHUNK workgroups, those of one XCD take XCD_CHUNK
// tiles that follow one another, so the tiles whose stencils overlap (neighbours
// along the second and third launch dimensions) share an L2 instead of fetching
// the same rows into two, while all XCDs work in one part of the grid and find
// in the shared cache what the others fetched.  (One run of n / 8 tiles per XCD,
// for n a multiple of 8 only, was up to 10% slower, us: Hybrid6 LES 192^3 x 405
// -> 378, y 533 -> 479, z 674 -> 638; SLAU6 NS 256^3 x 735 -> 702, y 778 -> 732, but
// z 1042 -> 1065; FP32 SLAU6 Euler 256^3 x 296 -> 270; FP32 Roe4 NS 190 x 187 x 181,
// undivided before, y 145 -> 137, z 271 -> 253; six FP32 requests 138.9 -> 133.9 ms; over
// the 256^3 Taylor-Green runs the step is the same within 0.6%.
// Chunks of 16 are equal, of 8 and 64 a little slower.  The price is traffic beyond
// L2: the x sweep's neighbours in z always come from another XCD's chunk.)  `few`: a
// launch of up to 2048 workgroups is one run per XCD instead.  The 2-D stage needs it
// (450 x 240, FP64: chunks 20.1 us, one run 14.1).  The line sweeps of a lone case
// take it too, where the two differ by 5% at most, either way: FP32 SLAU6 Euler 96^3 y
// with 864 workgroups chunks 22.9 us, one run 20.6; FP64 SLAU6 NS 160^3 z with 2400
// chunks 309 us, one run 319, and with 1200 296 and 306.  The x sweep and batches
// are faster in chunks (FP32 SLAU6 Euler 64^3 x 11.4 -> 10.4; the six requests 136.3
// -> 133.9 ms).  The map is a permutation of [0, n).
constexpr int XCD_CHUNK = 32;
__device__ __forceinline__ int xcd_tile(int b, int n, bool few = false) {
  int base = 0, m = n;
  if (!few || n > 2048) {
    base = b / (8 * XCD_CHUNK) * (8 * XCD_CHUNK);
    m = n - base < 8 * XCD_CHUNK ? n - base : 8 * XCD_CHUNK;
  }
  const int c = b - base, x = c & 7, r = m & 7;
  return base + x * (m >> 3) + (x < r ? x : r) + (c >> 3);
}

}  // namespace ox
