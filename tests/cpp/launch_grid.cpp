// launch_grid.cpp -- host check of ox_xcd.hpp: every tile of a launch is taken by
// one workgroup, and no launch has 2^32 or more work items in a dimension.
// Build: g++ -std=c++17 -O2 -I/opt/rocm/include -D__HIP_PLATFORM_AMD__ -x c++ launch_grid.cpp
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

static uint3 blockIdx;
static dim3 gridDim;
#include "../../ouxsbli_amd/csrc/ox_xcd.hpp"

int main() {
  // lengths: around the chunk, the few-workgroup line and the fold, and the longest
  const long long row = ox::LAUNCH_ROW;
  for (long long n : {1LL, 7LL, 8LL, 9LL, 255LL, 256LL, 257LL, 2047LL, 2048LL, 2049LL, 2303LL, 100003LL, row - 1, row, row + 1,
                      2 * row + 5, (1LL << 24) + 1, 19173961LL, (1LL << 31) - 1}) {
    gridDim = ox::launch_grid(n);
    if ((unsigned long long)gridDim.x * 512 >= 1ull << 32 || gridDim.y > 65535 || gridDim.z != 1) {
      std::printf("launch of %lld: %u x %u\n", n, gridDim.x, gridDim.y);
      return 1;
    }
    for (int few = 0; few < 2; ++few) {
      std::vector<bool> taken(n, false);
      long long count = 0;
      for (unsigned y = 0; y < gridDim.y; ++y)
        for (unsigned x = 0; x < gridDim.x; ++x) {
          blockIdx.x = x;
          blockIdx.y = y;
          const unsigned b = ox::launch_block();
          if (b >= (unsigned)n) continue;
          const int t = ox::xcd_tile((int)b, (int)n, few);
          if (t < 0 || t >= n || taken[t]) {
            std::printf("launch of %lld, few %d: workgroup %u takes tile %d\n", n, few, b, t);
            return 1;
          }
          taken[t] = true;
          ++count;
        }
      if (count != n) {
        std::printf("launch of %lld: %lld tiles taken\n", n, count);
        return 1;
      }
      if (n > (1LL << 26)) break;  // the longest once
    }
  }
  std::printf("launch grids ok\n");
  return 0;
}
