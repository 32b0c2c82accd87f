// k_tile.hip -- one-pass transforms of 2^15 and 2^16 FP32 points (tile_kernels.hpp).
#include "dispatch.hpp"

namespace pcxd {

void launch_tile(int lg, const TileArgs& a, int64_t grid, hipStream_t st) {
    const dim3 g((unsigned)std::min<int64_t>(a.a.nrows, grid));
    const bool one = a.a.src_lp == 0 && a.a.dst_lp == 0;
    const auto f   = lg == 15 ? (one ? k_tile<2, true> : k_tile<2, false>) : (one ? k_tile<4, true> : k_tile<4, false>);
    hipLaunchKernelGGL(f, g, dim3(kTileThreads), 0, st, a);
}

} // namespace pcxd
