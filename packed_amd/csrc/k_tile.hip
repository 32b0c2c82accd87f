// k_tile.hip -- one-pass transforms of 2^15 and 2^16 FP32 points (tile_kernels.hpp).
#include "dispatch.hpp"

namespace pcxd {

void launch_tile(int lg, const TileArgs& a, int64_t grid, hipStream_t st) {
    const dim3 g((unsigned)std::min<int64_t>(a.a.nrows, grid));
    if (lg == 15)
        hipLaunchKernelGGL(k_tile<2>, g, dim3(kTileThreads), 0, st, a);
    else
        hipLaunchKernelGGL(k_tile<4>, g, dim3(kTileThreads), 0, st, a);
}
void launch_tile_twiddles(float2* t, int lg, hipStream_t st) {
    hipLaunchKernelGGL(k_tile_twiddles, dim3((tile_table((1 << lg) / kTilePoints) + 255) / 256), dim3(256), 0, st, t, lg);
}

} // namespace pcxd
