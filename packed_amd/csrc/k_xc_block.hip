// k_xc_block.hip -- block path of the overlap-save correlation, block sizes 2^15 .. 2^24.
#include "dispatch.hpp"

namespace pcxd {
namespace {
// Rows as long as one fused row kernel takes (2^14) and columns of 2^7 while that reaches.  Column
// tiles of 4096 points (256 threads, up to four workgroups per CU): with 2^7-point columns, 32 per
// tile beat 128 per tile (1024 threads, one workgroup per CU) at every number of blocks, first /
// last kernel at N = 2^17: 2 blocks 6.1 / 4.2 against 8.7 / 7.2 us, 33 blocks 15.6 / 12.6 against
// 21.1 / 18.1, 512 blocks 193 / 181 against 211 / 205.
template<int LG>
constexpr XcBlockSet xc_block_set() {
    constexpr int N2 = LG <= 21 ? 7 : LG - 14, N1 = LG - N2, C = 4096 >> N2, TW = tw_cap<LG>();
    return {LG, N1, N2, &launch_xc_col<N2, C, TW, false>, &launch_xc_rows<N1, TW>, &launch_xc_col<N2, C, 0, true>};
}
template<int... L>
constexpr auto xc_block_table(std::integer_sequence<int, L...>) {
    return std::array<XcBlockSet, sizeof...(L)>{xc_block_set<kMaxSinglePass + 1 + L>()...};
}
const std::array<XcBlockSet, kMaxLog2 - kMaxSinglePass> kXcBlock =
    xc_block_table(std::make_integer_sequence<int, kMaxLog2 - kMaxSinglePass>{});
} // namespace

const std::array<XcBlockSet, kMaxLog2 - kMaxSinglePass>& xc_block_tab() { return kXcBlock; }

} // namespace pcxd
