// k_shapes_small.hip -- four-step shapes with small tiles, for calls of few points.
//
// The default shapes' tiles of 16384 points (FP64: 8192) fill a CU each and stream large batches
// through wide segments, but a call of 2^20 points has 64 of them for 256 CUs, and one of 2^24
// points runs in rounds of one workgroup per CU with nothing to overlap its loads and stores.
// Tiles of 2048 to 8192 points (128 to 512 threads) spread the first over the chip and put
// several workgroups on a CU for the second.  Each limit is the largest call, in points over all
// transforms, at which the shape is faster in both directions (pack 8, forward / inverse, us,
// default shape -> this one; sweeps at 2^16 .. 2^26 points):
#include "shapes.hpp"

namespace pcxd {
namespace {
constexpr SmallShapeT<float> kSmall[] = {
    {24, shape<15, 8, 7, 16, 32>()},  // one transform 16.9 / 17.0 -> 10.8 / 10.4; 2^24 points 119 / 125 -> 91 / 101
    {26, shape<16, 9, 7, 8, 32>()},   // 18.9 / 16.8 -> 11.6 / 11.3; 2^24 126 / 127 -> 97 / 106; 2^26 440 / 466 -> 437 / 423
    {24, shape<17, 9, 8, 8, 16>()},   // 2^20 20.8 / 19.3 -> 14.0 / 14.9; 2^24 129 / 127 -> 103 / 110
    {26, shape<17, 9, 8, 16, 32>()},  // 2^26 468 / 470 -> 421 / 420
    {20, shape<18, 9, 9, 8, 8>()},    // one 21.9 / 19.9 -> 13.9 / 14.1
    {26, shape<18, 9, 9, 16, 16>()},  // 2^24 136 / 134 -> 111 / 113; 2^26 507 / 498 -> 458 / 432
    {21, shape<19, 9, 10, 16, 8>()},  // one 34 / 32 -> 18.3 / 18.1; 2^21 40 / 39 -> 27.6 / 26.7
    {22, shape<19, 9, 10, 8, 16>()},  // 2^22 46 / 44 -> 35 / 39
    {21, shape<20, 10, 10, 8, 8>()},  // one 27.9 / 27.5 -> 23.4 / 23.1; 2^21 35 / 35 -> 33 / 31
    {22, shape<20, 10, 10, 16, 16>()}, // up to one tile per CU: 3 39 / 41, 4 42 / 45 with the default's columns
    // the permuted orders' split at 2^20 (bit_reversed): one 25.8 / 26.7 -> 19.8 / 20.4;
    // 2^24 135 / 141 -> 111 / 117; 2^26 496 / 524 -> 485 / 484
    {26, shape<20, 12, 8, 1, 16>()},
};
constexpr SmallShapeT<double> kSmall64[] = {
    {24, shape64<14, 7, 7, 16, 16>()},  // one 14.5 / 15.2 -> 10.1 / 10.4; 2^24 225 / 233 -> 208 / 215
    {20, shape64<15, 8, 7, 8, 16>()},   // one 17.2 / 17.5 -> 10.9 / 11.0
    {24, shape64<15, 8, 7, 16, 32>()},  // 2^24 255 / 256 -> 212 / 219
    {17, shape64<16, 8, 8, 8, 8>()},    // one 17.7 / 18.3 -> 11.7 / 11.7
    {24, shape64<16, 8, 8, 16, 16>()},  // 2^24 263 / 261 -> 218 / 221
    {18, shape64<18, 9, 9, 4, 4>()},    // one 18.1 / 18.2 (the default's 8, 8) -> 15.9 / 16.5
    {22, shape64<19, 10, 9, 4, 8>()},   // one 28.7 / 28.1 -> 22.1 / 22.2; 2^22 71 / 70 -> 61 / 60
    {22, shape64<20, 10, 10, 4, 4>()},  // one 37 / 37 -> 33 / 33; 2^22 77 / 75 -> 65 / 64
};
} // namespace
SmallList<float>  shapes_small() { return {kSmall, (int)(sizeof(kSmall) / sizeof(kSmall[0]))}; }
SmallList<double> shapes64_small() { return {kSmall64, (int)(sizeof(kSmall64) / sizeof(kSmall64[0]))}; }
} // namespace pcxd
