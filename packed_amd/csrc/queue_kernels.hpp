// queue_kernels.hpp -- work items of the persistent queue kernels for batches of uneven transform
// sizes: k_queue (k_misc.hip), transforms of 2^1 .. 2^14 points, and k_mixed (k_mixed.hip), of
// 2^1 .. 2^18.
//
// k_queue: an item is up to 512 / (2^la / 16) transforms of one size and one direction, run by the
// single-pass Stockham path of k_row.  Items hold 8192 points (2^14: 16384), so the workgroups stride
// through the list, largest size first, with no counter to share; two 512-thread workgroups fit a
// CU.  Larger transforms run as full-chip launches per size and direction: one workgroup that takes a
// 2^19 transform through an intermediate of its own holds it for about a millisecond while the others
// run out of work (us that way / with per-size launches: 2000 transforms of 2^6 .. 2^20 2458 / 2410,
// 998 of 2^4 .. 2^18 425 / 352, 63 of 2^8 .. 2^18 278 / 114; 558 of 2^5 .. 2^12, no large ones, with one
// 1024-thread workgroup per CU and a shared counter / these 23.3 / 12.2).
//
// k_mixed: where several classes of 2^15 .. 2^18 meet, none of them large enough to fill the chip
// for long, launches per class each end with a partly empty chip and start on cold data, while
// workgroups that each take whole transforms keep it full: 1400 transforms of 2^7 .. 2^16 176 us by
// launches per class and 144 in this one, 1000 of 2^10 .. 2^17 300 / 252, 1000 of 2^12 .. 2^18
// 651 / 565.  Items are sorted largest first; a 1024-thread workgroup per CU takes the next one from a
// device counter until it passes the end.  An item is up to 1024 / (2^la / 16) single-pass transforms,
// or one four-step transform, through an intermediate of the workgroup's own.
// Transforms are addressed through per-transform offset tables in split re/im layout (pack = N).
#pragma once
#include "fft_kernels.hpp"

namespace pcxk {

constexpr int kQueueThreads = 512;
constexpr int kQueueMaxLog2 = 14; // the persistent launch serves 2^1 .. 2^14

struct QItem {
    int32_t la;    // log2 of the transform size
    int32_t inv;   // inverse (conj in / conj out)
    int32_t first; // index of the first transform in the offset tables
    int32_t count; // transforms in the item
};

struct QueueArgs {
    const float*   src;
    float*         dst;
    const int64_t* src_offs;   // per transform, in item order
    const int64_t* dst_offs;
    const QItem*   items;
    int32_t        nitems;
    int32_t        normalized;
    const float2*  tw;         // W_A tables for A = 2, 4, ..., 2^14 back to back (table A at A - 2)
};

constexpr int kMixThreads = 1024;
constexpr int kMixMaxLog2 = 18; // (2^19 and larger transforms always run as full-chip launches)

struct MixArgs {
    QueueArgs     q;
    float*        tmp;        // four-step intermediates, tmp_floats per workgroup
    int64_t       tmp_floats;
    uint32_t*     counter;    // zeroed before every launch
    const float2* ptw;        // pass tables W_N of N = 2^15 .. 2^18: lo (2^ls entries) then hi
    int32_t       ptw_off[kMixMaxLog2 + 1]; // entry offset of N = 2^lg's tables in ptw
};

// Points per thread of an item's single-pass transforms: 16 (k_queue: 32 for 2^14, one transform per
// item), or the whole transform below 16 points.
constexpr int q_ppt(int la, int threads) { return la >= 14 && threads == kQueueThreads ? 32 : (la >= 4 ? 16 : 0); }
// The four-step split of k_mixed: rows of 2^q_n1(lg) points, columns of the rest; 1024-thread tiles of
// 16384 points (C = 16384 / N2 columns, G = 16384 / N1 rows).
constexpr int q_n1(int lg) { return lg == 15 ? 8 : 9; }

} // namespace pcxk
