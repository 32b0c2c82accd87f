// queue_kernels.hpp -- work items of the persistent queue kernel for batches of uneven transform
// sizes (the kernel, k_queue, is in k_misc.hip).
//
// One launch serves every transform of 2^1 .. 2^14 points: an item is up to 512 / (2^la / 16)
// transforms of one size and one direction, run by the single-pass Stockham path of k_row.  Items
// hold 8192 points (2^14: 16384), so the workgroups stride through the list, largest size first,
// with no counter to share; two 512-thread workgroups fit a CU.  Larger transforms run as
// full-chip launches per size and direction: one workgroup that takes a 2^19 transform through an
// intermediate of its own holds it for about a millisecond while the others run out of work
// (us that way / with per-size launches: 2000 transforms of 2^6 .. 2^20 2458 / 2410, 998 of
// 2^4 .. 2^18 425 / 352, 63 of 2^8 .. 2^18 278 / 114; 558 of 2^5 .. 2^12, no large ones, with one
// 1024-thread workgroup per CU and a shared counter / these 23.3 / 12.2).
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

// Points per thread of an item's transforms: 16 (32 for 2^14, one transform per item), or the whole
// transform below 16 points.
constexpr int q_ppt(int la) { return la >= 14 ? 32 : (la >= 4 ? 16 : 0); }

} // namespace pcxk
