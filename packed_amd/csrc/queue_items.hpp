// queue_items.hpp -- device functions of the queue kernels' work items.
#pragma once
#include "queue_kernels.hpp"

namespace pcxk {

// LDS of a single-pass item, and of the largest up to 2^14 (floats)
template<int LA, int NT>
constexpr int queue_single_lds() {
    constexpr int PX = q_ppt(LA, NT);
    constexpr int G  = NT / Plan<LA, false, float, PX>::TA;
    return RowShape<LA, G, float, PX>::DATA + TwTable<LA>::FLOATS;
}
template<int NT, int... L>
constexpr int queue_single_max(std::integer_sequence<int, L...>) {
    int m = 0;
    ((m = m > queue_single_lds<L + 1, NT>() ? m : queue_single_lds<L + 1, NT>()), ...);
    return m;
}
template<int NT>
constexpr int kQueueSingleLds = queue_single_max<NT>(std::make_integer_sequence<int, kQueueMaxLog2>{});

// A queue kernel's LDS, at file scope: the item functions are compiled separately (each with its own
// register budget) and address it directly as LDS.
template<int FLOATS>
static __shared__ float q_lds[FLOATS];

// Values an item function receives arrive in VGPRs (function arguments); these make the
// workgroup-uniform ones scalar again, so addresses and loop bounds stay in SGPRs.
__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni(int64_t v) {
    const uint64_t u  = (uint64_t)v;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
template<class T>
__device__ __forceinline__ T* uni(T* p) {
    return reinterpret_cast<T*>(uni((int64_t)reinterpret_cast<uintptr_t>(p)));
}
__device__ __forceinline__ QItem uni(const QItem& it) { return {uni(it.la), uni(it.inv), uni(it.first), uni(it.count)}; }

// ---- single-pass item: `count` transforms of 2^LA points, one row of the workgroup each
template<int LA, int NT, int LDS>
__device__ __noinline__ void queue_single(const QueueArgs& q, const QItem it_) {
    float*      lds = q_lds<LDS>;
    const QItem it  = uni(it_);
    constexpr int PX = q_ppt(LA, NT);
    constexpr int TA = Plan<LA, false, float, PX>::TA;
    constexpr int G  = NT / TA;
    static_assert(G * TA == NT, "single-pass items fill the workgroup");
    using S = RowShape<LA, G, float, PX>;
    RowArgs p{};
    p.src      = uni(q.src);
    p.dst      = uni(q.dst);
    p.src_offs = uni(q.src_offs) + it.first;
    p.dst_offs = uni(q.dst_offs) + it.first;
    p.src_size = (int64_t)1 << LA;
    p.nrows    = it.count;
    p.src_lp = p.dst_lp = LA;
    p.rows_lg           = 0;
    p.order             = 0;
    p.conj_in = p.conj_out = it.inv;
    p.scale                = (it.inv && uni(q.normalized)) ? 1.0f / (float)(1 << LA) : 1.0f;
    p.twA                  = uni(q.tw) + ((1 << LA) - 2);
    using LC               = LdsCarve<float, S::DATA, TwTable<LA>::FLOATS, 0>;
    float* ltw             = lds + LC::TOFF;
    float* lre             = lds + LC::DOFF;
    TwTable<LA>::fill(ltw, p.twA, threadIdx.x, NT);
    __syncthreads();
    row_group<LA, G, LD_CONTIG, ST_CONTIG, 0, (TA >= 64), 0, PREC_FP32, float, PX>(p, 0, lre, S::im(lre), ltw, nullptr);
}

// The single-pass item of size 2^la.
template<int NT, int LDS>
__device__ __forceinline__ void queue_single_any(const QueueArgs& q, const QItem w) {
    switch (w.la) {
    case 1: queue_single<1, NT, LDS>(q, w); break;
    case 2: queue_single<2, NT, LDS>(q, w); break;
    case 3: queue_single<3, NT, LDS>(q, w); break;
    case 4: queue_single<4, NT, LDS>(q, w); break;
    case 5: queue_single<5, NT, LDS>(q, w); break;
    case 6: queue_single<6, NT, LDS>(q, w); break;
    case 7: queue_single<7, NT, LDS>(q, w); break;
    case 8: queue_single<8, NT, LDS>(q, w); break;
    case 9: queue_single<9, NT, LDS>(q, w); break;
    case 10: queue_single<10, NT, LDS>(q, w); break;
    case 11: queue_single<11, NT, LDS>(q, w); break;
    case 12: queue_single<12, NT, LDS>(q, w); break;
    case 13: queue_single<13, NT, LDS>(q, w); break;
    case 14: queue_single<14, NT, LDS>(q, w); break;
    default: break;
    }
}

} // namespace pcxk
