// k_mixed.hip -- the persistent queue kernel over mixed sizes (2^1 .. 2^18 points), whose workgroups
// each take whole transforms.
#include "dispatch.hpp"
#include "queue_items.hpp"

#include <algorithm>

namespace pcxk {

template<int LG>
constexpr int queue_four_lds() {
    constexpr int N1L = q_n1(LG), N2L = LG - N1L, C = 16384 >> N2L, G = 16384 >> N1L;
    constexpr int cl  = 2 * (1 << N2L) * C + TwTable<N2L>::FLOATS + 2 * pass_tw_entries(LG);
    constexpr int rl  = RowShape<N1L, G>::DATA + TwTable<N1L>::FLOATS + 2 * pass_tw_entries(LG);
    return cl > rl ? cl : rl;
}
template<int... L>
constexpr int queue_four_max(std::integer_sequence<int, L...>) {
    int m = 0;
    ((m = m > queue_four_lds<L + kQueueMaxLog2 + 1>() ? m : queue_four_lds<L + kQueueMaxLog2 + 1>()), ...);
    return m;
}
constexpr int kMixLds = std::max(kQueueSingleLds<kMixThreads>,
                                 queue_four_max(std::make_integer_sequence<int, kMixMaxLog2 - kQueueMaxLog2>{}));
static_assert(4 * kMixLds <= 160 * 1024, "the largest item fits one CU's LDS");

// ---- four-step item: one transform of 2^LG points through this workgroup's intermediate.  Each
// pass is its own function (its own register budget); the workgroup runs the first pass over all
// tiles, then the second: the intermediate it wrote is read back by the same workgroup.
template<int LG>
struct QFour {
    static constexpr int N1L = q_n1(LG), N2L = LG - N1L;
    static constexpr int C   = 16384 >> N2L; // columns per column tile
    static constexpr int G   = 16384 >> N1L; // rows per row group
    static constexpr int TW  = pass_tw_entries(LG);
    static_assert(C * Plan<N2L>::TA == kMixThreads && G * Plan<N1L>::TA == kMixThreads, "four-step tiles");
    static_assert(TW <= 2048, "pass twiddles in LDS");
    static constexpr int64_t N = (int64_t)1 << LG;
    static constexpr int     LS = (LG + 1) / 2;
};

// column pass: forward pass A (src -> intermediate, times the pass twiddle) or inverse pass 2
// (intermediate -> dst, conj and the 1/N scale at the store)
template<int LG, bool INV>
__device__ __noinline__ void queue_cols(const MixArgs& m, const QItem it_) {
    using F              = QFour<LG>;
    constexpr int CT     = INV ? 0 : F::TW;
    float*        lds    = q_lds<kMixLds>;
    const QItem   it     = uni(it_);
    float*        tmp    = uni(m.tmp) + (int64_t)blockIdx.x * uni(m.tmp_floats);
    const float2* twl    = uni(m.ptw) + uni(m.ptw_off[LG]);
    ColArgs       ca{};
    ca.twA = uni(m.q.tw) + ((1 << F::N2L) - 2), ca.n1_lg = F::N1L, ca.ntiles = (1 << F::N1L) / F::C, ca.tw_lg = LG;
    ca.src_size = F::N, ca.src_lp = ca.dst_lp = LG; // split vectors and intermediate (pack = N)
    if constexpr (!INV) {
        ca.src = uni(m.q.src) + uni(uni(m.q.src_offs)[it.first]), ca.dst = tmp, ca.scale = 1.0f;
        ca.twl = twl, ca.twh = twl + (1 << F::LS), ca.tw_ls = F::LS;
    } else {
        ca.src = tmp, ca.dst = uni(m.q.dst) + uni(uni(m.q.dst_offs)[it.first]), ca.conj_out = 1;
        ca.scale = uni(m.q.normalized) ? (float)(1.0 / (double)F::N) : 1.0f;
    }
    using LC    = LdsCarve<float, 2 * (1 << F::N2L) * F::C, TwTable<F::N2L>::FLOATS, 2 * CT>;
    float* ltw  = lds + LC::TOFF;
    float* lptw = ltw + TwTable<F::N2L>::FLOATS;
    float* lre  = lds + LC::DOFF;
    float* lim  = lre + (1 << F::N2L) * F::C;
    TwTable<F::N2L>::fill(ltw, ca.twA, threadIdx.x, kMixThreads);
    if constexpr (CT > 0)
        PassTw<CT>::fill(lptw, ca.twl, ca.twh, ca.tw_ls, ca.tw_lg, threadIdx.x, kMixThreads);
    __syncthreads();
    for (int64_t tile = 0; tile < ca.ntiles; ++tile) {
        col_tile<F::N2L, F::C, CT>(ca, tile, lre, lim, ltw, lptw);
        __syncthreads(); // LDS is reused by the next tile
    }
}

// row pass: forward pass B (intermediate -> dst, strided store in natural order) or inverse pass
// 1 (src -> intermediate, strided load, times the pass twiddle)
template<int LG, bool INV>
__device__ __noinline__ void queue_rows(const MixArgs& m, const QItem it_) {
    using F            = QFour<LG>;
    constexpr int RT   = INV ? F::TW : 0;
    using S            = RowShape<F::N1L, F::G>;
    float*        lds  = q_lds<kMixLds>;
    const QItem   it   = uni(it_);
    float*        tmp  = uni(m.tmp) + (int64_t)blockIdx.x * uni(m.tmp_floats);
    const float2* twl  = uni(m.ptw) + uni(m.ptw_off[LG]);
    RowArgs       ra{};
    ra.twA = uni(m.q.tw) + ((1 << F::N1L) - 2), ra.rows_lg = F::N2L, ra.nrows = 1 << F::N2L, ra.order = 0, ra.tw_lg = LG;
    ra.src_size = F::N, ra.src_lp = ra.dst_lp = LG, ra.scale = 1.0f;
    if constexpr (!INV) {
        ra.src = tmp, ra.dst = uni(m.q.dst) + uni(uni(m.q.dst_offs)[it.first]);
    } else {
        ra.src = uni(m.q.src) + uni(uni(m.q.src_offs)[it.first]), ra.dst = tmp, ra.conj_in = 1;
        ra.twl = twl, ra.twh = twl + (1 << F::LS), ra.tw_ls = F::LS;
    }
    using LC    = LdsCarve<float, S::DATA, TwTable<F::N1L>::FLOATS, 2 * RT>;
    float* ltw  = lds + LC::TOFF;
    float* lptw = ltw + TwTable<F::N1L>::FLOATS;
    float* lre  = lds + LC::DOFF;
    TwTable<F::N1L>::fill(ltw, ra.twA, threadIdx.x, kMixThreads);
    if constexpr (RT > 0)
        PassTw<RT>::fill(lptw, ra.twl, ra.twh, ra.tw_ls, ra.tw_lg, threadIdx.x, kMixThreads);
    __syncthreads();
    for (int64_t wg = 0; wg < ra.nrows / F::G; ++wg) {
        if constexpr (!INV)
            row_group<F::N1L, F::G, LD_CONTIG, ST_STRIDED, 0, true, 0>(ra, wg, lre, S::im(lre), ltw, lptw);
        else
            row_group<F::N1L, F::G, LD_STRIDED, ST_CONTIG, RT, true, 0>(ra, wg, lre, S::im(lre), ltw, lptw);
        __syncthreads(); // LDS is reused by the next group
    }
}

template<int LG>
__device__ __forceinline__ void queue_four(const MixArgs& m, const QItem it) {
    if (!it.inv) {
        queue_cols<LG, false>(m, it);
        queue_rows<LG, false>(m, it);
    } else {
        queue_rows<LG, true>(m, it);
        queue_cols<LG, true>(m, it);
    }
}

__global__ __launch_bounds__(kMixThreads) void k_mixed(MixArgs m) {
    __shared__ int s_item;
    for (;;) {
        if (threadIdx.x == 0)
            s_item = (int)atomicAdd(m.counter, 1u);
        __syncthreads();
        const int it = s_item;
        if (it >= m.q.nitems)
            break; // uniform: every wavefront leaves together once the queue is drained
        const QItem w = m.q.items[it];
        switch (w.la) {
        case 15: queue_four<15>(m, w); break;
        case 16: queue_four<16>(m, w); break;
        case 17: queue_four<17>(m, w); break;
        case 18: queue_four<18>(m, w); break;
        default: queue_single_any<kMixThreads, kMixLds>(m.q, w); break;
        }
        __syncthreads(); // LDS and s_item are reused by the next item
    }
}

__global__ void k_reset_counter(uint32_t* c) {
    if (threadIdx.x == 0 && blockIdx.x == 0)
        *c = 0u;
}

} // namespace pcxk

namespace pcxd {

void launch_mixed(const MixArgs& a, int grid, hipStream_t st) {
    hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(64), 0, st, a.counter);
    hipLaunchKernelGGL(k_mixed, dim3(grid), dim3(kMixThreads), 0, st, a);
}

} // namespace pcxd
