// k_misc.hip -- the persistent uneven-batch queue kernel (one launch for every transform of
// 2^1 .. 2^14 points) and the vector-expression kernel.
#include "dispatch.hpp"

#include <algorithm>

namespace pcxk {

// LDS of the largest item (floats)
template<int LA>
constexpr int queue_single_lds() {
    constexpr int PX = q_ppt(LA);
    constexpr int G  = kQueueThreads / Plan<LA, false, float, PX>::TA;
    return RowShape<LA, G, float, PX>::DATA + TwTable<LA>::FLOATS;
}
template<int... L>
constexpr int queue_single_max(std::integer_sequence<int, L...>) {
    int m = 0;
    ((m = m > queue_single_lds<L + 1>() ? m : queue_single_lds<L + 1>()), ...);
    return m;
}
constexpr int kQueueLds = queue_single_max(std::make_integer_sequence<int, kQueueMaxLog2>{});
static_assert(4 * kQueueLds <= 80 * 1024, "two workgroups fit one CU's LDS");

// The queue kernel's LDS, at file scope: the item functions are compiled separately (each with
// its own register budget) and address it directly as LDS.
__shared__ float g_qlds[kQueueLds];

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
template<int LA>
__device__ __noinline__ void queue_single(const QueueArgs& q, const QItem it_) {
    float*      lds = g_qlds;
    const QItem it  = uni(it_);
    constexpr int PX = q_ppt(LA);
    constexpr int TA = Plan<LA, false, float, PX>::TA;
    constexpr int G  = kQueueThreads / TA;
    static_assert(G * TA == kQueueThreads, "single-pass items fill the workgroup");
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
    TwTable<LA>::fill(ltw, p.twA, threadIdx.x, kQueueThreads);
    __syncthreads();
    row_group<LA, G, LD_CONTIG, ST_CONTIG, 0, (TA >= 64), 0, PREC_FP32, float, PX>(p, 0, lre, S::im(lre), ltw, nullptr);
}

__global__ __launch_bounds__(kQueueThreads, 4) void k_queue(QueueArgs q) {
    for (int it = (int)blockIdx.x; it < q.nitems; it += (int)gridDim.x) {
        const QItem w = q.items[it];
        switch (w.la) {
        case 1: queue_single<1>(q, w); break;
        case 2: queue_single<2>(q, w); break;
        case 3: queue_single<3>(q, w); break;
        case 4: queue_single<4>(q, w); break;
        case 5: queue_single<5>(q, w); break;
        case 6: queue_single<6>(q, w); break;
        case 7: queue_single<7>(q, w); break;
        case 8: queue_single<8>(q, w); break;
        case 9: queue_single<9>(q, w); break;
        case 10: queue_single<10>(q, w); break;
        case 11: queue_single<11>(q, w); break;
        case 12: queue_single<12>(q, w); break;
        case 13: queue_single<13>(q, w); break;
        case 14: queue_single<14>(q, w); break;
        default: break;
        }
        __syncthreads(); // LDS is reused by the next item
    }
}

} // namespace pcxk

namespace pcxd {

void launch_queue(const QueueArgs& a, int grid, hipStream_t st) {
    hipLaunchKernelGGL(k_queue, dim3(grid), dim3(kQueueThreads), 0, st, a);
}
namespace {
// The stack form of a program: LOAD pushes (d is the number of values on the stack), a unary
// operation works on the top (d = a = top), a binary one on the top two (d = the lower, a and b
// the two in either order), and one value is left.  A program that uses its registers in another
// way has none (false).  A source beyond the preloaded ones, and with `preload` 0 every source, is
// loaded by its own LOAD.
template<class T>
bool vexpr_stack(const VExprArgsT<T>& a, int preload, VStackArgsT<T>& s) {
    int depth = 0, slot[kVMaxSrc];
    std::fill(slot, slot + kVMaxSrc, -1);
    for (int k = 0; k < a.nprog; ++k) {
        const VInstrT<T>& in   = a.prog[k];
        int               code = in.op;
        if (in.op == VOP_LOAD) {
            if (in.d != depth++)
                return false;
            if (slot[in.a] < 0)
                slot[in.a] = s.nsrc, s.src[s.nsrc++] = a.src[in.a];
            code      = slot[in.a] < preload ? VST_LOAD0 + slot[in.a] : VST_LOADX;
            s.load[k] = slot[in.a];
        } else if (in.op >= VOP_ADD && in.op <= VOP_DIV) {
            const int lo = depth - 2;
            if (lo < 0 || in.d != lo || in.a + in.b != 2 * lo + 1 || (in.a != lo && in.b != lo))
                return false;
            if (in.a != lo)
                code = VST_XADD + (in.op - VOP_ADD);
            --depth;
        } else if (depth < 1 || in.d != depth - 1 || in.a != depth - 1) {
            return false;
        }
        s.code[k / kVPerWord] |= (uint64_t)code << (5 * (k % kVPerWord));
        s.scalar[k] = {in.s_re, in.s_im};
    }
    s.nprog = a.nprog, s.dst = a.dst, s.dst_lp = a.dst_lp, s.n = a.n;
    return depth == 1;
}

template<class T>
void launch_vexpr_t(const VExprArgsT<T>& a, hipStream_t st) {
    constexpr int V    = 16 / (int)sizeof(T);
    auto          grid = [](int64_t items) { return dim3((unsigned)std::min<int64_t>((items + 255) / 256, 16384)); };
    // 16-byte accesses need 16-byte aligned vectors (whole allocations and storage slices are; a
    // caller's pointer into one may not be)
    bool wide = (reinterpret_cast<uintptr_t>(a.dst) & 15) == 0;
    for (int k = 0; k < a.nprog; ++k)
        if (a.prog[k].op == VOP_LOAD)
            wide = wide && (reinterpret_cast<uintptr_t>(a.src[a.prog[k].a].data) & 15) == 0;
    VStackArgsT<T> s{};
    if (!vexpr_stack(a, wide ? kVPreload : 0, s)) {
        hipLaunchKernelGGL(k_vexpr<T>, grid(a.n), dim3(256), 0, st, a);
        return;
    }
    const dim3 g = grid(wide ? a.n / V + a.n % V : a.n);
    if (!wide)
        hipLaunchKernelGGL((k_vstack<T, 1, 0>), g, dim3(256), 0, st, s);
    else if (s.nsrc == 1)
        hipLaunchKernelGGL((k_vstack<T, V, 1>), g, dim3(256), 0, st, s);
    else if (s.nsrc == 2)
        hipLaunchKernelGGL((k_vstack<T, V, 2>), g, dim3(256), 0, st, s);
    else if (s.nsrc == 3)
        hipLaunchKernelGGL((k_vstack<T, V, 3>), g, dim3(256), 0, st, s);
    else
        hipLaunchKernelGGL((k_vstack<T, V, 4>), g, dim3(256), 0, st, s);
}
} // namespace
void launch_vexpr(const VExprArgsT<float>& a, hipStream_t st) { launch_vexpr_t(a, st); }
void launch_vexpr(const VExprArgsT<double>& a, hipStream_t st) { launch_vexpr_t(a, st); }

} // namespace pcxd
