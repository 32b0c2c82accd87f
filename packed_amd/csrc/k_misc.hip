// k_misc.hip -- the persistent uneven-batch queue kernel (one launch for every transform of
// 2^1 .. 2^14 points) and the vector-expression kernel.
#include "dispatch.hpp"
#include "queue_items.hpp"

#include <algorithm>

namespace pcxk {

constexpr int kQueueLds = kQueueSingleLds<kQueueThreads>;
static_assert(4 * kQueueLds <= 80 * 1024, "two workgroups fit one CU's LDS");

__global__ __launch_bounds__(kQueueThreads, 4) void k_queue(QueueArgs q) {
    for (int it = (int)blockIdx.x; it < q.nitems; it += (int)gridDim.x) {
        const QItem w = q.items[it];
        queue_single_any<kQueueThreads, kQueueLds>(q, w);
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
