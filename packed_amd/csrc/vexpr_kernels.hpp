// vexpr_kernels.hpp -- fused element-wise evaluation of packed complex vector expressions.
//
// A program of up to 64 instructions runs per element on four complex registers.  Programs that
// use the registers as a stack -- every compiled expression does -- run on k_vstack, others on the
// register machine k_vexpr (register numbers are wave-uniform, so operand selection is a short
// chain of uniform selects).  Every source is read once per element and the destination written
// once: 8 B per source element plus 8 B per output element, bound by HBM bandwidth.
// Arithmetic follows simd_common.hpp:296-410 of the reference (complex division as
// (a conj(b)) / |b|^2 with fused multiply-adds; real scalars act on the real part for + and -).
#pragma once
#include "fft_kernels.hpp"

namespace pcxk {

enum : int32_t {
    VOP_LOAD = 0, VOP_ADD, VOP_SUB, VOP_MUL, VOP_DIV, VOP_CONJ, VOP_ADDS, VOP_SUBS, VOP_RSUBS, VOP_MULS, VOP_DIVS,
    VOP_RDIVS, VOP_ADDR, VOP_SUBR, VOP_RSUBR, VOP_MULR, VOP_DIVR, VOP_RDIVR, VOP_COUNT
};

// T = float or double: the element type of every vector and scalar of the program.
template<class T>
struct VInstrT {
    int32_t op, d, a, b;
    T       s_re, s_im;
};
template<class T>
struct VSourceT {
    const T* data;
    int64_t  lp; // log2 of the pack size
};
constexpr int kVMaxProg = 64, kVMaxSrc = 16, kVRegs = 4;
template<class T>
struct VExprArgsT {
    VSourceT<T> src[kVMaxSrc];
    VInstrT<T>  prog[kVMaxProg];
    int32_t     nprog;
    T*          dst;
    int         dst_lp;
    int64_t     n;
};

// The stack form of a program (vexpr_stack): one 5-bit code per instruction, 12 to a word.  The
// codes are the vop values, plus a LOAD of each of the first four sources (VST_LOAD0 + k), a LOAD
// of source load[k], and the binary operations with the operands' stack order reversed.
enum : int32_t { VST_LOAD0 = VOP_COUNT, VST_LOADX = VST_LOAD0 + 4, VST_XADD, VST_XSUB, VST_XMUL, VST_XDIV, VST_COUNT };
static_assert(VST_COUNT <= 32, "five bits per code");
constexpr int kVPreload = 4, kVPerWord = 12;
template<class T>
struct VStackArgsT {
    VSourceT<T> src[kVMaxSrc]; // in the order of their first LOAD
    uint64_t    code[(kVMaxProg + kVPerWord - 1) / kVPerWord];
    int32_t     load[kVMaxProg]; // source of a VST_LOADX
    cx<T>       scalar[kVMaxProg];
    int32_t     nprog, nsrc;
    T*          dst;
    int         dst_lp;
    int64_t     n;
};

// simd_common.hpp:296-309: (a conj(b)) / (br^2 + bi^2)
template<class T>
__device__ __forceinline__ cx<T> vdiv(cx<T> a, cx<T> b) {
    T den = fmat(b.y, b.y, b.x * b.x);
    T re  = fmat(a.y, b.y, a.x * b.x);
    T im  = fmat(a.y, b.x, -(a.x * b.y));
    return {re / den, im / den};
}
// simd_common.hpp:372-383: real s / b
template<class T>
__device__ __forceinline__ cx<T> vrdiv_real(T s, cx<T> b) {
    T den = fmat(b.y, b.y, b.x * b.x);
    return {(s * b.x) / den, -(s * b.y) / den};
}

template<class T>
__device__ __forceinline__ cx<T> vsel(const cx<T> (&r)[kVRegs], int i) {
    cx<T> v = r[0];
    v    = i == 1 ? r[1] : v;
    v    = i == 2 ? r[2] : v;
    v    = i == 3 ? r[3] : v;
    return v;
}

template<class T>
__global__ __launch_bounds__(256) void k_vexpr(VExprArgsT<T> p) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.n; i += stride) {
        cx<T> r[kVRegs] = {};
        for (int k = 0; k < p.nprog; ++k) {
            const VInstrT<T> in = p.prog[k]; // uniform: kernel arguments
            const cx<T>      x  = vsel(r, in.a);
            const cx<T>      y  = vsel(r, in.b);
            const cx<T>      s  = {in.s_re, in.s_im};
            cx<T>            z;
            switch (in.op) {
            case VOP_LOAD: {
                const VSourceT<T> src = p.src[in.a];
                const int64_t o   = pidx(i, (int)src.lp);
                z                 = {src.data[o], src.data[o + ((int64_t)1 << src.lp)]};
                break;
            }
            case VOP_ADD: z = cadd(x, y); break;
            case VOP_SUB: z = csub(x, y); break;
            case VOP_MUL: z = cmul(x, y); break;
            case VOP_DIV: z = vdiv(x, y); break;
            case VOP_CONJ: z = cconj(x); break;
            case VOP_ADDS: z = cadd(x, s); break;
            case VOP_SUBS: z = csub(x, s); break;
            case VOP_RSUBS: z = csub(s, x); break;
            case VOP_MULS: z = cmul(x, s); break;
            case VOP_DIVS: z = vdiv(x, s); break;
            case VOP_RDIVS: z = vdiv(s, x); break;
            case VOP_ADDR: z = {x.x + in.s_re, x.y}; break;
            case VOP_SUBR: z = {x.x - in.s_re, x.y}; break;
            case VOP_RSUBR: z = {in.s_re - x.x, -x.y}; break;
            case VOP_MULR: z = {x.x * in.s_re, x.y * in.s_re}; break;
            case VOP_DIVR: z = {x.x / in.s_re, x.y / in.s_re}; break;
            case VOP_RDIVR: z = vrdiv_real(in.s_re, x); break;
            default: z = x; break;
            }
            r[0] = in.d == 0 ? z : r[0];
            r[1] = in.d == 1 ? z : r[1];
            r[2] = in.d == 2 ? z : r[2];
            r[3] = in.d == 3 ? z : r[3];
        }
        const int64_t o                       = pidx(i, p.dst_lp);
        p.dst[o]                              = r[0].x;
        p.dst[o + ((int64_t)1 << p.dst_lp)]   = r[0].y;
    }
}

// ---------------------------------------------------------------------------------------------
// k_vstack: stack programs, V elements per thread (V = 16 / sizeof(T), or 1 where a vector is not
// 16-byte aligned).  Bound by HBM, so it keeps many bytes in flight and few instructions per
// element: the first NS sources are loaded together in 16-byte accesses before the program runs,
// the interpreter's branches are shared by V elements, a unary operation moves no registers and a
// binary one or a LOAD shifts the stack, and the codes come from one scalar word per 12
// instructions.
// a * conj(b) + s * c on 5,000,011 floats, packs 8, 8 and 1 (160 MB): 94 -> 30 us
// (5.3 TB/s); a product of two 2^20-element vectors of pack 8 (25 MB): 12.9 -> 7.6 us.  With one
// element per thread the selects of the register machine and the one load in flight per wave were
// the bound; four elements per thread on the register machine took 45 us.
template<class T, int V>
struct cxv {
    cx<T> e[V];
};

// The 2V values of elements i .. i + V - 1 (i a multiple of V) of a packed vector: V real parts and
// V imaginary parts, or 2V consecutive values for packs below V (vsplit separates them).
template<class T, int V>
struct vraw {
    typedef T vt __attribute__((ext_vector_type(V)));
    vt        a, b;
};
template<int V>
__device__ __forceinline__ int64_t vraw_second(int lp) {
    return lp >= ilog2c(V) ? (int64_t)1 << lp : (int64_t)V;
}
template<int V, class T>
__device__ __forceinline__ vraw<T, V> vload(const T* data, int lp, int64_t i) {
    using vt        = typename vraw<T, V>::vt;
    const int64_t o = pidx(i, lp); // packs below V: 2i
    return {*reinterpret_cast<const vt*>(data + o), *reinterpret_cast<const vt*>(data + o + vraw_second<V>(lp))};
}
template<int V, class T>
__device__ __forceinline__ cxv<T, V> vsplit(const vraw<T, V>& r, int lp) {
    cxv<T, V> z;
#pragma unroll
    for (int k = 0; k < V; ++k)
        z.e[k] = {r.a[k], r.b[k]};
    if constexpr (V > 1) {
        auto at = [&](int q) { return q < V ? r.a[q] : r.b[q - V]; };
        if (lp == 0) {
#pragma unroll
            for (int k = 0; k < V; ++k)
                z.e[k] = {at(2 * k), at(2 * k + 1)};
        }
        if constexpr (V > 2)
            if (lp == 1) {
#pragma unroll
                for (int k = 0; k < V; ++k)
                    z.e[k] = {at(k + (k & ~1)), at(k + (k & ~1) + 2)};
            }
    }
    return z;
}
template<int V, class T>
__device__ __forceinline__ void vstore(T* data, int lp, int64_t i, const cxv<T, V>& z) {
    vraw<T, V> r;
#pragma unroll
    for (int k = 0; k < V; ++k)
        r.a[k] = z.e[k].x, r.b[k] = z.e[k].y;
    if constexpr (V > 1) {
        auto put = [&](int q, T v) {
            if (q < V)
                r.a[q] = v;
            else
                r.b[q - V] = v;
        };
        if (lp == 0) {
#pragma unroll
            for (int k = 0; k < V; ++k)
                put(2 * k, z.e[k].x), put(2 * k + 1, z.e[k].y);
        }
        if constexpr (V > 2)
            if (lp == 1) {
#pragma unroll
                for (int k = 0; k < V; ++k)
                    put(k + (k & ~1), z.e[k].x), put(k + (k & ~1) + 2, z.e[k].y);
            }
    }
    using vt                                                = typename vraw<T, V>::vt;
    const int64_t o                                         = pidx(i, lp);
    *reinterpret_cast<vt*>(data + o)                        = r.a;
    *reinterpret_cast<vt*>(data + o + vraw_second<V>(lp))   = r.b;
}

template<class T, int V, int NS>
__device__ __forceinline__ void vstack_run(const VStackArgsT<T>& p, int64_t i) {
    using C = cx<T>;
    using E = cxv<T, V>;
    vraw<T, V> raw[NS > 0 ? NS : 1];
#pragma unroll
    for (int k = 0; k < NS; ++k)
        raw[k] = vload<V>(p.src[k].data, (int)p.src[k].lp, i);
    E in[NS > 0 ? NS : 1];
#pragma unroll
    for (int k = 0; k < NS; ++k)
        in[k] = vsplit<V>(raw[k], (int)p.src[k].lp);
    auto load = [&](int j) {
        const VSourceT<T> s = p.src[j];
        return vsplit<V>(vload<V>(s.data, (int)s.lp, i), (int)s.lp);
    };
    auto source = [&](auto jj) { // the last elements' threads preload nothing
        constexpr int j = decltype(jj)::value;
        if constexpr (j < NS)
            return in[j];
        else
            return load(j);
    };
    E        r0 = {}, r1 = {}, r2 = {}, r3 = {}; // r0: top of the stack
    uint64_t code = 0;
    for (int k = 0; k < p.nprog; ++k) {
        if (k % kVPerWord == 0)
            code = p.code[k / kVPerWord];
        const int op = (int)(code & 31);
        code >>= 5;
        auto un = [&](auto f) {
#pragma unroll
            for (int e = 0; e < V; ++e)
                r0.e[e] = f(r0.e[e]);
        };
        auto bin = [&](auto f) { // below, top
#pragma unroll
            for (int e = 0; e < V; ++e)
                r0.e[e] = f(r1.e[e], r0.e[e]);
            r1 = r2;
            r2 = r3;
        };
        auto push = [&](const E& z) {
            r3 = r2;
            r2 = r1;
            r1 = r0;
            r0 = z;
        };
        switch (op) {
        case VST_LOAD0: push(source(std::integral_constant<int, 0>{})); break;
        case VST_LOAD0 + 1: push(source(std::integral_constant<int, 1>{})); break;
        case VST_LOAD0 + 2: push(source(std::integral_constant<int, 2>{})); break;
        case VST_LOAD0 + 3: push(source(std::integral_constant<int, 3>{})); break;
        case VST_LOADX: push(load(p.load[k])); break;
        case VOP_ADD:
        case VST_XADD: bin([](C x, C y) { return cadd(x, y); }); break;
        case VOP_SUB: bin([](C x, C y) { return csub(x, y); }); break;
        case VOP_MUL: bin([](C x, C y) { return cmul(x, y); }); break;
        case VOP_DIV: bin([](C x, C y) { return vdiv(x, y); }); break;
        case VST_XSUB: bin([](C x, C y) { return csub(y, x); }); break;
        case VST_XMUL: bin([](C x, C y) { return cmul(y, x); }); break;
        case VST_XDIV: bin([](C x, C y) { return vdiv(y, x); }); break;
        case VOP_CONJ: un([](C x) { return cconj(x); }); break;
        case VOP_ADDS: un([s = p.scalar[k]](C x) { return cadd(x, s); }); break;
        case VOP_SUBS: un([s = p.scalar[k]](C x) { return csub(x, s); }); break;
        case VOP_RSUBS: un([s = p.scalar[k]](C x) { return csub(s, x); }); break;
        case VOP_MULS: un([s = p.scalar[k]](C x) { return cmul(x, s); }); break;
        case VOP_DIVS: un([s = p.scalar[k]](C x) { return vdiv(x, s); }); break;
        case VOP_RDIVS: un([s = p.scalar[k]](C x) { return vdiv(s, x); }); break;
        case VOP_ADDR: un([s = p.scalar[k].x](C x) { return C{x.x + s, x.y}; }); break;
        case VOP_SUBR: un([s = p.scalar[k].x](C x) { return C{x.x - s, x.y}; }); break;
        case VOP_RSUBR: un([s = p.scalar[k].x](C x) { return C{s - x.x, -x.y}; }); break;
        case VOP_MULR: un([s = p.scalar[k].x](C x) { return C{x.x * s, x.y * s}; }); break;
        case VOP_DIVR: un([s = p.scalar[k].x](C x) { return C{x.x / s, x.y / s}; }); break;
        case VOP_RDIVR: un([s = p.scalar[k].x](C x) { return vrdiv_real(s, x); }); break;
        default: break;
        }
    }
    vstore<V>(p.dst, p.dst_lp, i, r0);
}

// Thread q takes the V elements from V*q on; the n mod V last elements have a thread each.
template<class T, int V, int NS>
__global__ __launch_bounds__(256) void k_vstack(VStackArgsT<T> p) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t groups = p.n / V, items = groups + p.n % V;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < items; q += stride) {
        if (V == 1 || q < groups)
            vstack_run<T, V, NS>(p, q * V);
        else
            vstack_run<T, 1, 0>(p, groups * V + (q - groups));
    }
}

} // namespace pcxk
