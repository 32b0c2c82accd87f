// pcx_gpu.hip -- C ABI of the gfx950 FFT / overlap-save cross-correlation path (include/pcx_gpu.h).
//
// Plans own device twiddle tables and, for N > 16384, a buffer for the four-step intermediate.  Everything is launched asynchronously on the caller's stream.
#include "pcx_gpu.h"

#include "dispatch.hpp"

#include <hip/hip_runtime.h>

#include <array>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <queue>
#include <string>
#include <utility>
#include <vector>
#include <algorithm>

using namespace pcxk;
using namespace pcxd;

namespace {

thread_local std::string g_err;

int fail(int code, std::string msg) {
    g_err = std::move(msg);
    return code;
}

#define HIPCHK(x)                                                                                  \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess)                                                                      \
            return fail(PCX_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_));              \
    } while (0)

bool is_pow2(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }
int  ilog2(int64_t v) {
    int l = 0;
    while (((int64_t)1 << l) < v)
        ++l;
    return l;
}

std::string s(int64_t v) { return std::to_string(v); }

// fft.hpp:1806-1812
int check_size(int64_t n) {
    if (n > 1 && is_pow2(n))
        return PCX_SUCCESS;
    return fail(PCX_ERR_INVALID_SIZE, "fft_size (which is  " + s(n) + ") is not an integer power of two");
}
// fft.hpp:1814-1826
int check_sub_size(int64_t sub) {
    if (sub >= 8 && is_pow2(sub))
        return PCX_SUCCESS;
    if (sub < 8)
        return fail(PCX_ERR_INVALID_SUB_SIZE,
                    "fft_sub_size (which is  " + s(sub) + ") is smaller than minimum (which is 8)");
    return fail(PCX_ERR_INVALID_SUB_SIZE, "fft_sub_size (which is  " + s(sub) + ") is not an integer power of two");
}
int check_pack(int64_t p, const char* what) {
    if (is_pow2(p) && p <= ((int64_t)1 << 40))
        return PCX_SUCCESS;
    return fail(PCX_ERR_INVALID_PACK, std::string(what) + " pack size (which is " + s(p) + ") is not a power of two");
}

// Plan-time work (twiddle tables, kernel spectra) runs on one non-blocking stream per device, and
// set-up waits for that stream only: other streams of the process are never serialised by it.
constexpr int kMaxDevices = 64;
std::mutex    g_setup_mu;
hipStream_t   g_setup[kMaxDevices] = {};

hipError_t setup_stream(hipStream_t* out) {
    int        dev = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    if (dev < 0 || dev >= kMaxDevices)
        return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_setup_mu);
    if (!g_setup[dev]) {
        e = hipStreamCreateWithFlags(&g_setup[dev], hipStreamNonBlocking);
        if (e != hipSuccess)
            return e;
    }
    *out = g_setup[dev];
    return hipSuccess;
}

template<class V>
hipError_t gen_twiddles(V* t, int64_t M, int64_t stride, int64_t count, hipStream_t st) {
    using T    = decltype(V{}.x);
    int64_t nb = (count + 255) / 256;
    hipLaunchKernelGGL(k_twiddles<T>, dim3((unsigned)nb), dim3(256), 0, st, t, M, stride, count);
    return hipGetLastError();
}

// Twiddle tables filled by one launch: table k holds W_m^(stride e) for e < end[k] - end[k - 1], or
// (m = 0) the array that k_tile reads.
constexpr int kMaxTables = 10;
template<class T>
struct TablesArgs {
    vec2<T>* t[kMaxTables];
    int64_t  m[kMaxTables], stride[kMaxTables], end[kMaxTables];
    int      count, lg;
};
template<class T>
__global__ __launch_bounds__(256) void k_tables(TablesArgs<T> a) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int     k = 0;
    while (k < a.count && e >= a.end[k])
        ++k;
    if (k == a.count)
        return;
    if (k > 0)
        e -= a.end[k - 1];
    if constexpr (sizeof(T) == 4)
        if (a.m[k] == 0) {
            a.t[k][e] = tile_twiddle((int)e, a.lg);
            return;
        }
    a.t[k][e] = twiddle<T>((e * a.stride[k]) % a.m[k], a.m[k]);
}

// ---------------------------------------------------------------- shape lookup
template<class T>
const FourStepT<T>* find_in(const ShapeList<T>& l, int lg, int n2, int g, int c) {
    for (int i = 0; i < l.count; ++i) {
        const FourStepT<T>& f = l.data[i];
        if (f.lg == lg && (n2 == 0 || f.n2 == n2) && (g == 0 || f.g == g) && (c == 0 || f.c == c))
            return &f;
    }
    return nullptr;
}
// The first listed shape that matches (0 = any): the defaults first, then the alternatives.
const FourStep* find_shape(int lg, int n2, int g, int c) {
    if (const FourStep* f = find_in(shapes_default(), lg, n2, g, c))
        return f;
    return find_in(shapes_alt(), lg, n2, g, c);
}
// The default shape of a plan: the first listed one of its size, except for the permuted orders
// of 2^21 .. 2^24.  Their row pass stores contiguous blocks, so rows of 2^14 points, one per
// workgroup, with the widest column tiles that leaves win (per 2 GiB, forward / inverse, against
// the first listed shape, whose wide row groups serve the natural order's strided store):
// 2^21 2.09 / 2.12 ms (2.33 / 2.25), 2^22 2.05 / 2.19 (2.58 / 2.51), 2^23 2.29 / 2.46
// (3.14 / 3.21), 2^24 2.75 / 2.99 (2.93 / 3.29).  At 2^20, 4096-point rows (four per workgroup)
// and 64-column tiles: 1.97 / 1.93 ms against 2.12 / 2.06 (one 16384-point row per workgroup
// made the inverse slower there, 2.66 ms).
const FourStep* default_shape(int lg, int order) {
    if (order != PCX_ORDER_NORMAL && lg >= 21 && lg <= 24)
        if (const FourStep* f = find_shape(lg, lg - 14, 1, 16384 >> (lg - 14)))
            return f;
    if (order != PCX_ORDER_NORMAL && lg == 20)
        if (const FourStep* f = find_shape(20, 8, 4, 64))
            return f;
    return find_shape(lg, 0, 0, 0);
}
const FourStepT<double>* find_shape64(int lg, int n2, int g, int c) {
    if (const FourStepT<double>* f = find_in(shapes64_default(), lg, n2, g, c))
        return f;
    return find_in(shapes64_alt(), lg, n2, g, c);
}
// The small-tile shape for a call of `points` points with the plan's split, or null.
template<class T>
const FourStepT<T>* find_small(const SmallList<T>& l, const FourStepT<T>* sh, int64_t points) {
    for (int i = 0; i < l.count; ++i) {
        const SmallShapeT<T>& e = l.data[i];
        if (e.f.lg == sh->lg && e.f.n1 == sh->n1 && points <= ((int64_t)1 << e.max_lg))
            return &e.f;
    }
    return nullptr;
}
// The same for FP64: bit_reversed 2^21 .. 2^23 take rows of 2^13 points, one per workgroup, and
// the widest column tiles (per 2 GiB, forward / inverse: 2.02 / 1.92, 2.06 / 2.14, 2.53 / 2.61 ms
// against 2.41 / 2.47, 2.53 / 2.64, 4.23 / 4.44 with the first listed shapes).
const FourStepT<double>* default_shape64(int lg, int order) {
    if (order != PCX_ORDER_NORMAL && lg >= 21 && lg <= 23)
        if (const FourStepT<double>* f = find_shape64(lg, lg - 13, 1, 8192 >> (lg - 13)))
            return f;
    return find_shape64(lg, 0, 0, 0);
}
// The split kernels for the plan's shape: same size and the same N1 x N2 split (the plan's
// scratch layout and row / column counts follow its shape); only the default shapes have them.
const FourStepMfma* find_mfma(int lg, const FourStep* sh) {
    for (const auto& f : shapes_mfma())
        if (f.lg == lg && sh == find_shape(lg, 0, 0, 0) && f.n1 == sh->n1 && f.n2 == sh->n2)
            return &f;
    return nullptr;
}
// The same above 2^20: the split shapes of 2^21 .. 2^24 follow the default shapes.
// (Same split N1 x N2 as the plan's shape: the plan's tables follow the split; rows per
// workgroup and columns per tile are the split kernels' own.)
const FourStep* find_mfma_big(int lg, const FourStep* sh, int precision) {
    if (lg < 21 || lg > 24 || precision < PCX_PREC_BF16X3 || precision > PCX_PREC_FP16X2 || !sh)
        return nullptr;
    const FourStep* f = &shapes_mfma_big()[precision - 1][lg - 21];
    return f->n1 == sh->n1 && f->n2 == sh->n2 ? f : nullptr;
}

} // namespace

// ---------------------------------------------------------------- plan
struct pcx_plan_s {
    int64_t n     = 0;
    int     lg    = 0;
    int     order = 0;
    bool    two_pass = false;
    int     n1_lg = 0, n2_lg = 0; // N = N1 * N2, N1 contiguous (row) length, N2 column length
    void*   tables = nullptr;     // the allocation that holds every table below
    float2* tw_row = nullptr;     // W_N (single pass) or W_N1
    float2* tw_col = nullptr;     // W_N2
    float2* twl    = nullptr;     // W_N^e, e < 2^tw_ls
    float2* twh    = nullptr;     // W_N^(e << tw_ls)
    int     tw_ls  = 0;
    // four-step intermediate of one chunk (allocated on the first large call); calls on different
    // streams are ordered on it: tmp_ev is recorded after the last use, on tmp_stream
    float*      tmp        = nullptr;
    int64_t     tmp_cap    = 0; // transforms the intermediate holds
    hipEvent_t  tmp_ev     = nullptr;
    hipStream_t tmp_stream = nullptr;
    bool        tmp_used   = false;
    int64_t chunk        = 0; // transforms per four-step chunk
    const FourStep* shape = nullptr; // four-step kernels and tile sizes
    int     precision    = PCX_PREC_FP32;
    // grid caps of the two passes (persistent loop; 0: one workgroup per tile; -1: the shape's own)
    int64_t grid_col     = -1;
    int64_t grid_row     = -1;
    bool    auto_shape   = true; // no shape was chosen by the caller: calls of few points take small tiles
    int     nt_flags     = 0; // bit 0/1: streaming load/store of src/dst, bit 2/3: of the intermediate
    float2* tw_dif       = nullptr; // W_M for the one-pass k_dif kernel
    // one-pass forms (pcx_plan_set_one_pass): one workgroup per transform of 2^15 (FP64: 2^14) points
    // (W_N in tw_one), k_dif, k_tile
    bool    use_one      = true;
    void*   tw_one       = nullptr;
    // natural-order 2^15 / 2^16: one pass over tiles held by one workgroup (k_tile): W_N in thread
    // order, W_128, W_(N/128)^(c t); one workgroup per CU
    float2* tw_tile      = nullptr;
    int     ncu          = 0;
    // three-pass natural-order transforms of 2^21 .. 2^24 (FP64: 2^21 .. 2^23): stage tables
    // W_N2, W_Nb, W_Na and the two-level W_N1 pass table (lo, hi), in the plan's precision
    bool    use_three    = false;
    void*   tw3[5]       = {};
    int     tw_ls1       = 0;
    // FP64 plans (pcx_plan_create_f64): the same roles in double precision
    bool     f64      = false;
    double2* tw64_row = nullptr;
    double2* tw64_col = nullptr;
    double2* twl64    = nullptr;
    double2* twh64    = nullptr;
    const FourStepT<double>* shape64 = nullptr;
    std::mutex mu;
};

extern "C" int pcx_version(void) { return 2; }
extern "C" const char* pcx_last_error(void) { return g_err.c_str(); }

namespace {

// Default bytes of one four-step chunk's intermediate (2 GiB: the whole 2^28-point headline batch
// in one chunk; a 288 GB part holds it several times over).
constexpr int64_t kChunkBytes = (int64_t)2048 << 20;

// The twiddle tables of a plan for its N1 x N2 split, in one allocation filled by one launch (a 2^15
// plan has seven tables: 32 us to create with an allocation and a launch for each, 16 so).  A
// plan that has tables keeps them if the new ones cannot be made; its callers see to it that no
// enqueued work uses the old ones.
template<class T>
hipError_t plan_tables(pcx_plan_t p, hipStream_t st) {
    using V            = vec2<T>;
    constexpr bool F64 = sizeof(T) == 8;
    TablesArgs<T>  a{};
    void**         place[kMaxTables];
    int64_t        offset[kMaxTables], bytes = 0;
    auto           add = [&](auto** table, int64_t m, int64_t stride, int64_t count) {
        const int k = a.count++;
        place[k]    = (void**)table;
        offset[k]   = bytes;
        a.m[k] = m, a.stride[k] = stride, a.end[k] = (k > 0 ? a.end[k - 1] : 0) + count;
        bytes += (count * (int64_t)sizeof(V) + 255) & ~(int64_t)255;
    };
    V **row, **col, **lo, **hi;
    if constexpr (F64)
        row = &p->tw64_row, col = &p->tw64_col, lo = &p->twl64, hi = &p->twh64;
    else
        row = &p->tw_row, col = &p->tw_col, lo = &p->twl, hi = &p->twh;
    const int64_t n = p->n;
    if (!p->two_pass) {
        add(row, n, 1, n);
    } else {
        // W_N1, W_N2 and the pass tables W_N = lo[e mod 2^ls] * hi[e >> ls]
        const int64_t n1 = (int64_t)1 << p->n1_lg, n2 = (int64_t)1 << p->n2_lg, nl = (int64_t)1 << p->tw_ls;
        add(row, n1, 1, n1);
        add(col, n2, 1, n2);
        add(lo, n, 1, nl);
        add(hi, n, nl, n / nl);
        // the three-pass form: stage tables W_N2, W_Nb, W_Na and the two-level W_N1 table of pass 2
        if (const ThreePassT<T>* tp = three_of<T>(p->lg)) {
            const int l1 = p->lg - tp->n2_lg, ls = (l1 + 1) / 2;
            add(&p->tw3[0], (int64_t)1 << tp->n2_lg, 1, (int64_t)1 << tp->n2_lg);
            add(&p->tw3[1], (int64_t)1 << kThreeNbLog2, 1, (int64_t)1 << kThreeNbLog2);
            add(&p->tw3[2], (int64_t)1 << tp->na_lg, 1, (int64_t)1 << tp->na_lg);
            add(&p->tw3[3], (int64_t)1 << l1, 1, (int64_t)1 << ls);
            add(&p->tw3[4], (int64_t)1 << l1, (int64_t)1 << ls, (int64_t)1 << (l1 - ls));
            p->tw_ls1 = ls;
        }
        if (p->lg == (F64 ? kOnePassLog2_64 : kOnePassLog2))
            add(&p->tw_one, n, 1, n);
        if constexpr (!F64) {
            const int64_t m = (int64_t)1 << dif_core_log2(p->order);
            if (p->lg == kOnePassLog2)
                add(&p->tw_dif, m, 1, m);
            if (p->order == PCX_ORDER_NORMAL && p->lg >= kCuTileMinLog2 && p->lg <= kCuTileMaxLog2)
                add(&p->tw_tile, 0, 0, tile_table((int)(n / kTilePoints)));
        }
    }
    char*      block = nullptr;
    hipError_t he    = hipMalloc(&block, bytes);
    if (he != hipSuccess)
        return he;
    for (int k = 0; k < a.count; ++k)
        a.t[k] = reinterpret_cast<V*>(block + offset[k]);
    a.lg = p->lg;
    if (a.count == 1) { // 14.3 us for a single pass, 15.3 with k_tables
        he = gen_twiddles(a.t[0], a.m[0], a.stride[0], a.end[0], st);
    } else {
        hipLaunchKernelGGL(k_tables<T>, dim3((unsigned)((a.end[a.count - 1] + 255) / 256)), dim3(256), 0, st, a);
        he = hipGetLastError();
    }
    if (he == hipSuccess)
        he = hipStreamSynchronize(st);
    if (he != hipSuccess) {
        (void)hipFree(block);
        return he;
    }
    for (int k = 0; k < a.count; ++k)
        *place[k] = a.t[k];
    (void)hipFree(p->tables);
    p->tables = block;
    return hipSuccess;
}

} // namespace

extern "C" int pcx_plan_create(int64_t fft_size, int64_t sub_size, int order, pcx_plan_t* out) {
    if (!out)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan output pointer is null");
    *out = nullptr;
    if (int e = check_size(fft_size))
        return e;
    if (int e = check_sub_size(sub_size))
        return e;
    if (order < 0 || order > 2)
        return fail(PCX_ERR_INVALID_ARGUMENT, "order (which is " + s(order) + ") is not a fft_order");
    int lg = ilog2(fft_size);
    if (lg > kMaxLog2)
        return fail(PCX_ERR_UNSUPPORTED, "fft_size (which is " + s(fft_size) + ") exceeds the supported maximum 2^24");
    if (order == PCX_ORDER_UNORDERED && lg < 5)
        return fail(PCX_ERR_UNSUPPORTED,
                    "unordered fft_size (which is " + s(fft_size) + ") is below the 32-point finisher size");
    hipStream_t st = nullptr;
    HIPCHK(setup_stream(&st));
    auto* p  = new pcx_plan_s;
    p->n     = fft_size;
    p->lg    = lg;
    p->order = order;
    if (lg > kMaxSinglePass) {
        p->two_pass = true;
        p->shape    = default_shape(lg, order);
        if (!p->shape) {
            delete p;
            return fail(PCX_ERR_UNSUPPORTED, "no four-step kernels for fft_size " + s(fft_size));
        }
        p->n2_lg = p->shape->n2;
        p->n1_lg = p->shape->n1;
        p->tw_ls = (lg + 1) / 2;
        // transforms per four-step chunk: the intermediate holds one chunk
        p->chunk = std::max<int64_t>(1, kChunkBytes / (fft_size * 8));
    }
    // three passes are the default where they exist: 2^21 / 2^22 / 2^23 / 2^24 in 2.74 / 2.83 / 2.93 /
    // 2.95 ms per 2 GiB forward against 3.03 / 3.67 / 4.45 / 6.00 with the four-step
    hipError_t he = plan_tables<float>(p, st);
    p->use_three  = p->tw3[0] != nullptr;
    if (he == hipSuccess && p->tw_tile) {
        int dev = 0;
        he      = hipGetDevice(&dev);
        if (he == hipSuccess)
            he = hipDeviceGetAttribute(&p->ncu, hipDeviceAttributeMultiprocessorCount, dev);
    }
    if (he == hipSuccess && p->two_pass)
        he = hipEventCreateWithFlags(&p->tmp_ev, hipEventDisableTiming);
    if (he != hipSuccess) {
        pcx_plan_destroy(p);
        return fail(PCX_ERR_HIP, std::string("plan setup: ") + hipGetErrorString(he));
    }
    *out = p;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_destroy(pcx_plan_t p) {
    if (!p)
        return PCX_SUCCESS;
    // the intermediate may still be in use by enqueued work
    if (p->tmp_ev && p->tmp_used)
        (void)hipEventSynchronize(p->tmp_ev);
    (void)hipFree(p->tables);
    (void)hipFree(p->tmp);
    if (p->tmp_ev)
        (void)hipEventDestroy(p->tmp_ev);
    delete p;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_create_f64(int64_t fft_size, int64_t sub_size, int order, pcx_plan_t* out) {
    if (!out)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan output pointer is null");
    *out = nullptr;
    if (int e = check_size(fft_size))
        return e;
    if (int e = check_sub_size(sub_size))
        return e;
    if (order < 0 || order > 2)
        return fail(PCX_ERR_INVALID_ARGUMENT, "order (which is " + s(order) + ") is not a fft_order");
    if (order == PCX_ORDER_UNORDERED)
        return fail(PCX_ERR_UNSUPPORTED, "the unordered order is defined for float only (the reference's "
                                         "unsorted kernels are float-only)");
    int lg = ilog2(fft_size);
    if (lg > kMaxLog2_64)
        return fail(PCX_ERR_UNSUPPORTED,
                    "double fft_size (which is " + s(fft_size) + ") exceeds the supported maximum 2^23");
    hipStream_t st = nullptr;
    HIPCHK(setup_stream(&st));
    auto* p  = new pcx_plan_s;
    p->n     = fft_size;
    p->lg    = lg;
    p->order = order;
    p->f64   = true;
    if (lg > kMaxSinglePass64) {
        p->two_pass = true;
        p->shape64  = default_shape64(lg, order);
        p->n1_lg    = p->shape64->n1;
        p->n2_lg    = p->shape64->n2;
        p->tw_ls    = (lg + 1) / 2;
        p->chunk    = std::max<int64_t>(1, kChunkBytes / (fft_size * 16));
    }
    hipError_t he = plan_tables<double>(p, st);
    p->use_three  = p->tw3[0] != nullptr;
    if (he == hipSuccess && p->two_pass)
        he = hipEventCreateWithFlags(&p->tmp_ev, hipEventDisableTiming);
    if (he != hipSuccess) {
        pcx_plan_destroy(p);
        return fail(PCX_ERR_HIP, std::string("plan setup: ") + hipGetErrorString(he));
    }
    *out = p;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_element_size(pcx_plan_t p) { return p ? (p->f64 ? 8 : 4) : 0; }

extern "C" int64_t pcx_plan_size(pcx_plan_t p) { return p ? p->n : 0; }

namespace {
int plan_apply_shape(pcx_plan_t p, const FourStep* sh);
}

extern "C" int pcx_plan_set_precision(pcx_plan_t p, int precision) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (p->f64)
        return fail(PCX_ERR_UNSUPPORTED, "a double plan has no precision modes");
    if (precision == PCX_PREC_FP32) {
        p->precision = precision;
        return PCX_SUCCESS;
    }
    if (precision != PCX_PREC_BF16X3 && precision != PCX_PREC_FP16X2)
        return fail(PCX_ERR_UNSUPPORTED, "precision " + s(precision) + " is not implemented");
    // the split kernels of four-step sizes follow the first listed shape's split: a plan on
    // another one (the permuted orders' default at 2^20 .. 2^24) moves to it
    if (p->two_pass && p->lg <= 24) {
        const FourStep* d = find_shape(p->lg, 0, 0, 0);
        const bool has = p->lg <= 20 ? find_mfma(p->lg, p->shape) != nullptr
                                     : find_mfma_big(p->lg, p->shape, precision) != nullptr;
        const bool d_has = d && (p->lg <= 20 ? find_mfma(p->lg, d) != nullptr
                                             : find_mfma_big(p->lg, d, precision) != nullptr);
        if (!has && d_has)
            if (int e = plan_apply_shape(p, d))
                return e;
    }
    const bool covered = p->lg >= 4 && (p->lg <= 20 ? (!p->two_pass || find_mfma(p->lg, p->shape))
                                                     : find_mfma_big(p->lg, p->shape, precision) != nullptr);
    if (!covered)
        return fail(PCX_ERR_UNSUPPORTED, "split-precision transforms cover 2^4 .. 2^24 (default four-step shapes)");
    p->precision = precision;
    return PCX_SUCCESS;
}
extern "C" int pcx_plan_precision(pcx_plan_t p) { return p ? p->precision : -1; }
extern "C" int     pcx_plan_order(pcx_plan_t p) { return p ? p->order : -1; }

namespace {

// Moves a four-step plan to the split of another instantiated shape: the tables follow the split.
template<class T>
int plan_apply_split(pcx_plan_t p, int n1_lg, int n2_lg) {
    if (n1_lg == p->n1_lg && n2_lg == p->n2_lg)
        return PCX_SUCCESS;
    // every enqueued use of the old tables must end
    HIPCHK(hipDeviceSynchronize());
    hipStream_t st = nullptr;
    HIPCHK(setup_stream(&st));
    std::swap(p->n1_lg, n1_lg), std::swap(p->n2_lg, n2_lg);
    const hipError_t he = plan_tables<T>(p, st);
    if (he != hipSuccess)
        p->n1_lg = n1_lg, p->n2_lg = n2_lg; // the tables are still the old split's
    HIPCHK(he);
    return PCX_SUCCESS;
}

int plan_apply_shape(pcx_plan_t p, const FourStep* sh) {
    if (!p->two_pass || p->f64 || !sh || sh->lg != p->lg)
        return fail(PCX_ERR_INVALID_ARGUMENT, "shape does not match the plan");
    if (int e = plan_apply_split<float>(p, sh->n1, sh->n2))
        return e;
    p->shape = sh;
    return PCX_SUCCESS;
}

int plan_apply_shape64(pcx_plan_t p, const FourStepT<double>* sh) {
    if (!p->two_pass || !p->f64 || !sh || sh->lg != p->lg)
        return fail(PCX_ERR_INVALID_ARGUMENT, "shape does not match the plan");
    if (int e = plan_apply_split<double>(p, sh->n1, sh->n2))
        return e;
    p->shape64 = sh;
    return PCX_SUCCESS;
}

} // namespace

namespace {

// A four-step intermediate the caller provides (the allocation-free entry point): `bytes` of
// device memory at `buf`, used instead of the plan's own.
struct ExtTmp {
    void*   buf;
    int64_t bytes;
};

// Transforms from which a call of 2^15 points (FP64: 2^14) runs one workgroup per transform; fewer
// run as k_dif where that serves (out of place, forward or natural order) and spread over the chip
// as small four-step tiles where it does not.  2^15, forward, pack 8, four-step / k_dif / one pass,
// us: 1 transform 14.6 / 20.2 / 22.4, 32 16.4 / 21.6 / -, 64 22.7 / 23.7 / 25.5, 256 51 / 41.9 / 36.9,
// 1024 248 / 188 / 159, 4096 (2^27 points) - / 710 / 546; bit_reversed 64 23.1 / 18.8 / 29.8, 256
// 51 / 43.9 / 40.6, 1024 264 / 199 / 181.  FP64 2^14, four-step / one pass: 64 19.1 / 23.3, 256 48 / 32.3,
// 4096 790 / 484.  (k_dif keeps the calls of less than 48 transforms although the four-step is faster
// there: it needs no intermediate, so a fresh plan's first call may be captured, replays and calls on
// several streams are independent, and the result does not depend on any of that.)
constexpr int64_t kOnePassBatch = 160, kOnePassBatch64 = 96;

// How many of a call's natural-order 2^15 / 2^16 transforms k_tile takes (one per CU and round, `ncu`
// CUs): 2^16 in full rounds and a last one filled to more than 0.7, the others the four-step.
// Forward in packs of 8, us, four-step / k_tile: 160 transforms 61 / 62, 180 73 / 62, 256 103 / 69,
// 512 227 / 146, 769 331 / 244, 4096 1575 / 1120; 257 105 / 116 in two rounds, 85 in one and a
// four-step, 300 136 / 117, 1025 460 / 313.  2^15 beyond three rounds, in one pass over halves in LDS (below) / k_tile: 257
// 57 / 55, packs of 1 63 / 65, 513 92 / 92 and 97 / 107, 769 138 / 129 and 150 / 152, 1024 160 / 136
// and 179 / 156, 4096 555 / 465 and 626 / 587.
int64_t tile_batch(int lg, int64_t batch, int64_t ncu) {
    if (lg == 15)
        return batch > 3 * ncu ? batch : 0;
    const int64_t last = batch % ncu;
    return 10 * last > 7 * ncu ? batch : batch - last;
}

// src_offs / dst_offs (optional, device arrays of `batch` element offsets) replace b * dist.
// T is the element type: float, or double for a plan made by pcx_plan_create_f64.
template<class T>
int run_batch(pcx_plan_t p, int inverse, int normalized, T* dst, int64_t dst_pack, int64_t dst_dist,
              const T* src, int64_t src_pack, int64_t src_dist, int64_t src_size, int64_t batch,
              hipStream_t st, const int64_t* src_offs = nullptr, const int64_t* dst_offs = nullptr,
              const ExtTmp* ext = nullptr) {
    constexpr bool F64 = std::is_same_v<T, double>;
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (p->f64 != F64)
        return fail(PCX_ERR_INVALID_ARGUMENT, p->f64 ? "the plan is for double data (use the _f64 functions)"
                                                     : "the plan is for float data (made by pcx_plan_create)");
    if (!dst || !src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    if (batch < 0)
        return fail(PCX_ERR_INVALID_ARGUMENT, "batch (which is " + s(batch) + ") is negative");
    if (int e = check_pack(dst_pack, "destination"))
        return e;
    if (int e = check_pack(src_pack, "source"))
        return e;
    const int64_t n = p->n;
    if (src_size > n)
        return fail(PCX_ERR_SIZE_MISMATCH,
                    "source size (which is " + s(src_size) + ") is bigger than fft size (which is " + s(n) + ")");
    if (src_size < 0)
        return fail(PCX_ERR_SIZE_MISMATCH, "source size (which is " + s(src_size) + ") is negative");
    // spectra in unordered order keep pack max(P, 8) (avx2_fft.hpp:209-213, 227)
    if (p->order == PCX_ORDER_UNORDERED) {
        if (inverse && src_pack < 8)
            src_pack = 8;
        if (!inverse && dst_pack < 8)
            dst_pack = 8;
    }
    // fft.hpp:783, 889: a pack change wider than one SIMD register (8 floats, 4 doubles) cannot run
    // in place
    constexpr int64_t kReg = F64 ? 4 : 8;
    if ((const T*)dst == src && dst_pack != src_pack && (dst_pack > kReg || src_pack > kReg))
        return fail(PCX_ERR_INPLACE_REPACK, "cannot perform in-place repack from source pack size (which is " +
                                                s(src_pack) + ") to destination pack size (which is " + s(dst_pack) + ")");
    if (batch == 0)
        return PCX_SUCCESS;
    const int   src_lp = ilog2(src_pack), dst_lp = ilog2(dst_pack);
    const T     scale  = (inverse && normalized) ? (T)(1.0 / (double)n) : T(1);
    if (inverse)
        src_size = n;
    const vec2<T> *tw_row, *tw_col, *twl, *twh;
    if constexpr (F64)
        tw_row = p->tw64_row, tw_col = p->tw64_col, twl = p->twl64, twh = p->twh64;
    else
        tw_row = p->tw_row, tw_col = p->tw_col, twl = p->twl, twh = p->twh;

    // a cap of the row pass also holds for the workgroups that run whole transforms
    const int64_t row_cap = std::max<int64_t>(p->grid_row, 0);

    // ---- one pass over a CU's registers and LDS
    if constexpr (!F64) {
        // offsets of multiples of 128 add under packs up to 128 and from N on
        auto fits = [&](int lp) { return lp <= ilog2c(kTileEdge) || (lp >= p->lg && lp <= 27); };
        if (p->tw_tile && p->use_one && p->auto_shape && p->precision == PCX_PREC_FP32 &&
            src_size == n && fits(src_lp) && fits(dst_lp)) {
            if (const int64_t nb = tile_batch(p->lg, batch, p->ncu); nb > 0) {
                TileArgs t{};
                t.a.src = src, t.a.dst = dst, t.a.src_dist = src_dist, t.a.dst_dist = dst_dist;
                t.a.src_size = n, t.a.nrows = nb, t.a.src_lp = src_lp, t.a.dst_lp = dst_lp;
                t.a.conj_in = inverse, t.a.conj_out = inverse, t.a.scale = scale;
                t.a.src_offs = src_offs, t.a.dst_offs = dst_offs;
                t.tw = p->tw_tile, t.tw128 = p->tw_tile + kTilePoints, t.twr = t.tw128 + kTileEdge;
                t.src_sh = src_lp < p->lg, t.dst_sh = dst_lp < p->lg;
                launch_tile(p->lg, t, row_cap > 0 ? std::min<int64_t>(row_cap, p->ncu) : p->ncu, st);
                HIPCHK(hipGetLastError());
                if (nb == batch)
                    return PCX_SUCCESS;
                src += src_offs ? 0 : nb * src_dist, dst += dst_offs ? 0 : nb * dst_dist, batch -= nb;
                src_offs = src_offs ? src_offs + nb : nullptr, dst_offs = dst_offs ? dst_offs + nb : nullptr;
            }
        }
    }

    // ---- one pass: one workgroup (or several, for small sizes) per group of whole transforms
    // (a named shape is the one that runs)
    const bool whole = p->tw_one && p->use_one && p->auto_shape && p->precision == PCX_PREC_FP32 &&
                       batch >= (F64 ? kOnePassBatch64 : kOnePassBatch);
    if (!p->two_pass || whole) {
        RowArgsT<T> a{};
        a.src = src, a.dst = dst, a.src_dist = src_dist, a.dst_dist = dst_dist;
        a.src_size = src_size, a.nrows = batch, a.src_lp = src_lp, a.dst_lp = dst_lp, a.rows_lg = 0;
        a.order = p->order, a.conj_in = inverse, a.conj_out = inverse, a.scale = scale;
        a.twA = whole ? (const vec2<T>*)p->tw_one : tw_row, a.twl = nullptr, a.twh = nullptr, a.tw_ls = 0;
        a.src_offs = src_offs, a.dst_offs = dst_offs;
        const int v = single_variant(inverse, p->order);
        if constexpr (F64)
            (whole ? one_pass64_tab() : single64_tab()[p->lg - 1])[v](a, batch, whole ? row_cap : 0, st);
        else if (whole)
            one_pass_tab()[v](a, batch, row_cap, st);
        else if (p->precision != PCX_PREC_FP32 && p->order == PCX_ORDER_NORMAL)
            single_mfma_tab()[p->precision - 1][p->lg - 4](a, batch, 0, st);
        else if (p->precision != PCX_PREC_FP32)
            single_mfma_perm_tab()[p->precision - 1][p->lg - 4][v](a, batch, 0, st);
        else
            single_tab()[p->lg - 1][v](a, batch, 0, st);
        HIPCHK(hipGetLastError());
        return PCX_SUCCESS;
    }

    // ---- one pass, radix-R decimation in frequency + M-point Stockham (no intermediate)
    if constexpr (!F64)
    if (p->tw_dif && p->use_one && p->precision == PCX_PREC_FP32 && (const float*)dst != src && !src_offs &&
        (!inverse || p->order == PCX_ORDER_NORMAL)) {
        RowArgs a{};
        a.src = src, a.dst = dst, a.src_dist = src_dist, a.dst_dist = dst_dist;
        a.src_size = src_size, a.nrows = batch, a.src_lp = src_lp, a.dst_lp = dst_lp;
        a.conj_in = inverse, a.conj_out = inverse, a.scale = scale;
        a.twA = p->tw_dif, a.twl = p->twl, a.twh = p->twh, a.tw_ls = p->tw_ls, a.tw_lg = p->lg;
        a.nt_store = (p->nt_flags >> 1) & 1;
        a.src_offs = src_offs, a.dst_offs = dst_offs;
        dif_tab()[p->order](a, batch, st);
        HIPCHK(hipGetLastError());
        return PCX_SUCCESS;
    }

    // ---- four-step: N = N1 * N2 through an intermediate, `chunk` transforms at a time
    std::lock_guard<std::mutex> lock(p->mu);
    int64_t chunk = batch < p->chunk ? batch : p->chunk;
    T*      tmp   = nullptr;
    if (ext) {
        const int64_t cap = ext->bytes / (int64_t)(2 * sizeof(T) * n);
        if (cap < 1)
            return fail(PCX_ERR_UNSUPPORTED, "fft_size (which is " + s(n) + ") needs " + s(2 * sizeof(T) * n) +
                                                 " bytes of intermediate; the fixed workspace holds " + s(ext->bytes));
        chunk = std::min(chunk, cap);
        tmp   = reinterpret_cast<T*>(ext->buf);
    } else {
        // Calls on different streams share the plan's intermediate: a call on another stream than
        // the last user waits for that use (copies of a C++ fft_unit share one plan).  Not while
        // the stream is being captured into a graph (the event belongs to no capture).
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        HIPCHK(hipStreamIsCapturing(st, &cs));
        const bool capturing = cs != hipStreamCaptureStatusNone;
        if (p->tmp_cap < chunk) {
            if (capturing)
                return fail(PCX_ERR_INVALID_ARGUMENT, "the plan's intermediate must be allocated before graph capture "
                                                      "(run one call of this batch size first)");
            if (p->tmp) {
                HIPCHK(hipEventSynchronize(p->tmp_ev)); // the last use, on whichever stream, has ended
                HIPCHK(hipFree(p->tmp));
                p->tmp     = nullptr;
                p->tmp_cap = 0;
            }
            hipError_t he = hipMalloc(&p->tmp, sizeof(T) * 2 * n * chunk);
            if (he != hipSuccess)
                return fail(PCX_ERR_OUT_OF_MEMORY,
                            "intermediate allocation of " + s(2 * sizeof(T) * n * chunk) + " bytes failed");
            p->tmp_cap = chunk;
        } else if (p->tmp_used && p->tmp_stream != st && !capturing) {
            HIPCHK(hipStreamWaitEvent(st, p->tmp_ev, 0));
        }
        tmp = reinterpret_cast<T*>(p->tmp);
    }
    const FourStepT<T>* shape;
    SmallList<T>        small;
    if constexpr (F64)
        shape = p->shape64, small = shapes64_small();
    else
        shape = p->shape, small = shapes_small();
    // by the whole call, not the chunk: every chunk size then runs the same kernels
    if (p->auto_shape && p->precision == PCX_PREC_FP32)
        if (const FourStepT<T>* f = find_small(small, shape, batch << p->lg))
            shape = f;
    int           C    = shape->c;
    ColLaunchT<T> colf = shape->cols[inverse ? 0 : 1];
    RowLaunchT<T> rowf = shape->rows[(inverse ? 3 : 0) + p->order];
    if constexpr (!F64)
    if (p->precision != PCX_PREC_FP32 && p->lg > 20) {
        const FourStep* fb = find_mfma_big(p->lg, p->shape, p->precision);
        if (!fb)
            return fail(PCX_ERR_UNSUPPORTED, "no split-precision kernels for this four-step shape");
        colf = fb->cols[inverse ? 0 : 1];
        rowf = fb->rows[(inverse ? 3 : 0) + p->order];
        C    = fb->c;
    } else if (p->precision != PCX_PREC_FP32) {
        const FourStepMfma* fm = find_mfma(p->lg, p->shape);
        if (!fm)
            return fail(PCX_ERR_UNSUPPORTED, "no split-precision kernels for this four-step shape");
        colf = fm->cols[p->precision - 1][inverse ? 0 : 1];
        rowf = p->order == PCX_ORDER_NORMAL
                   ? fm->rows[p->precision - 1][inverse ? 1 : 0]
                   : shapes_mfma_perm()[fm - shapes_mfma().data()][p->precision - 1][(inverse ? 2 : 0) + p->order - 1];
        C    = fm->c; // the split kernels keep their own column tile
    }
    const int64_t n1 = (int64_t)1 << p->n1_lg, n2 = (int64_t)1 << p->n2_lg;
    const ThreePassT<T>* tp3 = p->use_three && p->order == PCX_ORDER_NORMAL && p->precision == PCX_PREC_FP32
                                   ? three_of<T>(p->lg)
                                   : nullptr;
    const bool    wide     = tp3 || p->precision != PCX_PREC_FP32;
    const int64_t grid_col = p->grid_col >= 0 ? p->grid_col : (wide ? kWideGrid : shape->grid_col);
    const int64_t grid_row = p->grid_row >= 0 ? p->grid_row : (wide ? kWideGrid : shape->grid_row);
    for (int64_t b0 = 0; b0 < batch; b0 += chunk) {
        int64_t      cb = batch - b0 < chunk ? batch - b0 : chunk;
        const T*       cs  = src_offs ? src : src + b0 * src_dist;
        T*             cd  = dst_offs ? dst : dst + b0 * dst_dist;
        const int64_t* cso = src_offs ? src_offs + b0 : nullptr;
        const int64_t* cdo = dst_offs ? dst_offs + b0 : nullptr;
        if (tp3) {
            // natural order, forward or inverse (conj in pass 1, conj and 1/N in pass 3)
            using V          = vec2<T>;
            const int     l1 = p->lg - tp3->n2_lg; // log2 N1; the intermediate's pack
            const int64_t m1 = (int64_t)1 << l1;
            ColArgsT<T>   c1{}, c2{};
            RowArgsT<T>   r3{};
            c1.src = cs, c1.src_dist = src_dist, c1.src_lp = src_lp, c1.src_size = src_size, c1.src_offs = cso;
            c1.dst = tmp, c1.dst_dist = 2 * n, c1.dst_lp = l1;
            c1.ntiles = cb * (m1 / tp3->c1), c1.n1_lg = l1, c1.conj_in = inverse, c1.conj_out = 0, c1.scale = T(1);
            c1.twA = (const V*)p->tw3[0], c1.twl = twl, c1.twh = twh, c1.tw_ls = p->tw_ls, c1.tw_lg = p->lg;
            c1.nt_load = p->nt_flags & 1, c1.nt_store = (p->nt_flags >> 2) & 1;
            tp3->col1(c1, grid_col, st);
            c2.src = tmp, c2.src_dist = 2 * m1, c2.src_lp = l1, c2.src_size = m1;
            c2.dst = tmp, c2.dst_dist = 2 * m1, c2.dst_lp = l1;
            c2.ntiles = (cb << tp3->n2_lg) * (((int64_t)1 << tp3->na_lg) / tp3->c2), c2.n1_lg = tp3->na_lg;
            c2.conj_in = 0, c2.conj_out = 0, c2.scale = T(1);
            c2.twA = (const V*)p->tw3[1], c2.twl = (const V*)p->tw3[3], c2.twh = (const V*)p->tw3[4];
            c2.tw_ls = p->tw_ls1, c2.tw_lg = l1;
            tp3->col2(c2, grid_col, st);
            r3.src = tmp, r3.src_dist = 2 * n, r3.src_lp = l1, r3.src_size = n;
            r3.dst = cd, r3.dst_dist = dst_dist, r3.dst_lp = dst_lp, r3.dst_offs = cdo;
            r3.rows_lg = p->lg - tp3->na_lg, r3.rsplit_lg = tp3->n2_lg, r3.nrows = cb << (p->lg - tp3->na_lg);
            r3.order = PCX_ORDER_NORMAL, r3.conj_in = 0, r3.conj_out = inverse, r3.scale = scale;
            r3.twA = (const V*)p->tw3[2];
            r3.nt_load = (p->nt_flags >> 3) & 1, r3.nt_store = (p->nt_flags >> 1) & 1;
            tp3->row3(r3, r3.nrows, grid_row, st);
            HIPCHK(hipGetLastError());
            continue;
        }
        ColArgsT<T>  ca{};
        RowArgsT<T>  ra{};
        ca.twA = tw_col, ca.n1_lg = p->n1_lg, ca.ntiles = cb * (n1 / C);
        ra.twA = tw_row, ra.rows_lg = p->n2_lg, ra.nrows = cb * n2, ra.order = p->order;
        ca.tw_lg = p->lg, ra.tw_lg = p->lg;
        if (!inverse) {
            // pass A: columns of src -> intermediate, times W_N^(n1*k2)
            ca.src = cs, ca.src_dist = src_dist, ca.src_lp = src_lp, ca.src_size = src_size, ca.src_offs = cso;
            ca.dst = tmp, ca.dst_dist = 2 * n, ca.dst_lp = p->lg;
            ca.conj_in = 0, ca.conj_out = 0, ca.scale = T(1);
            ca.twl = twl, ca.twh = twh, ca.tw_ls = p->tw_ls;
            ca.nt_load = p->nt_flags & 1, ca.nt_store = (p->nt_flags >> 2) & 1;
            colf(ca, grid_col, st);
            // pass B: rows of the intermediate -> dst in the plan's order
            ra.src = tmp, ra.src_dist = 2 * n, ra.src_lp = p->lg, ra.src_size = n;
            ra.dst = cd, ra.dst_dist = dst_dist, ra.dst_lp = dst_lp, ra.dst_offs = cdo;
            ra.conj_in = 0, ra.conj_out = 0, ra.scale = T(1);
            ra.twl = nullptr, ra.twh = nullptr;
            ra.nt_load = (p->nt_flags >> 3) & 1, ra.nt_store = (p->nt_flags >> 1) & 1;
            rowf(ra, ra.nrows, grid_row, st);
        } else {
            // pass 1: rows (over k1) of the spectrum -> intermediate, times W_N^(n1*k2)
            ra.src = cs, ra.src_dist = src_dist, ra.src_lp = src_lp, ra.src_size = n, ra.src_offs = cso;
            ra.dst = tmp, ra.dst_dist = 2 * n, ra.dst_lp = p->lg;
            ra.conj_in = 1, ra.conj_out = 0, ra.scale = T(1);
            ra.twl = twl, ra.twh = twh, ra.tw_ls = p->tw_ls;
            ra.nt_load = p->nt_flags & 1, ra.nt_store = (p->nt_flags >> 2) & 1;
            rowf(ra, ra.nrows, grid_row, st);
            // pass 2: columns (over k2) of the intermediate -> dst, natural order
            ca.src = tmp, ca.src_dist = 2 * n, ca.src_lp = p->lg, ca.src_size = n;
            ca.dst = cd, ca.dst_dist = dst_dist, ca.dst_lp = dst_lp, ca.dst_offs = cdo;
            ca.conj_in = 0, ca.conj_out = 1, ca.scale = scale;
            ca.twl = nullptr, ca.twh = nullptr;
            ca.nt_load = (p->nt_flags >> 3) & 1, ca.nt_store = (p->nt_flags >> 1) & 1;
            colf(ca, grid_col, st);
        }
        HIPCHK(hipGetLastError());
    }
    if (!ext) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        HIPCHK(hipStreamIsCapturing(st, &cs));
        if (cs == hipStreamCaptureStatusNone) {
            HIPCHK(hipEventRecord(p->tmp_ev, st));
            p->tmp_stream = st;
            p->tmp_used   = true;
        }
    }
    return PCX_SUCCESS;
}

int64_t footprint(int64_t n, int64_t pack) { return ((n + pack - 1) / pack) * pack * 2; }

} // namespace

// ---------------------------------------------------------------- tuning of four-step plans
extern "C" int pcx_plan_set_shape(pcx_plan_t p, int n2_log2, int cols, int rows) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (!p->two_pass)
        return fail(PCX_ERR_UNSUPPORTED, "a single-pass plan (fft_size " + s(p->n) + ") has no four-step shape");
    if (p->precision != PCX_PREC_FP32)
        return fail(PCX_ERR_UNSUPPORTED, "split-precision plans keep the default four-step shape");
    if (n2_log2 < 0 || cols < 0 || rows < 0)
        return fail(PCX_ERR_INVALID_ARGUMENT, "shape selectors are negative");
    std::lock_guard<std::mutex> lock(p->mu);
    if (p->f64) {
        const FourStepT<double>* sh = find_shape64(p->lg, n2_log2, rows, cols);
        if (!sh)
            return fail(PCX_ERR_UNSUPPORTED, "no double four-step shape of fft_size " + s(p->n) + " matches");
        if (int e = plan_apply_shape64(p, sh))
            return e;
    } else {
        const FourStep* sh = find_shape(p->lg, n2_log2, rows, cols);
        if (!sh)
            return fail(PCX_ERR_UNSUPPORTED, "no four-step shape of fft_size " + s(p->n) + " matches");
        if (int e = plan_apply_shape(p, sh))
            return e;
    }
    p->auto_shape = n2_log2 == 0 && cols == 0 && rows == 0;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_shape(pcx_plan_t p, int* n2_log2, int* cols, int* rows) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    int a = 0, c = 0, g = 0;
    if (p->two_pass) {
        a = p->n2_lg;
        c = p->f64 ? p->shape64->c : p->shape->c;
        g = p->f64 ? p->shape64->g : p->shape->g;
    }
    if (n2_log2)
        *n2_log2 = a;
    if (cols)
        *cols = c;
    if (rows)
        *rows = g;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_set_grid(pcx_plan_t p, int64_t grid_col, int64_t grid_row) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (grid_col < 0 || grid_row < 0 || grid_col > ((int64_t)1 << 31) || grid_row > ((int64_t)1 << 31))
        return fail(PCX_ERR_INVALID_ARGUMENT, "grid caps are not in [0, 2^31]");
    std::lock_guard<std::mutex> lock(p->mu);
    p->grid_col = grid_col, p->grid_row = grid_row;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_set_chunk(pcx_plan_t p, int64_t bytes) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (bytes < 0)
        return fail(PCX_ERR_INVALID_ARGUMENT, "chunk size (which is " + s(bytes) + ") is negative");
    std::lock_guard<std::mutex> lock(p->mu);
    const int64_t per = p->n * (p->f64 ? 16 : 8);
    p->chunk          = std::max<int64_t>(1, (bytes ? bytes : kChunkBytes) / per);
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_set_three_pass(pcx_plan_t p, int enable) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (!p->tw3[0])
        return enable ? fail(PCX_ERR_UNSUPPORTED, "no three-pass form for fft_size " + s(p->n)) : PCX_SUCCESS;
    p->use_three = enable != 0;
    return PCX_SUCCESS;
}

extern "C" int pcx_plan_set_one_pass(pcx_plan_t p, int enable) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (!p->tw_one && !p->tw_tile)
        return enable ? fail(PCX_ERR_UNSUPPORTED, "no one-pass kernel for fft_size " + s(p->n)) : PCX_SUCCESS;
    p->use_one = enable != 0;
    return PCX_SUCCESS;
}

extern "C" int pcx_fft(pcx_plan_t p, float* dst, int64_t dst_pack, const float* src, int64_t src_pack,
                       int64_t src_size, void* stream) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    return run_batch(p, 0, 0, dst, dst_pack, 0, src, src_pack, 0, src_size, 1, (hipStream_t)stream);
}

extern "C" int pcx_ifft(pcx_plan_t p, int normalized, float* dst, int64_t dst_pack, const float* src,
                        int64_t src_pack, void* stream) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    return run_batch(p, 1, normalized, dst, dst_pack, 0, src, src_pack, 0, p->n, 1, (hipStream_t)stream);
}

namespace {
template<class T>
int fft_batch(pcx_plan_t p, int inverse, int normalized, T* dst, int64_t dst_pack, int64_t dst_dist, const T* src,
              int64_t src_pack, int64_t src_dist, int64_t src_size, int64_t batch, void* stream,
              const ExtTmp* ext = nullptr) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (batch > 1) {
        int64_t dp = dst_pack, sp = src_pack;
        if (p->order == PCX_ORDER_UNORDERED) {
            if (!inverse && dp < 8)
                dp = 8;
            if (inverse && sp < 8)
                sp = 8;
        }
        // a forward source holds src_size values (zero-extended to the fft size)
        const int64_t src_n = inverse ? p->n : std::min(std::max<int64_t>(src_size, 0), p->n);
        if (is_pow2(dp) && is_pow2(sp) &&
            (dst_dist < footprint(p->n, dp) || src_dist < footprint(src_n, sp)))
            return fail(PCX_ERR_INVALID_ARGUMENT, "batch distance is smaller than one vector");
        if ((const T*)dst == src && dst_dist != src_dist)
            return fail(PCX_ERR_INVALID_ARGUMENT, "in-place batch needs equal source and destination distances");
    }
    return run_batch(p, inverse, normalized, dst, dst_pack, dst_dist, src, src_pack, src_dist,
                     inverse ? p->n : src_size, batch, (hipStream_t)stream, nullptr, nullptr, ext);
}
} // namespace

extern "C" int pcx_fft_batch(pcx_plan_t p, int inverse, int normalized, float* dst, int64_t dst_pack,
                             int64_t dst_dist, const float* src, int64_t src_pack, int64_t src_dist,
                             int64_t src_size, int64_t batch, void* stream) {
    return fft_batch(p, inverse, normalized, dst, dst_pack, dst_dist, src, src_pack, src_dist, src_size, batch,
                     stream);
}

// ---------------------------------------------------------------- allocation-free batched FFT
// The four-step intermediate of pcx_fft_batch_noalloc: a fixed 128 MiB array per GPU (one
// 2^24-point FP32 transform, the largest plan), held until the process ends.  Host code uses the
// address hipGetSymbolAddress returns for the current device, never the array's name (a host-side
// stand-in).  The array needs no clearing: pass A writes every element pass B reads.
constexpr int64_t kNoAllocBytes = (int64_t)128 << 20;
static __device__ __align__(256) float scratch[kNoAllocBytes / (int64_t)sizeof(float)];

namespace {
std::mutex g_scratch_mu;
void*      g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device.
int noalloc_scratch(void** out) {
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return fail(PCX_ERR_UNSUPPORTED, "device " + s(dev) + " is beyond the supported " + s(kMaxDevices));
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        HIPCHK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr)
            return fail(PCX_ERR_HIP, "hipGetSymbolAddress returned no address for the fixed intermediate");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return PCX_SUCCESS;
}
} // namespace

extern "C" int pcx_fft_batch_noalloc(pcx_plan_t p, int inverse, int normalized, float* dst, int64_t dst_pack,
                                     int64_t dst_dist, const float* src, int64_t src_pack, int64_t src_dist,
                                     int64_t src_size, int64_t batch, void* stream) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (p->two_pass && 8 * p->n > kNoAllocBytes)
        return fail(PCX_ERR_UNSUPPORTED, "fft_size (which is " + s(p->n) + ") needs " + s(8 * p->n) +
                                             " bytes of intermediate; the fixed intermediate holds " + s(kNoAllocBytes));
    void* buf = nullptr;
    if (int e = noalloc_scratch(&buf))
        return e;
    const ExtTmp ext{buf, kNoAllocBytes};
    return fft_batch(p, inverse, normalized, dst, dst_pack, dst_dist, src, src_pack, src_dist, src_size, batch, stream,
                     &ext);
}

// ---------------------------------------------------------------- FP64 transforms
extern "C" int pcx_fft_f64(pcx_plan_t p, double* dst, int64_t dst_pack, const double* src, int64_t src_pack,
                           int64_t src_size, void* stream) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    return run_batch(p, 0, 0, dst, dst_pack, 0, src, src_pack, 0, src_size, 1, (hipStream_t)stream);
}

extern "C" int pcx_ifft_f64(pcx_plan_t p, int normalized, double* dst, int64_t dst_pack, const double* src,
                            int64_t src_pack, void* stream) {
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    return run_batch(p, 1, normalized, dst, dst_pack, 0, src, src_pack, 0, p->n, 1, (hipStream_t)stream);
}

extern "C" int pcx_fft_batch_f64(pcx_plan_t p, int inverse, int normalized, double* dst, int64_t dst_pack,
                                 int64_t dst_dist, const double* src, int64_t src_pack, int64_t src_dist,
                                 int64_t src_size, int64_t batch, void* stream) {
    return fft_batch(p, inverse, normalized, dst, dst_pack, dst_dist, src, src_pack, src_dist, src_size, batch,
                     stream);
}

// ---------------------------------------------------------------- cross-correlation
struct pcx_fxcorr_s {
    int64_t    n = 0, m = 0;
    int        lg        = 0;
    int        precision = PCX_PREC_FP32;
    float2*    tw        = nullptr; // W_N of the fused kernel (N <= 16384), or W_N1 of the block path
    float*     kspec     = nullptr; // FFT(g)/N, split re[N] im[N]: natural order, or the block path's rows
    // block path (N > 16384): its kernels, W_N2 and the pass table W_N = lo[e mod 2^ls] * hi[e >> ls]
    const XcBlockSet* blk = nullptr;
    float2*    tw_col = nullptr, *twl = nullptr, *twh = nullptr;
    int        tw_ls  = 0;
    // the unit's own buffers: the in-place overlap of every block (fused kernel) or the blocks in
    // flight (block path); calls on another stream than the last user wait for that use (ev)
    float*      own      = nullptr;
    int64_t     own_cap  = 0; // floats
    hipEvent_t  ev       = nullptr;
    hipStream_t ev_stream = nullptr;
    bool        ev_used  = false;
    std::mutex  mu;
};

namespace {

// Block path: at most this many bytes of blocks in flight in the unit's own buffer.
constexpr int64_t kXcBlockBytes = (int64_t)512 << 20;

// The unit's own buffer with at least `floats` floats, ordered after its last use on any stream.
int xc_own(pcx_fxcorr_t x, int64_t floats, hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIPCHK(hipStreamIsCapturing(st, &cs));
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (x->own_cap < floats) {
        if (capturing)
            return fail(PCX_ERR_INVALID_ARGUMENT, "the correlation's buffers must be allocated before graph capture "
                                                  "(run one call of this size first)");
        if (x->own) {
            if (x->ev_used)
                HIPCHK(hipEventSynchronize(x->ev));
            HIPCHK(hipFree(x->own));
            x->own     = nullptr;
            x->own_cap = 0;
        }
        if (hipMalloc(&x->own, sizeof(float) * floats) != hipSuccess)
            return fail(PCX_ERR_OUT_OF_MEMORY, "correlation buffer allocation of " + s(4 * floats) + " bytes failed");
        x->own_cap = floats;
    } else if (x->ev_used && x->ev_stream != st && !capturing) {
        HIPCHK(hipStreamWaitEvent(st, x->ev, 0));
    }
    return PCX_SUCCESS;
}
int xc_own_done(pcx_fxcorr_t x, hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIPCHK(hipStreamIsCapturing(st, &cs));
    if (cs == hipStreamCaptureStatusNone) {
        HIPCHK(hipEventRecord(x->ev, st));
        x->ev_stream = st;
        x->ev_used   = true;
    }
    return PCX_SUCCESS;
}

// The block path's arguments that do not depend on the call.
XcBlockArgs xc_block_args(pcx_fxcorr_t x) {
    XcBlockArgs a{};
    a.ksp = x->kspec, a.tw_row = x->tw, a.tw_col = x->tw_col, a.twl = x->twl, a.twh = x->twh;
    a.lg = x->lg, a.n1_lg = x->blk->n1, a.tw_ls = x->tw_ls;
    return a;
}

int64_t grid_of(int64_t work) { return std::max<int64_t>(1, std::min<int64_t>((work + 255) / 256, (int64_t)1 << 20)); }

} // namespace

extern "C" int pcx_fxcorr_create(const float* g, int64_t g_pack, int64_t g_size, int64_t fft_size, void* stream,
                                 pcx_fxcorr_t* out) {
    if (!out)
        return fail(PCX_ERR_INVALID_ARGUMENT, "output pointer is null");
    *out = nullptr;
    if (!g)
        return fail(PCX_ERR_INVALID_ARGUMENT, "kernel pointer is null");
    if (int e = check_size(fft_size))
        return e;
    if (int e = check_pack(g_pack, "kernel"))
        return e;
    if (g_size < 1 || g_size > fft_size)
        return fail(PCX_ERR_SIZE_MISMATCH,
                    "source size (which is " + s(g_size) + ") is bigger than fft size (which is " + s(fft_size) + ")");
    int lg = ilog2(fft_size);
    if (lg > kMaxLog2)
        return fail(PCX_ERR_UNSUPPORTED, "fxcorr fft_size (which is " + s(fft_size) + ") exceeds 2^24");
    hipStream_t st    = (hipStream_t)stream;
    hipStream_t setup = nullptr;
    HIPCHK(setup_stream(&setup));
    auto* x = new pcx_fxcorr_s;
    x->n = fft_size, x->m = g_size, x->lg = lg;
    x->blk        = lg > kMaxSinglePass ? &xc_block_tab()[lg - kMaxSinglePass - 1] : nullptr;
    hipError_t he = hipMalloc(&x->kspec, sizeof(float) * 2 * fft_size);
    if (he == hipSuccess)
        he = hipEventCreateWithFlags(&x->ev, hipEventDisableTiming);
    auto table = [&](float2** t, int64_t m, int64_t stride, int64_t count) {
        if (he == hipSuccess)
            he = hipMalloc(t, sizeof(float2) * count);
        if (he == hipSuccess)
            he = gen_twiddles(*t, m, stride, count, setup);
    };
    const int64_t n1 = x->blk ? (int64_t)1 << x->blk->n1 : fft_size, n2 = fft_size / n1;
    table(&x->tw, n1, 1, n1);
    if (x->blk) {
        x->tw_ls         = (lg + 1) / 2;
        const int64_t nl = (int64_t)1 << x->tw_ls;
        table(&x->tw_col, n2, 1, n2);
        table(&x->twl, fft_size, 1, nl);
        table(&x->twh, fft_size, nl, fft_size / nl);
        // the two passes of FFT(g) below go through the unit's own buffer
        if (he == hipSuccess)
            he = hipMalloc(&x->own, sizeof(float) * 2 * fft_size);
        x->own_cap = 2 * fft_size;
    }
    if (he == hipSuccess)
        he = hipStreamSynchronize(setup);
    if (he != hipSuccess) {
        pcx_fxcorr_destroy(x);
        return fail(PCX_ERR_HIP, std::string("fxcorr setup: ") + hipGetErrorString(he));
    }
    // kernel spectrum: FFT of g zero-extended to N, scaled by 1/N (fxcorr.hpp:67-68); in the block
    // path its column pass and then its rows, each stored where it stands
    RowArgs a{};
    a.dst = x->kspec, a.nrows = n2, a.dst_lp = lg, a.rows_lg = 0;
    a.order = 0, a.conj_in = 0, a.conj_out = 0, a.scale = (float)(1.0 / (double)fft_size);
    a.twA = x->tw;
    if (x->blk) {
        XcBlockArgs b = xc_block_args(x);
        b.src = g, b.src_lp = ilog2(g_pack), b.len = g_size, b.step = fft_size, b.nblocks = 1, b.nb = 1, b.buf = x->own;
        x->blk->col_in(b, st);
        he    = hipGetLastError();
        a.src = x->own, a.src_lp = lg, a.src_dist = n1, a.dst_dist = n1, a.src_size = n1;
    } else {
        a.src = g, a.src_lp = ilog2(g_pack), a.src_size = g_size;
    }
    if (he == hipSuccess) {
        single_tab()[ilog2(n1) - 1][0](a, n2, 0, st);
        he = hipGetLastError();
    }
    if (he == hipSuccess)
        he = hipStreamSynchronize(st);
    if (he != hipSuccess) {
        pcx_fxcorr_destroy(x);
        return fail(PCX_ERR_HIP, std::string("fxcorr kernel spectrum: ") + hipGetErrorString(he));
    }
    *out = x;
    return PCX_SUCCESS;
}

extern "C" int pcx_fxcorr_destroy(pcx_fxcorr_t x) {
    if (!x)
        return PCX_SUCCESS;
    if (x->ev && x->ev_used)
        (void)hipEventSynchronize(x->ev);
    (void)hipFree(x->tw);
    (void)hipFree(x->kspec);
    (void)hipFree(x->tw_col);
    (void)hipFree(x->twl);
    (void)hipFree(x->twh);
    (void)hipFree(x->own);
    if (x->ev)
        (void)hipEventDestroy(x->ev);
    delete x;
    return PCX_SUCCESS;
}

extern "C" int64_t pcx_fxcorr_step(pcx_fxcorr_t x, int64_t src_pack) {
    if (!x || !is_pow2(src_pack))
        return -1;
    int64_t overlap = x->m - 1;
    if (x->n <= overlap)
        return -1;
    // fxcorr.hpp:110: step = ((N - overlap) / P) * P
    return (x->n - overlap) / src_pack * src_pack;
}

extern "C" int64_t pcx_fxcorr_workspace_min(pcx_fxcorr_t x) { return x ? 8 * x->n : -1; }

extern "C" int pcx_fxcorr_set_precision(pcx_fxcorr_t x, int precision) {
    if (!x)
        return fail(PCX_ERR_INVALID_ARGUMENT, "fxcorr handle is null");
    if (precision != PCX_PREC_FP32 && precision != PCX_PREC_BF16X3 && precision != PCX_PREC_FP16X2)
        return fail(PCX_ERR_UNSUPPORTED, "precision " + s(precision) + " is not implemented");
    if (precision != PCX_PREC_FP32 && (x->lg < 4 || x->lg > kMaxSinglePass))
        return fail(PCX_ERR_UNSUPPORTED, "split-precision correlation covers fft_size 16 .. 16384");
    x->precision = precision;
    return PCX_SUCCESS;
}

namespace {

int fxcorr_run(pcx_fxcorr_t x, float* dst, int64_t dst_pack, int64_t dst_dist, const float* src, int64_t src_pack,
               int64_t src_dist, int64_t len, int64_t channels, const ExtTmp* ws, hipStream_t st) {
    if (!x)
        return fail(PCX_ERR_INVALID_ARGUMENT, "fxcorr handle is null");
    if (!dst || !src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    if (int e = check_pack(dst_pack, "destination"))
        return e;
    if (int e = check_pack(src_pack, "source"))
        return e;
    if (len < 0 || channels < 0)
        return fail(PCX_ERR_SIZE_MISMATCH, "signal length (which is " + s(len) + ") or channel count is negative");
    int64_t step = pcx_fxcorr_step(x, src_pack);
    if (step <= 0)
        return fail(PCX_ERR_SIZE_MISMATCH, "fft size (which is " + s(x->n) + ") leaves no output per block for a kernel of " +
                                               s(x->m) + " taps at pack " + s(src_pack));
    const bool inplace = (const float*)dst == src;
    if (channels > 1 && (src_dist < footprint(len, src_pack) || dst_dist < footprint(len, dst_pack)))
        return fail(PCX_ERR_INVALID_ARGUMENT, "channel distance is smaller than one signal");
    if (inplace && (dst_pack != src_pack || dst_dist != src_dist))
        return fail(PCX_ERR_INPLACE_REPACK, "cannot perform in-place repack from source pack size (which is " +
                                                s(src_pack) + ") to destination pack size (which is " + s(dst_pack) + ")");
    if (ws && (!ws->buf || ws->bytes < 8 * x->n))
        return fail(PCX_ERR_INVALID_ARGUMENT, "workspace (which is " + s(ws ? ws->bytes : 0) +
                                                  " bytes) is smaller than one fft_size vector (which is " + s(8 * x->n) +
                                                  " bytes)");
    if (len == 0 || channels == 0)
        return PCX_SUCCESS;
    const int64_t nblocks = (len + step - 1) / step;
    const int64_t total   = nblocks * channels;
    const int64_t n       = x->n;
    std::lock_guard<std::mutex> lock(x->mu);

    if (x->lg > kMaxSinglePass) {
        // ---- block path: column pass from the signal, rows with the product, column pass to the
        // destination (fxcorr_kernels.hpp), nb blocks at a time.  Blocks run in increasing order,
        // and a block's outputs lie below every later block's samples, so in place needs no saved
        // overlap.
        float*  buf = nullptr;
        int64_t nb  = 0;
        if (ws) {
            buf = reinterpret_cast<float*>(ws->buf);
            nb  = std::min(total, ws->bytes / (8 * n));
        } else {
            nb = std::min(total, std::max<int64_t>(1, kXcBlockBytes / (8 * n)));
            if (int e = xc_own(x, 2 * n * nb, st))
                return e;
            buf = x->own;
        }
        XcBlockArgs a = xc_block_args(x);
        a.src = src, a.dst = dst, a.buf = buf;
        a.len = len, a.step = step, a.nblocks = nblocks, a.src_dist = src_dist, a.dst_dist = dst_dist;
        a.src_lp = ilog2(src_pack), a.dst_lp = ilog2(dst_pack);
        for (a.bg0 = 0; a.bg0 < total; a.bg0 += nb) {
            a.nb = std::min(nb, total - a.bg0);
            x->blk->col_in(a, st);
            HIPCHK(hipGetLastError());
            x->blk->rows(a, st);
            HIPCHK(hipGetLastError());
            x->blk->col_out(a, st);
            HIPCHK(hipGetLastError());
        }
        return ws ? PCX_SUCCESS : xc_own_done(x, st);
    }

    // ---- fused kernel: one workgroup per block
    XcArgs a{};
    a.src = src, a.dst = dst, a.kre = x->kspec, a.kim = x->kspec + n, a.twA = x->tw;
    a.len = len, a.step = step, a.nblocks = nblocks, a.hlen = n - step;
    a.src_lp = ilog2(src_pack), a.dst_lp = ilog2(dst_pack);
    a.src_dist = src_dist, a.dst_dist = dst_dist, a.channels = channels;
    const XcLaunch launch = x->precision != PCX_PREC_FP32 ? xc_mfma_tab()[x->precision - 1][x->lg - 4] : xc_tab()[x->lg - 1];
    if (!(inplace && nblocks > 1 && a.hlen > 0)) {
        a.blk0 = 0, a.blk1 = total;
        launch(a, st);
        HIPCHK(hipGetLastError());
        return PCX_SUCCESS;
    }
    // In place: a block overwrites samples that its predecessor reads.  When they lie within the
    // next block only (N - step <= step), workgroups run in ticket order and each stores after its
    // predecessor has read (XcArgs::order: one word per workgroup and launch); a workspace of W
    // bytes takes W / 4 - 8 blocks per group of launches.
    const int64_t owords = ws ? ws->bytes / 4 - 8 : total;
    if (a.hlen <= step && owords >= 1) {
        const int64_t group = std::min(total, owords);
        uint32_t*     obuf  = nullptr;
        if (ws) {
            obuf = reinterpret_cast<uint32_t*>(ws->buf);
        } else {
            if (int e = xc_own(x, total + 8, st))
                return e;
            obuf = reinterpret_cast<uint32_t*>(x->own);
        }
        a.order = obuf;
        for (int64_t g0 = 0; g0 < total; g0 += group) {
            a.blk0 = g0, a.blk1 = std::min(total, g0 + group);
            launch(a, st);
            HIPCHK(hipGetLastError());
        }
        return ws ? PCX_SUCCESS : xc_own_done(x, st);
    }
    // Otherwise the overlap is saved first.  With a workspace of W bytes the blocks run in groups
    // of W / (8 * (N - step)), one group after another (a group only overwrites samples of its own
    // blocks).
    const int64_t group = ws ? std::min(total, ws->bytes / (8 * a.hlen)) : total;
    float*        hbuf  = nullptr;
    if (ws) {
        hbuf = reinterpret_cast<float*>(ws->buf);
    } else {
        if (int e = xc_own(x, 2 * total * a.hlen, st))
            return e;
        hbuf = x->own;
    }
    for (int64_t g0 = 0; g0 < total; g0 += group) {
        const int64_t cnt = std::min(group, total - g0);
        a.hre = hbuf, a.him = hbuf + cnt * a.hlen;
        a.blk0 = g0, a.blk1 = g0 + cnt, a.hblk0 = g0;
        hipLaunchKernelGGL(k_fxcorr_halo, dim3((unsigned)grid_of(cnt * a.hlen)), dim3(256), 0, st, src, a.src_lp,
                           src_dist, len, step, a.hlen, nblocks, g0, cnt, hbuf, hbuf + cnt * a.hlen);
        HIPCHK(hipGetLastError());
        launch(a, st);
        HIPCHK(hipGetLastError());
    }
    return ws ? PCX_SUCCESS : xc_own_done(x, st);
}

} // namespace

extern "C" int pcx_fxcorr_exec_batch(pcx_fxcorr_t x, float* dst, int64_t dst_pack, int64_t dst_dist, const float* src,
                                     int64_t src_pack, int64_t src_dist, int64_t len, int64_t channels, void* stream) {
    return fxcorr_run(x, dst, dst_pack, dst_dist, src, src_pack, src_dist, len, channels, nullptr, (hipStream_t)stream);
}

extern "C" int pcx_fxcorr_exec(pcx_fxcorr_t x, float* dst, int64_t dst_pack, const float* src, int64_t src_pack,
                               int64_t len, void* stream) {
    return pcx_fxcorr_exec_batch(x, dst, dst_pack, 0, src, src_pack, 0, len, 1, stream);
}

extern "C" int pcx_fxcorr_exec_batch_ws(pcx_fxcorr_t x, float* dst, int64_t dst_pack, int64_t dst_dist,
                                        const float* src, int64_t src_pack, int64_t src_dist, int64_t len,
                                        int64_t channels, void* workspace, int64_t workspace_bytes, void* stream) {
    const ExtTmp ws{workspace, workspace_bytes};
    return fxcorr_run(x, dst, dst_pack, dst_dist, src, src_pack, src_dist, len, channels, &ws, (hipStream_t)stream);
}

// ---------------------------------------------------------------- memory and utilities
extern "C" int pcx_malloc(void** ptr, size_t bytes) {
    if (!ptr)
        return fail(PCX_ERR_INVALID_ARGUMENT, "pointer is null");
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess)
        return fail(PCX_ERR_OUT_OF_MEMORY, std::string("hipMalloc: ") + hipGetErrorString(e));
    return PCX_SUCCESS;
}
extern "C" int pcx_free(void* ptr) {
    HIPCHK(hipFree(ptr));
    return PCX_SUCCESS;
}
extern "C" int pcx_memcpy_htod(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return PCX_SUCCESS;
}
extern "C" int pcx_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return PCX_SUCCESS;
}
extern "C" int pcx_memcpy_dtod(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
    return PCX_SUCCESS;
}
extern "C" int pcx_memset(void* dst, int value, size_t bytes) {
    HIPCHK(hipMemset(dst, value, bytes));
    return PCX_SUCCESS;
}
extern "C" int pcx_synchronize(void* stream) {
    HIPCHK(hipStreamSynchronize((hipStream_t)stream));
    return PCX_SUCCESS;
}
extern "C" int pcx_generate(float* dst, int64_t pack, int64_t n, uint64_t seed, int dist, double sigma, void* stream) {
    if (!dst)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    if (int e = check_pack(pack, "destination"))
        return e;
    if (n <= 0)
        return PCX_SUCCESS;
    int64_t nb = std::min<int64_t>((n + 255) / 256, (int64_t)1 << 20);
    hipLaunchKernelGGL(k_generate<float>, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, dst, ilog2(pack), n, seed,
                       dist, sigma);
    HIPCHK(hipGetLastError());
    return PCX_SUCCESS;
}
extern "C" int pcx_generate_f64(double* dst, int64_t pack, int64_t n, uint64_t seed, int dist, double sigma,
                                void* stream) {
    if (!dst)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    if (int e = check_pack(pack, "destination"))
        return e;
    if (n <= 0)
        return PCX_SUCCESS;
    int64_t nb = std::min<int64_t>((n + 255) / 256, (int64_t)1 << 20);
    hipLaunchKernelGGL(k_generate<double>, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, dst, ilog2(pack), n,
                       seed, dist, sigma);
    HIPCHK(hipGetLastError());
    return PCX_SUCCESS;
}

// ---------------------------------------------------------------- uneven-batch work queue
namespace {

struct QGroup { // transforms of one size and one direction that run as full-chip launches
    int        lg    = 0;
    int        inv   = 0;
    int64_t    count = 0;
    int64_t    first = 0; // index of the first one in the offset tables
    pcx_plan_t plan  = nullptr;
    bool       own   = false; // the plan is this group's (else the other direction's)
};

} // namespace

struct pcx_queue_s {
    int                 normalized = 1;
    int64_t             njobs      = 0;
    double              flops = 0, bytes = 0;
    // persistent part: transforms of 2^1 .. 2^14 points (k_queue), or of 2^1 .. 2^18 (k_mixed)
    bool                mixed      = false;
    int                 choice     = -1;      // of the two: as tuned, or -1 by queue_prefers_mixed
    int32_t             nitems     = 0;
    QItem*              items      = nullptr; // device
    int64_t*            src_offs   = nullptr; // per transform: items first, then the groups
    int64_t*            dst_offs   = nullptr;
    float2*             tw         = nullptr; // W_A for A = 2 .. 2^14
    int                 grid       = 0;       // workgroups of k_queue
    int                 grid_cap   = 0;
    float2*             ptw        = nullptr; // k_mixed: pass tables, the item counter
    int32_t             ptw_off[kMixMaxLog2 + 1] = {};
    uint32_t*           counter    = nullptr;
    int64_t             mix_floats = 0;       // of a workgroup's intermediate
    // grouped part, largest size first: the sizes above the persistent part's, and the classes the
    // autotuner moved out of k_queue (grouped[log2n][inverse]); the groups run one after another
    // through one four-step intermediate (k_mixed's workgroups have theirs in it, too)
    std::vector<QGroup> groups;
    void*               tmp        = nullptr;
    int64_t             tmp_bytes  = 0;
    // a call on another stream than the intermediate's last user waits for that use
    hipEvent_t          tmp_ev     = nullptr;
    hipStream_t         tmp_stream = nullptr;
    bool                tmp_used   = false;
    std::mutex          mu;
    bool                grouped[kQueueMaxLog2 + 1][2] = {};
    std::vector<pcx_job> jobs; // the job list, to rebuild the items when the split changes
    // captured graph
    hipGraph_t          graph = nullptr;
    hipGraphExec_t      exec  = nullptr;
};

namespace {

int queue_run_group(pcx_queue_t q, const QGroup& g, float* dst, const float* src, hipStream_t st) {
    const int64_t n = (int64_t)1 << g.lg;
    const ExtTmp  ext{q->tmp, q->tmp_bytes};
    return run_batch(g.plan, g.inv, q->normalized, dst, n, 2 * n, src, n, 2 * n, n, g.count, st, q->src_offs + g.first,
                     q->dst_offs + g.first, &ext);
}

// Runs fn, which enqueues work on st through the queue's intermediate, after the intermediate's last
// use on any stream.  (In a capture there is nothing to order: the replay is ordered when it is launched.)
template<class F>
int queue_on_tmp(pcx_queue_t q, hipStream_t st, F&& fn) {
    if (!q->tmp)
        return fn();
    std::lock_guard<std::mutex> lock(q->mu);
    hipStreamCaptureStatus      cs = hipStreamCaptureStatusNone;
    HIPCHK(hipStreamIsCapturing(st, &cs));
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (q->tmp_used && q->tmp_stream != st && !capturing)
        HIPCHK(hipStreamWaitEvent(st, q->tmp_ev, 0));
    const int e = fn();
    if (!capturing) { // also after an error: what was enqueued before it uses the intermediate
        HIPCHK(hipEventRecord(q->tmp_ev, st));
        q->tmp_stream = st, q->tmp_used = true;
    }
    return e;
}

int queue_run(pcx_queue_t q, float* dst, const float* src, hipStream_t st) {
    QueueArgs a{};
    a.src = src, a.dst = dst;
    a.src_offs = q->src_offs, a.dst_offs = q->dst_offs;
    a.items = q->items, a.nitems = q->nitems, a.normalized = q->normalized;
    a.tw = q->tw;
    if (q->nitems > 0 && !q->mixed) {
        launch_queue(a, std::min<int>(q->grid, q->nitems), st);
        HIPCHK(hipGetLastError());
    }
    return queue_on_tmp(q, st, [&] {
        if (q->mixed) {
            MixArgs m{a, (float*)q->tmp, q->mix_floats, q->counter, q->ptw, {}};
            std::copy(std::begin(q->ptw_off), std::end(q->ptw_off), m.ptw_off);
            launch_mixed(m, std::min<int>(q->grid_cap / 2, q->nitems), st);
            HIPCHK(hipGetLastError());
        }
        for (const auto& g : q->groups)
            if (int e = queue_run_group(q, g, dst, src, st))
                return e;
        return (int)PCX_SUCCESS;
    });
}

// Frees the device side of the item list and the groups (the job list and settings stay).
void queue_release(pcx_queue_t q) {
    if (q->exec)
        (void)hipGraphExecDestroy(q->exec);
    if (q->graph)
        (void)hipGraphDestroy(q->graph);
    q->exec = nullptr, q->graph = nullptr;
    if (q->tmp_ev && q->tmp_used)
        (void)hipEventSynchronize(q->tmp_ev);
    if (q->tmp_ev)
        (void)hipEventDestroy(q->tmp_ev);
    q->tmp_ev = nullptr, q->tmp_used = false;
    (void)hipFree(q->items);
    (void)hipFree(q->src_offs);
    (void)hipFree(q->dst_offs);
    (void)hipFree(q->tw);
    (void)hipFree(q->ptw);
    (void)hipFree(q->counter);
    (void)hipFree(q->tmp);
    q->ptw = nullptr, q->counter = nullptr, q->mixed = false, q->mix_floats = 0;
    q->items = nullptr, q->src_offs = q->dst_offs = nullptr, q->tw = nullptr, q->nitems = 0;
    q->tmp = nullptr, q->tmp_bytes = 0;
    for (auto& g : q->groups)
        if (g.own)
            pcx_plan_destroy(g.plan);
    q->groups.clear();
}

void queue_free(pcx_queue_t q) {
    queue_release(q);
    delete q;
}

using QueueCounts = std::array<std::array<int64_t, 2>, kMaxLog2 + 1>; // transforms by size and direction

// Whether the sizes up to 2^18 of a list run faster as one launch of workgroups that take whole
// transforms (k_mixed) than as k_queue and a full-chip launch per class, from the times that these take
// on `ncu` CUs, us:
//   k_mixed   0.97 the longest workgroup's load + 0.8 the mean one + 0.46 as much again, up to half of
//             the longest transform (the chip is shared from the first transform on); a load counts
//             a transform's time on an otherwise empty chip;
//   per class 12.5 and a time per transform, or rounds of one transform per CU (k_tile, and one-array
//             passes of 2^15); 15 and 6 per 10^6 points for k_queue.
// Over 420 lists (16 .. 2000 jobs, smallest 2^4 .. 2^18, largest 2^15 .. 2^19, either direction or both)
// the choice is 0.4 % from the faster of the two on average and 6 % at worst.  Launches per class alone:
// 1.9 % on average and 21 % at worst (more than 3 % for 71 lists); k_mixed alone 41 %, and 6.2 times.
bool queue_prefers_mixed(const QueueCounts& n, int ncu) {
    constexpr double kAlone[4][2] = {{35, 45}, {63, 68}, {112, 121}, {246, 263}}; // 2^15 .. 2^18
    constexpr double kEach[4]     = {0.166, 0.389, 0.863, 1.863};
    const double     scale        = 256.0 / ncu;
    double split = 0, total = 0, longest = 0, small = 0; // small: points up to 2^14
    std::vector<double> load(ncu, 0.0);
    std::priority_queue<double, std::vector<double>, std::greater<double>> least(std::greater<double>(), std::move(load));
    auto take = [&](double us, int64_t count) {
        for (int64_t k = 0; k < count; ++k) {
            const double l = least.top() + us;
            least.pop();
            least.push(l);
            longest = std::max(longest, l);
        }
        total += us * (double)count;
    };
    double one   = 0; // the longest transform
    int    sizes = 0;
    for (int lg = kMixMaxLog2; lg > kQueueMaxLog2; --lg) {
        sizes += n[lg][0] + n[lg][1] > 0;
        for (int inv = 1; inv >= 0; --inv) {
            const int     k     = lg - kQueueMaxLog2 - 1;
            const int64_t count = n[lg][inv];
            if (count == 0)
                continue;
            take(kAlone[k][inv], count);
            one                = std::max(one, kAlone[k][inv]);
            const int64_t last = count % ncu, tiles = lg != 16 ? 0 : 10 * last > 7 * ncu ? count : count - last;
            if (lg == 15 && count >= kOnePassBatch)
                split += 28.6 * (double)((count + ncu - 1) / ncu) + 0.06 * scale * (double)count;
            else if (count > tiles)
                split += 12.5 + kEach[k] * scale * (double)(count - tiles);
            split += 71 * (double)((tiles + ncu - 1) / ncu);
        }
    }
    if (sizes < 2) // nothing to mix: launches per class are faster
        return false;
    for (int lg = 1; lg <= kQueueMaxLog2; ++lg)
        small += (double)((n[lg][0] + n[lg][1]) << lg);
    if (small > 0)
        split += 15 + 6e-6 * scale * small;
    take(9, (int64_t)std::ceil(small / 16384));
    const double mean = total / ncu;
    return 1.02 * (0.97 * longest + 0.8 * mean + 0.46 * std::min(mean, one / 2)) < split;
}

// Builds the persistent items (every class up to 2^18 with k_mixed, else up to 2^14, not marked
// grouped) and the grouped launches (the rest), both largest first, from the job list.
int queue_build(pcx_queue_t q) {
    const pcx_job* jobs  = q->jobs.data();
    const int64_t  njobs = (int64_t)q->jobs.size();
    std::vector<std::vector<int64_t>> bucket((kMaxLog2 + 1) * 2);
    for (int64_t i = 0; i < njobs; ++i)
        bucket[jobs[i].log2n * 2 + jobs[i].inverse].push_back(i);
    std::vector<QItem>   items;
    std::vector<int64_t> qs, qd;
    auto                 put = [&](int64_t job) {
        qs.push_back(jobs[job].src_offset);
        qd.push_back(jobs[job].dst_offset);
    };
    const int   ncu = q->grid_cap / 2;
    QueueCounts n{};
    for (int lg = 1; lg <= kMaxLog2; ++lg)
        n[lg] = {(int64_t)bucket[2 * lg].size(), (int64_t)bucket[2 * lg + 1].size()};
    int four = 0; // the largest four-step size of k_mixed
    for (int lg = kQueueMaxLog2 + 1; lg <= kMixMaxLog2; ++lg)
        four = n[lg][0] + n[lg][1] > 0 ? lg : four;
    // by estimate only for vectors on whole 128-byte lines: k_mixed loses a quarter of its rate on others,
    // launches per class 3 - 7 % (1000 of 2^12 .. 2^18: 567 -> 747 us, 654 -> 691)
    bool lines = true;
    for (const pcx_job& j : q->jobs)
        if (j.log2n > kQueueMaxLog2)
            lines = lines && ((j.src_offset | j.dst_offset) & 31) == 0;
    q->mixed          = four > 0 && (q->choice < 0 ? lines && queue_prefers_mixed(n, ncu) : q->choice == 1);
    const int top     = q->mixed ? kMixMaxLog2 : kQueueMaxLog2;
    const int threads = q->mixed ? kMixThreads : kQueueThreads;
    auto      persistent = [&](int lg, int inv) { return lg <= top && (lg > kQueueMaxLog2 || !q->grouped[lg][inv]); };
    for (int lg = top; lg >= 1; --lg) {
        const int per = std::max(1, threads / (lg >= 4 ? (1 << lg) / 16 : 1));
        for (int inv = 0; inv < 2; ++inv) {
            if (!persistent(lg, inv))
                continue;
            auto& b = bucket[lg * 2 + inv];
            for (size_t k = 0; k < b.size(); k += per) {
                int cnt = (int)std::min<size_t>(per, b.size() - k);
                items.push_back({lg, inv, (int32_t)qs.size(), cnt});
                for (int c = 0; c < cnt; ++c)
                    put(b[k + c]);
            }
        }
    }
    q->nitems       = (int32_t)items.size();
    int64_t tmp_min = 0; // one transform of the largest grouped size
    for (int lg = kMaxLog2; lg >= 1; --lg)
        for (int inv = 0; inv < 2; ++inv) {
            auto& b = bucket[lg * 2 + inv];
            if (b.empty() || persistent(lg, inv))
                continue;
            QGroup g;
            g.lg = lg, g.inv = inv, g.count = (int64_t)b.size(), g.first = (int64_t)qs.size();
            for (int64_t job : b)
                put(job);
            // both directions of a size share a plan (until they are tuned)
            g.own = q->groups.empty() || q->groups.back().lg != lg;
            if (!g.own)
                g.plan = q->groups.back().plan;
            else if (int e = pcx_plan_create((int64_t)1 << lg, 2048, PCX_ORDER_NORMAL, &g.plan))
                return e;
            q->groups.push_back(g);
            if (lg > kQueueMaxLog2) {
                // k_tile leaves less than a round of its sizes to the four-step
                const int64_t most = g.plan->tw_tile ? g.plan->ncu : g.plan->chunk;
                q->tmp_bytes       = std::max(q->tmp_bytes, std::min(g.count, most) * 8 * g.plan->n);
                tmp_min            = std::max(tmp_min, 8 * g.plan->n);
            }
        }
    hipStream_t setup = nullptr;
    hipError_t  he    = setup_stream(&setup);
    auto        upload = [&](auto** dev, const auto& v) {
        if (v.empty() || he != hipSuccess)
            return;
        he = hipMalloc(dev, sizeof(v[0]) * v.size());
        if (he == hipSuccess)
            he = hipMemcpy(*dev, v.data(), sizeof(v[0]) * v.size(), hipMemcpyHostToDevice);
    };
    upload(&q->items, items);
    upload(&q->src_offs, qs);
    upload(&q->dst_offs, qd);
    if (q->mixed) { // every workgroup its own intermediate of the largest size
        q->mix_floats = (int64_t)2 << four;
        q->tmp_bytes  = std::max<int64_t>(q->tmp_bytes, 4 * q->mix_floats * std::min<int64_t>(ncu, q->nitems));
        tmp_min       = std::max(tmp_min, q->tmp_bytes);
    }
    if (q->tmp_bytes > 0 && he == hipSuccess) {
        // on a full device less will do, down to one transform at a time
        while ((he = hipMalloc(&q->tmp, q->tmp_bytes)) == hipErrorOutOfMemory && q->tmp_bytes > tmp_min) {
            (void)hipGetLastError();
            q->tmp_bytes = std::max(tmp_min, q->tmp_bytes / 2);
        }
        if (he == hipErrorOutOfMemory && q->mixed) { // launches per class need less
            (void)hipGetLastError();
            queue_release(q);
            q->choice = 0;
            return queue_build(q);
        }
    }
    if (q->tmp_bytes > 0 && he == hipSuccess)
        he = hipEventCreateWithFlags(&q->tmp_ev, hipEventDisableTiming);
    if (!items.empty() && he == hipSuccess) {
        he = hipMalloc(&q->tw, sizeof(float2) * ((1 << (kQueueMaxLog2 + 1)) - 2));
        for (int lg = 1; lg <= kQueueMaxLog2 && he == hipSuccess; ++lg)
            he = gen_twiddles(q->tw + ((1 << lg) - 2), (int64_t)1 << lg, 1, (int64_t)1 << lg, setup);
        if (he == hipSuccess && q->mixed) {
            // pass tables W_N^e = lo[e mod 2^ls] * hi[e >> ls] of every four-step size
            int32_t at = 0;
            for (int lg = kQueueMaxLog2 + 1; lg <= four; ++lg)
                q->ptw_off[lg] = at, at += pass_tw_entries(lg);
            he = hipMalloc(&q->ptw, sizeof(float2) * at);
            for (int lg = kQueueMaxLog2 + 1; lg <= four && he == hipSuccess; ++lg) {
                const int64_t nl = (int64_t)1 << (lg + 1) / 2, size = (int64_t)1 << lg;
                he = gen_twiddles(q->ptw + q->ptw_off[lg], size, 1, nl, setup);
                if (he == hipSuccess)
                    he = gen_twiddles(q->ptw + q->ptw_off[lg] + nl, size, nl, size / nl, setup);
            }
            if (he == hipSuccess)
                he = hipMalloc(&q->counter, sizeof(uint32_t));
        }
        if (he == hipSuccess)
            he = hipStreamSynchronize(setup);
    }
    if (he != hipSuccess)
        return fail(PCX_ERR_HIP, std::string("queue setup: ") + hipGetErrorString(he));
    return PCX_SUCCESS;
}

// Gives a group a plan of its own, so that tuning it leaves the other direction's alone.
int queue_own_plan(QGroup& g) {
    if (g.own)
        return PCX_SUCCESS;
    if (int e = pcx_plan_create((int64_t)1 << g.lg, 2048, PCX_ORDER_NORMAL, &g.plan))
        return e;
    g.own = true;
    return PCX_SUCCESS;
}

} // namespace

extern "C" int pcx_queue_create(const pcx_job* jobs, int64_t njobs, int normalized, pcx_queue_t* out) {
    if (!out)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue output pointer is null");
    *out = nullptr;
    if (njobs < 0 || (njobs > 0 && !jobs))
        return fail(PCX_ERR_INVALID_ARGUMENT, "job list is null or negative");
    for (int64_t i = 0; i < njobs; ++i) {
        if (jobs[i].log2n < 1 || jobs[i].log2n > kMaxLog2)
            return fail(PCX_ERR_INVALID_SIZE, "fft_size (which is  2^" + s(jobs[i].log2n) + ") is not supported");
        if (jobs[i].inverse != 0 && jobs[i].inverse != 1)
            return fail(PCX_ERR_INVALID_ARGUMENT, "job " + s(i) + ": inverse must be 0 or 1");
        if (jobs[i].src_offset < 0 || jobs[i].dst_offset < 0)
            return fail(PCX_ERR_INVALID_ARGUMENT, "job " + s(i) + ": negative offset");
    }
    int dev = 0, ncu = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    auto* q       = new pcx_queue_s;
    q->normalized = normalized ? 1 : 0;
    q->njobs      = njobs;
    // two workgroups per CU; the autotuner may pick fewer
    q->grid = q->grid_cap = 2 * std::max(1, ncu);
    for (int64_t i = 0; i < njobs; ++i) {
        double n = (double)((int64_t)1 << jobs[i].log2n);
        q->flops += 5.0 * n * (double)jobs[i].log2n;
        q->bytes += 16.0 * n;
    }
    q->jobs.assign(jobs, jobs + njobs);
    if (int e = queue_build(q)) {
        queue_free(q);
        return e;
    }
    *out = q;
    return PCX_SUCCESS;
}

extern "C" int pcx_queue_destroy(pcx_queue_t q) {
    if (q)
        queue_free(q);
    return PCX_SUCCESS;
}

extern "C" int pcx_queue_exec(pcx_queue_t q, float* dst, const float* src, void* stream) {
    if (!q)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue is null");
    if (!dst || !src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    return queue_run(q, dst, src, (hipStream_t)stream);
}

extern "C" int pcx_queue_capture(pcx_queue_t q, float* dst, const float* src, void* stream) {
    if (!q)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue is null");
    if (!dst || !src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    hipStream_t st = (hipStream_t)stream;
    if (!st)
        return fail(PCX_ERR_INVALID_ARGUMENT, "graph capture needs a non-default stream");
    HIPCHK(hipStreamSynchronize(st));
    if (q->exec) {
        HIPCHK(hipGraphExecDestroy(q->exec));
        q->exec = nullptr;
    }
    if (q->graph) {
        HIPCHK(hipGraphDestroy(q->graph));
        q->graph = nullptr;
    }
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    int        e  = queue_run(q, dst, src, st);
    hipGraph_t gr = nullptr;
    hipError_t he = hipStreamEndCapture(st, &gr);
    if (e)
        return e;
    if (he != hipSuccess)
        return fail(PCX_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(he));
    q->graph = gr;
    HIPCHK(hipGraphInstantiate(&q->exec, q->graph, nullptr, nullptr, 0));
    return PCX_SUCCESS;
}

extern "C" int pcx_queue_launch(pcx_queue_t q, void* stream) {
    if (!q || !q->exec)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue has no captured graph");
    // the graph's kernels use the same intermediate as the eager calls
    return queue_on_tmp(q, (hipStream_t)stream, [&] {
        HIPCHK(hipGraphLaunch(q->exec, (hipStream_t)stream));
        return (int)PCX_SUCCESS;
    });
}

extern "C" int pcx_queue_work(pcx_queue_t q, double* flops, double* bytes) {
    if (!q)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue is null");
    if (flops)
        *flops = q->flops;
    if (bytes)
        *bytes = q->bytes;
    return PCX_SUCCESS;
}

namespace {

// Times fn (which enqueues work on st) with events: best of `reps` after one warm-up.
template<class F>
float time_ms(hipStream_t st, F&& fn, int reps = 3) {
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess)
        return 1e30f;
    if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return 1e30f;
    }
    float best = 1e30f;
    if (fn() != PCX_SUCCESS)
        best = -1.f;
    for (int r = 0; r < reps && best >= 0.f; ++r) {
        float ms = 0.f;
        (void)hipEventRecord(a, st);
        if (fn() != PCX_SUCCESS) {
            best = -1.f;
            break;
        }
        (void)hipEventRecord(b, st);
        (void)hipEventSynchronize(b);
        (void)hipEventElapsedTime(&ms, a, b);
        best = ms < best ? ms : best;
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return best < 0.f ? 1e30f : best;
}

} // namespace

// Autotuner: k_mixed or launches per class, workgroups of k_queue, then per grouped size the four-step
// shape and grid caps.  Winners are written to cache_path (one "key value..." line each) and read back
// from it when present.
extern "C" int pcx_queue_autotune(pcx_queue_t q, float* dst, const float* src, void* stream, const char* cache_path) {
    if (!q)
        return fail(PCX_ERR_INVALID_ARGUMENT, "queue is null");
    if (!dst || !src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "data pointer is null");
    if ((const float*)dst == src)
        return fail(PCX_ERR_INVALID_ARGUMENT, "autotuning overwrites dst many times: it must not alias src");
    hipStream_t st = (hipStream_t)stream;
    // a captured graph holds the kernels, grids and twiddle tables of the shapes it was captured
    // with; the tuning below may change all of them, so the graph is dropped (capture again after)
    HIPCHK(hipDeviceSynchronize());
    if (q->exec) {
        HIPCHK(hipGraphExecDestroy(q->exec));
        q->exec = nullptr;
    }
    if (q->graph) {
        HIPCHK(hipGraphDestroy(q->graph));
        q->graph = nullptr;
    }
    if (cache_path) { // reuse earlier decisions
        if (FILE* f = std::fopen(cache_path, "r")) {
            char key[32];
            int  a = 0, b = 0, c = 0, d = 0, e = 0;
            long long gc = 0, gr = 0;
            // the split between the persistent launch and grouped launches comes first (a file without
            // a "mixed" line leaves that choice as it is)
            bool mask[kQueueMaxLog2 + 1][2] = {};
            int  choice = q->choice;
            long pos = std::ftell(f);
            while (std::fscanf(f, "%31s", key) == 1) {
                if (!std::strcmp(key, "grouped") && std::fscanf(f, "%d %d", &a, &b) == 2 && a >= 1 && a <= kQueueMaxLog2 &&
                    (b == 0 || b == 1))
                    mask[a][b] = true;
                else if (!std::strcmp(key, "mixed") && std::fscanf(f, "%d", &a) == 1 && (a == 0 || a == 1))
                    choice = a;
            }
            std::fseek(f, pos, SEEK_SET);
            if (std::memcmp(mask, q->grouped, sizeof(mask)) != 0 || choice != q->choice) {
                std::memcpy(q->grouped, mask, sizeof(mask));
                q->choice = choice;
                queue_release(q);
                if (int err = queue_build(q)) {
                    std::fclose(f);
                    return err;
                }
            }
            while (std::fscanf(f, "%31s", key) == 1) {
                if (!std::strcmp(key, "grouped") && std::fscanf(f, "%d %d", &a, &b) == 2) {
                    continue;
                } else if (!std::strcmp(key, "mixed") && std::fscanf(f, "%d", &a) == 1) {
                    continue;
                } else if (!std::strcmp(key, "queue_grid") && std::fscanf(f, "%d", &a) == 1) {
                    q->grid = std::max(1, std::min(a, q->grid_cap));
                } else if (!std::strcmp(key, "group") && std::fscanf(f, "%d %d %d %d %d %lld %lld", &a, &b, &c, &d, &e, &gc, &gr) == 7) {
                    for (auto& g : q->groups)
                        if (g.lg == a && g.inv == b && g.plan->two_pass) {
                            if (const FourStep* sh = find_shape(a, c, d, e)) {
                                int err = queue_own_plan(g);
                                if (!err)
                                    err = plan_apply_shape(g.plan, sh);
                                if (err) {
                                    std::fclose(f);
                                    return err;
                                }
                                // grid caps of -1: the plan's own choice of shape and caps won
                                g.plan->grid_col = gc, g.plan->grid_row = gr;
                                g.plan->auto_shape = gc < 0;
                            }
                        }
                } else {
                    break;
                }
            }
            std::fclose(f);
            return PCX_SUCCESS;
        }
    }
    auto whole   = [&] { return queue_run(q, dst, src, st); };
    auto rebuild = [&]() -> int {
        queue_release(q);
        return queue_build(q);
    };
    // one launch over the sizes up to 2^18, or launches per class
    bool four = false;
    for (const auto& j : q->jobs)
        four = four || (j.log2n > kQueueMaxLog2 && j.log2n <= kMixMaxLog2);
    if (four) {
        std::memset(q->grouped, 0, sizeof(q->grouped));
        float ms[2];
        for (int c = 1; c >= 0; --c) {
            q->choice = c;
            if (int e = rebuild())
                return e;
            ms[c] = q->mixed == (c == 1) ? time_ms(st, whole) : 1e30f; // (no room for k_mixed)
        }
        if (ms[1] < ms[0]) {
            q->choice = 1;
            if (int e = rebuild())
                return e;
        }
    }
    if (q->nitems > 0 && !q->mixed) {
        float best = 1e30f;
        int   bg   = q->grid;
        for (int grid : {q->grid_cap / 2, (3 * q->grid_cap) / 4, q->grid_cap}) {
            if (grid < 1)
                continue;
            q->grid  = grid;
            float ms = time_ms(st, [&] {
                std::vector<QGroup> keep;
                keep.swap(q->groups); // time the persistent part alone
                int e = queue_run(q, dst, src, st);
                keep.swap(q->groups);
                return e;
            });
            if (ms < best)
                best = ms, bg = grid;
        }
        q->grid = bg;
    }
    // the sizes of k_queue move out to grouped launches when that makes the whole pass faster
    if (!q->mixed) {
        bool present[kQueueMaxLog2 + 1] = {}, any = false;
        for (const auto& j : q->jobs)
            if (j.log2n <= kQueueMaxLog2)
                present[j.log2n] = any = true;
        if (any) {
            const float best = time_ms(st, whole);
            for (int lg = 1; lg <= kQueueMaxLog2; ++lg)
                q->grouped[lg][0] = q->grouped[lg][1] = present[lg];
            if (int e = rebuild())
                return e;
            if (!(time_ms(st, whole) < best)) {
                std::memset(q->grouped, 0, sizeof(q->grouped));
                if (int e = rebuild())
                    return e;
            }
        }
    }
    for (auto& g : q->groups) {
        if (!g.plan->two_pass)
            continue;
        if (int err = queue_own_plan(g))
            return err;
        pcx_plan_t      p    = g.plan;
        auto            time = [&] { return time_ms(st, [&] { return queue_run_group(q, g, dst, src, st); }); };
        // the plan's own choice first (grid caps -1), then every instantiated shape and cap
        const FourStep* best = p->shape;
        int64_t         bgc  = -1;
        float           bms  = time();
        std::vector<const FourStep*> cands;
        for (const ShapeList<float>& l : {shapes_default(), shapes_alt()})
            for (int i = 0; i < l.count; ++i)
                if (l.data[i].lg == g.lg)
                    cands.push_back(&l.data[i]);
        p->auto_shape = false;
        for (const FourStep* sh : cands) {
            if (int err = plan_apply_shape(p, sh))
                return err;
            for (int64_t gc : {(int64_t)0, (int64_t)1024, (int64_t)2048}) {
                p->grid_col = p->grid_row = gc;
                const float ms = time();
                if (ms < bms)
                    bms = ms, best = sh, bgc = gc;
            }
        }
        if (int err = plan_apply_shape(p, best))
            return err;
        p->grid_col = p->grid_row = bgc;
        p->auto_shape = bgc < 0;
    }
    if (cache_path) {
        if (FILE* f = std::fopen(cache_path, "w")) {
            for (int lg = 1; lg <= kQueueMaxLog2; ++lg)
                for (int inv = 0; inv < 2; ++inv)
                    if (q->grouped[lg][inv])
                        std::fprintf(f, "grouped %d %d\n", lg, inv);
            std::fprintf(f, "queue_grid %d\n", q->grid);
            for (auto& g : q->groups)
                if (g.plan->two_pass)
                    std::fprintf(f, "group %d %d %d %d %d %lld %lld\n", g.lg, g.inv, g.plan->shape->n2, g.plan->shape->g,
                                 g.plan->shape->c, (long long)g.plan->grid_col, (long long)g.plan->grid_row);
            if (four)
                std::fprintf(f, "mixed %d\n", q->mixed ? 1 : 0);
            std::fclose(f);
        }
    }
    return PCX_SUCCESS;
}

// ---------------------------------------------------------------- vector expressions
namespace {
// One validation and launch path for both element types (S, I: the C ABI's source and
// instruction structs of that type).
template<class T, class S, class I>
int vexpr_eval(const S* srcs, int32_t nsrc, const I* prog, int32_t nprog, T* dst, int64_t dst_pack, int64_t n,
               void* stream) {
    if (nsrc < 0 || nsrc > PCX_VEXPR_MAX_SRC || (nsrc > 0 && !srcs))
        return fail(PCX_ERR_INVALID_ARGUMENT, "source count (which is " + s(nsrc) + ") is not in [0, 16]");
    if (nprog < 1 || nprog > PCX_VEXPR_MAX_PROG || !prog)
        return fail(PCX_ERR_INVALID_ARGUMENT, "program length (which is " + s(nprog) + ") is not in [1, 64]");
    if (!dst)
        return fail(PCX_ERR_INVALID_ARGUMENT, "destination pointer is null");
    if (n < 0)
        return fail(PCX_ERR_INVALID_ARGUMENT, "size (which is " + s(n) + ") is negative");
    if (int e = check_pack(dst_pack, "destination"))
        return e;
    VExprArgsT<T> a{};
    for (int k = 0; k < nsrc; ++k) {
        if (!srcs[k].data)
            return fail(PCX_ERR_INVALID_ARGUMENT, "source " + s(k) + " is null");
        if (int e = check_pack(srcs[k].pack, "source"))
            return e;
        if ((const T*)dst == srcs[k].data && srcs[k].pack != dst_pack)
            return fail(PCX_ERR_INPLACE_REPACK, "cannot perform in-place repack from source pack size (which is " +
                                                    s(srcs[k].pack) + ") to destination pack size (which is " +
                                                    s(dst_pack) + ")");
        a.src[k].data = srcs[k].data;
        a.src[k].lp   = ilog2(srcs[k].pack);
    }
    for (int k = 0; k < nprog; ++k) {
        const I& in = prog[k];
        bool     ok = in.op >= 0 && in.op < VOP_COUNT && in.d >= 0 && in.d < PCX_VEXPR_REGS;
        if (in.op == VOP_LOAD)
            ok = ok && in.a >= 0 && in.a < nsrc;
        else
            ok = ok && in.a >= 0 && in.a < PCX_VEXPR_REGS && (in.b >= 0 && in.b < PCX_VEXPR_REGS);
        if (!ok)
            return fail(PCX_ERR_INVALID_ARGUMENT, "instruction " + s(k) + " is malformed");
        a.prog[k] = VInstrT<T>{in.op, in.d, in.a, in.b, in.s_re, in.s_im};
    }
    a.nprog  = nprog;
    a.dst    = dst;
    a.dst_lp = ilog2(dst_pack);
    a.n      = n;
    if (n == 0)
        return PCX_SUCCESS;
    launch_vexpr(a, (hipStream_t)stream);
    HIPCHK(hipGetLastError());
    return PCX_SUCCESS;
}
} // namespace

extern "C" int pcx_vexpr_eval(const pcx_vsource* srcs, int32_t nsrc, const pcx_vinstr* prog, int32_t nprog, float* dst,
                              int64_t dst_pack, int64_t n, void* stream) {
    return vexpr_eval(srcs, nsrc, prog, nprog, dst, dst_pack, n, stream);
}

extern "C" int pcx_repack(float* dst, int64_t dst_pack, const float* src, int64_t src_pack, int64_t n, void* stream) {
    pcx_vsource sv{src, src_pack};
    pcx_vinstr  ld{PCX_VOP_LOAD, 0, 0, 0, 0.f, 0.f};
    return pcx_vexpr_eval(&sv, 1, &ld, 1, dst, dst_pack, n, stream);
}

extern "C" int pcx_vexpr_eval_f64(const pcx_vsource_f64* srcs, int32_t nsrc, const pcx_vinstr_f64* prog, int32_t nprog,
                                  double* dst, int64_t dst_pack, int64_t n, void* stream) {
    return vexpr_eval(srcs, nsrc, prog, nprog, dst, dst_pack, n, stream);
}

extern "C" int pcx_repack_f64(double* dst, int64_t dst_pack, const double* src, int64_t src_pack, int64_t n,
                              void* stream) {
    pcx_vsource_f64 sv{src, src_pack};
    pcx_vinstr_f64  ld{PCX_VOP_LOAD, 0, 0, 0, 0.0, 0.0};
    return pcx_vexpr_eval_f64(&sv, 1, &ld, 1, dst, dst_pack, n, stream);
}

// ---------------------------------------------------------------- FFT across vectors
namespace {
template<class T, class Tab>
int fft_across(pcx_plan_t p, int inverse, int normalized, T* const* dst_vecs, int64_t dst_pack, const T* const* src_vecs,
               int64_t src_pack, int64_t length, hipStream_t st, const Tab& tab) {
    constexpr bool F64 = std::is_same_v<T, double>;
    if (!p)
        return fail(PCX_ERR_INVALID_ARGUMENT, "plan is null");
    if (p->f64 != F64)
        return fail(PCX_ERR_INVALID_ARGUMENT, p->f64 ? "the plan is for double data (use pcx_fft_across_f64)"
                                                     : "the plan is for float data (use pcx_fft_across)");
    if (!dst_vecs || !src_vecs)
        return fail(PCX_ERR_INVALID_ARGUMENT, "vector table is null");
    if (length < 0)
        return fail(PCX_ERR_INVALID_ARGUMENT, "length (which is " + s(length) + ") is negative");
    if (int e = check_pack(dst_pack, "destination"))
        return e;
    if (int e = check_pack(src_pack, "source"))
        return e;
    if (p->order != PCX_ORDER_NORMAL)
        return fail(PCX_ERR_UNSUPPORTED, "transforms across vectors are built for the normal order");
    if (p->lg > (int)tab.size())
        return fail(PCX_ERR_UNSUPPORTED, "transforms across vectors cover at most " + s((int64_t)1 << tab.size()) +
                                             " vectors (fft_size " + s(p->n) + ")");
    if (length == 0)
        return PCX_SUCCESS;
    AcrossArgsT<T> a{};
    a.src = src_vecs, a.dst = dst_vecs, a.len = length;
    a.src_lp = ilog2(src_pack), a.dst_lp = ilog2(dst_pack);
    a.conj_in = inverse, a.conj_out = inverse;
    a.scale   = (inverse && normalized) ? (T)(1.0 / (double)p->n) : T(1);
    if constexpr (F64)
        a.twA = p->tw64_row;
    else
        a.twA = p->tw_row;
    tab[p->lg - 1](a, 2048, st);
    HIPCHK(hipGetLastError());
    return PCX_SUCCESS;
}
} // namespace

extern "C" int pcx_fft_across(pcx_plan_t p, int inverse, int normalized, float* const* dst_vecs, int64_t dst_pack,
                              const float* const* src_vecs, int64_t src_pack, int64_t length, void* stream) {
    return fft_across(p, inverse, normalized, dst_vecs, dst_pack, src_vecs, src_pack, length, (hipStream_t)stream,
                      across_tab());
}

extern "C" int pcx_fft_across_f64(pcx_plan_t p, int inverse, int normalized, double* const* dst_vecs,
                                  int64_t dst_pack, const double* const* src_vecs, int64_t src_pack, int64_t length,
                                  void* stream) {
    return fft_across(p, inverse, normalized, dst_vecs, dst_pack, src_vecs, src_pack, length, (hipStream_t)stream,
                      across64_tab());
}
