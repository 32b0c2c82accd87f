// tile_kernels.hpp -- natural-order transforms of 2^15 and 2^16 FP32 points in one pass over HBM.
//
// A 2^16-point transform (512 KiB) exceeds a CU's LDS, but not its registers and LDS together: one
// workgroup of 1024 threads holds it as R = N / 2^14 tiles of 128 x 128 points, 16 points (32
// VGPRs) per thread and tile.  With n = 128 T + c + 128R n2 and k = k2 + 128 t + 128R q
// (T, t < R; c, n2, k2, q < 128):
//   columns   A_T[c][k2] = sum_n2 x[n] W_128^(n2 k2), tile by tile through LDS;
//   radix R   y_t[c][k2] = W_N^(c k2) W_(128R)^(c t) * sum_T A_T[c][k2] W_(128R)^(T k2) W_R^(T t), in
//             each thread's registers (every tile has the same thread for (c, k2));
//   rows      X[k] = sum_c y_t[c][k2] W_128^(c q), tile by tile through LDS.
// Every load and store covers 128 consecutive elements.  At R = 4, two tiles stay in registers and
// one in LDS (128 KiB) while the fourth is transformed, its exchanges in quarters through the 32
// KiB left.  The kernel is persistent: a tile's registers take the next transform's loads as soon
// as its outputs are stored, so HBM keeps streaming behind the arithmetic.
//
// Bound: vector arithmetic (4500 instructions per wave and 2^16-point transform, 30 us of the 62 of
// a round of 256) and HBM (50 us), half overlapped: one workgroup of 16 waves in step per CU, 63
// vector memory operations in flight per wave.  Without its loads the kernel takes 0.82, without its
// stores 0.76 of its time.  Loading a third tile ahead, or the last two during the second, spilled
// in-flight registers and cost 10 - 20 %; 512 threads of two sub-blocks per tile (half the
// temporaries, but half the operations in flight) cost 15 %.
// Twiddles: W_N^(c k2) once per element of all tiles, from a 128 KiB table in the threads' own order
// (coalesced, from L2); W_128 and W_(128R)^(T k2) wave-uniform through the scalar cache.  (A table of
// W_N^((128T+c) k2), 512 KiB at R = 4, applied per tile, did not stay in L2 beside the stream: 760
// against 556 us for 2048 transforms of 2^16 with and without its loads.)
// 2 GiB of 2^16 split 1560 (two passes) -> 990 us, 4.3 TB/s; in packs of 8 1575 -> 1120, of 1 1880 ->
// 1330 with 4-byte accesses (2^25 points 177, 149 with both parts of an element in one); 2^15 (one
// pass over LDS halves) 1020 -> 900.
#pragma once
#include "fft_kernels.hpp"

namespace pcxk {

constexpr int kTileThreads = 1024, kTileEdge = 128, kTilePoints = kTileEdge * kTileEdge;

struct TileArgs {
    RowArgs       a;     // one row per transform; src_size = N
    const float2* tw;    // W_N^(c k2) at [slot][thread] (tile_twiddle)
    const float2* tw128; // W_128
    const float2* twr;   // W_(128R)^(c t) at [t][c] (and W_(128R)^(T k2) at [T][k2])
    int           src_sh, dst_sh; // 1 for packs up to 128, 0 for packs >= N: poff(128 x) = 128 x << sh
};

// k_tile's tables in one array: W_N^(c k2) at [slot][thread], slot = 8m + r, thread = 128 j8 + c,
// k2 = j8 + 8m + 16r; then W_128; then W_(128R)^(c t) at [t][c].  Entry e of 2^lg points' array:
constexpr int tile_table(int r) { return kTilePoints + kTileEdge * (1 + r); }
__device__ __forceinline__ float2 tile_twiddle(int e, int lg) {
    const int r = (1 << lg) / kTilePoints, f = e - kTilePoints;
    if (f < 0) {
        const int th = e & 1023, slot = e >> 10;
        return twiddle<float>((th & 127) * ((th >> 7) + 8 * (slot >> 3) + 16 * (slot & 7)), 1 << lg);
    }
    if (f < kTileEdge)
        return twiddle<float>(f, kTileEdge);
    return twiddle<float>((f % kTileEdge) * (f / kTileEdge - 1), kTileEdge * r);
}

// LDS floats.  Exchanges of a tile: re and im arrays of 128 rows; columns unpadded, rows at a stride
// of 129 (lanes run over rows: distinct banks).  R = 4: the stashed tile takes the first 32768, the
// quarter exchanges the 8192 after it.
constexpr int kTileRowStride = kTileEdge + 1;
template<int R>
constexpr int tile_lds_floats() {
    return R == 4 ? 2 * kTilePoints + kTilePoints / 2 : 2 * kTileEdge * kTileRowStride;
}

// One resource for both parts of a packed vector: the imaginary part is `im` bytes behind the real
// one (a scalar offset).  With `on` false nothing is read (loads return zero).
struct TileBuf {
    __amdgpu_buffer_rsrc_t r;
    __device__ TileBuf(const float* base, bool on = true) : r(rsrc(base, on ? 0x7FFFFFFFu : 0u)) {}
};

// Base of transform b (uniform): with an offset table the entry is loaded by vector memory, as the
// kernel also stores, and made scalar again here.
__device__ __forceinline__ int64_t tile_off(const int64_t* offs, int64_t dist, int64_t b) {
    const uint64_t o = (uint64_t)(offs ? offs[b] : b * dist);
    return (int64_t)((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(o >> 32)) << 32 |
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)o));
}

// W_128^e at a wave-uniform e, through the scalar cache (the table is constant; the kernel's stores
// keep the compiler from seeing that).
__device__ __forceinline__ cf tile_w(const float2* t, int e) {
    typedef const float __attribute__((address_space(4))) cfloat;
    cfloat* q = (cfloat*)(const float*)(t + e);
    return {q[0], q[1]};
}

// Fixes the order of a phase's arithmetic: the values are computed before this point and used after
// it.  (Instruction selection otherwise moves arithmetic across the barriers, and with it several
// phases' temporaries are live at once.)
template<int CNT>
__device__ __forceinline__ void tile_pin(cf* v) {
#pragma unroll
    for (int s = 0; s < CNT; s += 4)
        asm volatile(""
                     : "+v"(v[s].x), "+v"(v[s].y), "+v"(v[s + 1].x), "+v"(v[s + 1].y), "+v"(v[s + 2].x),
                       "+v"(v[s + 2].y), "+v"(v[s + 3].x), "+v"(v[s + 3].y));
}

// The two radix stages of 128-point transforms around an exchange: butterfly index j8 (0 .. 7,
// wave-uniform), v[r] = x[j8 + 8r] on entry, element j8 + 8m + 16r in slot 8m + r on exit.
template<class X>
__device__ __forceinline__ void tile_fft128(cf* v, int j8, const float2* tw128, const X& exchange) {
    dft<16>(v);
    tile_pin<16>(v);
    exchange(v); // element 16 j8 + r out, j8 + 8m + 16r back in slot 8m + r
    tile_pin<16>(v);
    const int k = opaque_s(j8);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        cf* w = v + 8 * m;
#pragma unroll
        for (int r = 1; r < 8; ++r)
            w[r] = cmul(w[r], tile_w(tw128, r * (k + 8 * m)));
        dft<8>(w);
        tile_pin<8>(w);
    }
}

// ONE: pack 1 on both sides
template<int R, bool ONE>
__global__ __launch_bounds__(kTileThreads, 4) void k_tile(TileArgs q) {
    constexpr int E = kTileEdge, RS = kTileRowStride, V = 16;
    static_assert(R == 2 || R == 4, "two or four tiles");
    __shared__ float lds[tile_lds_floats<R>()];
    const RowArgs&   p   = q.a;
    const int        slp = ONE ? 0 : p.src_lp, dlp = ONE ? 0 : p.dst_lp;
    const int        tid = threadIdx.x;
    auto             ln  = [&] { return opaque(tid) & (E - 1); };          // column c, or row k2
    const int        jb  = __builtin_amdgcn_readfirstlane(tid >> 7);       // butterfly index j8
    const int        hw  = __builtin_amdgcn_readfirstlane((tid >> 6) & 1); // which half of the lanes' 128
    // element (without jb) in slot s after the radix-8 stage: 8m + 16r
    auto el = [](int s) { return 8 * (s >> 3) + 16 * (s & 7); };
    const float      ci  = p.conj_in ? -1.f : 1.f;
    const float      so_ = p.conj_out ? -p.scale : p.scale;

    // Element i = lane part + multiples of 128: poff adds over those (packs up to 128, or >= N)
    auto lane_at = [&](int lp) { return poff((uint32_t)ln() + (uint32_t)(E * R) * (uint32_t)jb, lp) * 4; };

    // (addresses are made opaque per use: loop-invariant, they would all be hoisted and spilled)
    auto load = [&](cf* v, const TileBuf& src, int T) {
        const int      sh = opaque_s(q.src_sh);
        const uint32_t vi = lane_at(slp);
        const uint32_t im = 4u << slp;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < V; ++r) { // element j8 + 8r
            const uint32_t o = (uint32_t)(4 * (E * T + E * R * 8 * r)) << sh;
            if constexpr (ONE)
                v[r] = buf_ld2((float*)nullptr, src.r, vi, o);
            else
                v[r] = cf{buf_ld((float*)nullptr, src.r, vi, o), buf_ld((float*)nullptr, src.r, vi, o + im)};
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // ---- exchanges: each starts after every thread's reads of the one before it
    auto sync = [] {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto xcol = [&](cf* v) {
        sync();
        {
            float* x = lds + ln() + 16 * E * jb;
#pragma unroll
            for (int r = 0; r < V; ++r) {
                const int o        = r * E;
                x[o]               = v[r].x;
                x[o + kTilePoints] = v[r].y;
            }
        }
        sync();
        const float* x = lds + ln() + E * jb;
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int o = el(s) * E;
            v[s]        = cf{x[o], x[o + kTilePoints]};
        }
    };
    // the same through 32 KiB behind the stash, one component at a time: outputs 0 .. 7 of every
    // radix-16 butterfly (read back as m = 0), then 8 .. 15 (m = 1).  Position [8 j8 + r][lane], for
    // columns and (not transposing) rows alike.
    auto x_q = [&](cf* v) {
        float* const x = lds + 2 * kTilePoints;
#pragma unroll
        for (int comp = 0; comp < 2; ++comp)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                sync();
                {
                    float* y = x + ln() + 8 * E * jb;
#pragma unroll
                    for (int s = 8 * m; s < 8 * m + 8; ++s)
                        y[(s & 7) * E] = comp ? v[s].y : v[s].x;
                }
                sync();
                const float* y = x + ln() + E * jb;
#pragma unroll
                for (int s = 8 * m; s < 8 * m + 8; ++s) {
                    const float e = y[8 * (s & 7) * E];
                    (comp ? v[s].y : v[s].x) = e;
                }
            }
    };
    const __amdgpu_buffer_rsrc_t tab = rsrc((const float*)q.tw);
    auto col = [&](cf* v, int T, auto quarter) {
#pragma unroll
        for (int r = 0; r < V; ++r)
            v[r].y *= ci;
        tile_fft128(v, jb, q.tw128, [&](cf* u) {
            if constexpr (decltype(quarter)::value)
                x_q(u);
            else
                xcol(u);
        });
    };
    // (c; k2 = j8 + 8m + 16r) -> (k2; c = j8 + 8r), then the row stage's exchange
    auto xrow = [&](cf* v, auto transpose) {
        constexpr bool TR = decltype(transpose)::value;
        constexpr int  IM = E * RS;
        sync();
        {
            float* x = lds + (TR ? ln() + RS * jb : ln() * RS + 16 * jb);
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const int o = TR ? el(s) * RS : s;
                x[o]        = v[s].x;
                x[o + IM]   = v[s].y;
            }
        }
        sync();
        const float* x = lds + ln() * RS + jb;
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const int o = TR ? 8 * s : el(s);
            v[s]        = cf{x[o], x[o + IM]};
        }
    };
    // the same through 32 KiB, one component at a time: first the elements whose row and column lie
    // in equal halves of the tile, then the others, so that every thread writes and reads 8 of its 16
    // in each step.  Column c of row y at 64 y + (c + y) mod 64 (distinct banks along rows and
    // columns).
    auto xt_q = [&](cf* v) {
        float* const x = lds + 2 * kTilePoints;
#pragma unroll
        for (int comp = 0; comp < 2; ++comp) {
            float t[V];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool up = hw != h; // the other coordinate's half (uniform over the wave)
                sync();
                {
                    const int c = ln(), k = opaque_s(jb + (up ? E / 2 : 0));
#pragma unroll
                    for (int s = 0; s < V; ++s)
                        if ((s & 7) < 4) { // row el(s) + jb of the lower half, or 64 further: slot s + 4
                            const float lo = comp ? v[s].y : v[s].x, hi = comp ? v[s + 4].y : v[s + 4].x;
                            const int   y  = k + el(s);
                            x[y * 64 + ((c + y) & 63)] = up ? hi : lo;
                        }
                }
                sync();
                const int y = ln();
#pragma unroll
                for (int s = 0; s < 8; ++s) { // column jb + 8 s of the lower half, or 64 further: slot s + 8
                    const float e = x[y * 64 + ((jb + 8 * s + y) & 63)];
                    t[s]          = up && h ? t[s] : e;
                    t[s + 8]      = up || !h ? e : t[s + 8];
                }
            }
#pragma unroll
            for (int s = 0; s < V; ++s)
                (comp ? v[s].y : v[s].x) = t[s];
        }
    };
    auto row = [&](cf* v, int t, const TileBuf& dst, auto quarter) {
        auto x = [&](cf* u, auto transpose) {
            if constexpr (!decltype(quarter)::value)
                xrow(u, transpose);
            else if constexpr (decltype(transpose)::value)
                xt_q(u);
            else
                x_q(u);
        };
        x(v, std::true_type{});
        tile_pin<V>(v);
        tile_fft128(v, jb, q.tw128, [&](cf* u) { x(u, std::false_type{}); });
        const int      sh = opaque_s(q.dst_sh);
        const uint32_t vo = lane_at(dlp);
        const uint32_t im = 4u << dlp;
#pragma unroll
        for (int s = 0; s < V; ++s) {
            const uint32_t o = (uint32_t)(4 * (E * t + E * R * el(s))) << sh;
            const cf       y{v[s].x * p.scale, v[s].y * so_};
            if constexpr (ONE) {
                buf_st2(y, dst.r, vo, o);
            } else {
                buf_st(y.x, dst.r, vo, o);
                buf_st(y.y, dst.r, vo, o + im);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    std::false_type whole;
    std::true_type  quarter;

    int64_t b = blockIdx.x;
    if (b >= p.nrows)
        return; // uniform over the workgroup
    cf s0[V], s1[V], w[R == 4 ? V : 1];
    {
        const TileBuf src(p.src + tile_off(p.src_offs, p.src_dist, b));
        load(s0, src, 0);
        load(s1, src, 1);
    }
    for (;;) {
        const int64_t nb = b + gridDim.x;
        const bool    more = nb < p.nrows; // uniform
        const TileBuf next(p.src + tile_off(p.src_offs, p.src_dist, more ? nb : b), more);
        const TileBuf dst(p.dst + tile_off(p.dst_offs, p.dst_dist, b));
        if constexpr (R == 4) {
            col(s0, 0, whole);
            {
                const TileBuf src(p.src + tile_off(p.src_offs, p.src_dist, b));
                load(w, src, 2);
            }
            col(s1, 1, whole);
            col(w, 2, whole);
            sync(); // the last exchange's reads are done
            float* z = lds + opaque(tid);
#pragma unroll
            for (int s = 0; s < V; ++s) {
                z[s * kTileThreads]               = w[s].x;
                z[s * kTileThreads + kTilePoints] = w[s].y;
            }
            const TileBuf src(p.src + tile_off(p.src_offs, p.src_dist, b));
            load(w, src, 3);
            col(w, 3, quarter);
        } else {
            col(s0, 0, whole);
            col(s1, 1, whole);
        }
        // the radix-R step; k2 = jb + el(s) is wave-uniform, so W_(128R)^(T k2) is scalar
        const uint32_t at  = (uint32_t)opaque_after_memory(tid) * 8u;
        const int      kb  = opaque_s(jb);
        auto           wn  = [&](int s) { // W_N^(c k2); the table's thread is 128 j8 + c = tid
            return __builtin_bit_cast(cf, __builtin_amdgcn_raw_buffer_load_b64(
                                              tab, at, (uint32_t)(8 * kTileThreads * s), 0));
        };
        auto ct = [&](int t) { // W_(128R)^(c t)
            const float2 u = q.twr[E * t + (opaque_after_memory(tid) & (E - 1))];
            return cf{u.x, u.y};
        };
        if constexpr (R == 2) {
            const cf t1 = ct(1);
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const cf w1 = wn(s), a = s0[s], c = cmul(s1[s], tile_w(q.twr, E + kb + el(s)));
                s0[s]       = cmul(cadd(a, c), w1);
                s1[s]       = cmul(csub(a, c), cmul(w1, t1));
                if (s % 4 == 3) {
                    tile_pin<4>(s0 + s - 3);
                    tile_pin<4>(s1 + s - 3);
                }
            }
        } else {
            const cf t1 = ct(1), t2 = ct(2), t3 = ct(3);
            float*   z  = lds + opaque(tid);
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const int k  = kb + el(s);
                const cf  w1 = wn(s), a0 = s0[s], a1 = cmul(s1[s], tile_w(q.twr, E + k));
                const cf  a2 = cmul(cf{z[s * kTileThreads], z[s * kTileThreads + kTilePoints]}, tile_w(q.twr, 2 * E + k));
                const cf  a3 = cmul(w[s], tile_w(q.twr, 3 * E + k));
                const cf  e = cadd(a0, a2), f = csub(a0, a2), g = cadd(a1, a3), h = csub(a1, a3);
                const cf  ih = cf{h.y, -h.x}; // -i h
                s0[s]        = cmul(cadd(e, g), w1);
                s1[s]        = cmul(cadd(f, ih), cmul(w1, t1));
                const cf y2  = cmul(csub(e, g), cmul(w1, t2));
                w[s]         = cmul(csub(f, ih), cmul(w1, t3));
                z[s * kTileThreads]               = y2.x;
                z[s * kTileThreads + kTilePoints] = y2.y;
                if (s % 4 == 3) { // four elements' loads in flight
                    tile_pin<4>(s0 + s - 3);
                    tile_pin<4>(s1 + s - 3);
                    tile_pin<4>(w + s - 3);
                }
            }
            row(w, 3, dst, quarter);
#pragma unroll
            for (int s = 0; s < V; ++s)
                w[s] = cf{z[s * kTileThreads], z[s * kTileThreads + kTilePoints]};
            row(w, 2, dst, whole);
        }
        row(s0, 0, dst, whole);
        load(s0, next, 0);
        row(s1, 1, dst, whole);
        if (!more)
            break;
        load(s1, next, 1);
        b = nb;
    }
}

} // namespace pcxk
