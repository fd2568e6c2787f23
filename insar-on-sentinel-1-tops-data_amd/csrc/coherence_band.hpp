// coherence_band.hpp -- boxcar coherence for windows of 2 .. 8 lines and 4 or
// more samples: a workgroup walks down a band of columns, 4 adjacent columns
// per thread.
//
// Same semantics as the LDS-tiled form (EstCoh.cu Cohbasic, 413-456, with the
// zero padding of CohMatSet, 101-139).
//
// Per input row each thread loads 4 samples (one 16-byte CInt16 load, two
// 16-byte CF32 loads, any alignment of the samples' own 4 and 8 bytes), forms
// their products and, in registers, the azimuth sums over the WA latest rows;
// windows of 4, 6 and 8 lines share the pair (and quad) sums of neighbouring
// rows.  The range sum over winRg = 4 kmin + a columns starting at column j of
// the thread's 4 is the sum of
//     the thread's own columns j .. 3              (registers),
//     the 4-column totals of the next kmin - 1 threads, one more for j + a > 4,
//     the first columns of the thread after those
// where a thread leaves its running sums of 1 .. 4 columns in LDS, so every
// window is a plain sum of its own terms, rounding relative to its own sum of
// magnitudes, and the same for every split into bands and row blocks (bands
// start at multiples of 4 columns).
// What bounds it: memory for windows of up to 7 lines (1500 x 21000, 0.5 GB:
// 97-105 us, 5.1 TB/s at 3 lines), waves in flight above (8 lines, 205 VGPRs: 2
// waves per SIMD).  Against the tiles, whose LDS traffic and halo bound them, on 1500 x
// 21000 / 1487 x 24491, us: 5 x 20 183 / 214 -> 100 / 116, 6 x 24 153 / 174 ->
// 105 / 117, 8 x 32 286 / 334 -> 131 / 144, 4 x 9 161 / 188 -> 96 / 114, 2 x 8
// 223 / 262 -> 96 / 123.  Against one row of products at a time in LDS for a
// fixed 3 x 10 window, 2 columns per thread: 95 / 130 -> 97 / 113, 42 -> 35 on
// 1400 x 9000.
#pragma once

#include "tile_window.hpp"
#include "tops_internal.hpp"

#include <type_traits>

namespace tops {

constexpr int CB_PER_THREAD = 4;   // columns per thread
constexpr int CB_MAX_AZ = 8;       // tallest window
constexpr int CB_MAX_RG = 64;       // widest window
constexpr int CB_MAX_WIDTH = 1 << 28;   // widest raster (32-bit byte offsets in a row)

// 16-byte accesses at the samples' own alignment
typedef int BandI4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float BandF4 __attribute__((ext_vector_type(4), aligned(4)));

// products of the 4 samples, or sums of them
struct BandSum {
    float v[CB_PER_THREAD][4];   // Re(M S*), Im(M S*), |S|^2, |M|^2 per column
    __device__ __forceinline__ BandSum operator+(const BandSum& o) const
    {
        BandSum r;
#pragma unroll
        for (int j = 0; j < CB_PER_THREAD; j++)
#pragma unroll
            for (int k = 0; k < 4; k++) r.v[j][k] = v[j][k] + o.v[j][k];
        return r;
    }
};

// Azimuth sums over the WA latest rows.  push(p, q) takes row number q (mod
// kPeriod, a compile-time constant after unrolling) and returns the sum: rows
// a steps from the two ends in pairs, pairs in two halves.  The order depends
// neither on q nor on which end of the window came first, so a walk up and a
// walk down give the same bits.
template <int WA>
struct BandColumns {
    static constexpr int kPeriod = WA - 1;   // direct: the WA - 1 rows before this one
    static_assert(WA <= CB_MAX_AZ, "up to four terms");
    BandSum ring[WA - 1];
    __device__ __forceinline__ BandSum push(const BandSum& p, int q)
    {
        constexpr int D = WA - 1;
        constexpr int N = (WA + 1) / 2;   // terms: pairs, and the middle row of an odd WA
        const BandSum ends = p + ring[q % D];   // with the oldest
        ring[q % D] = p;
        auto term = [&](int a) {
            const BandSum& y = ring[(q + D - a) % D];
            return 2 * a == D ? y : y + ring[(q + a) % D];
        };
        if constexpr (N == 1) return ends;
        else if constexpr (N == 2) return ends + term(1);
        else if constexpr (N == 3) return ends + (term(1) + term(2));
        else return (ends + term(1)) + (term(2) + term(3));
    }
};
// pairs S2(r) = P(r) + P(r - 1): 4 lines are S2(r) + S2(r - 2)
template <>
struct BandColumns<4> {
    static constexpr int kPeriod = 2;
    BandSum last, s2[2];
    __device__ __forceinline__ BandSum push(const BandSum& p, int q)
    {
        const BandSum n = p + last, s = n + s2[q % 2];
        last = p;
        s2[q % 2] = n;
        return s;
    }
};
// 6 lines: S2(r) + S2(r - 4) + S2(r - 2)
template <>
struct BandColumns<6> {
    static constexpr int kPeriod = 4;
    BandSum last, s2[4];
    __device__ __forceinline__ BandSum push(const BandSum& p, int q)
    {
        const BandSum n = p + last, s = (n + s2[q % 4]) + s2[(q + 2) % 4];
        last = p;
        s2[q % 4] = n;
        return s;
    }
};
// 8 lines: quads S4(r) = S2(r) + S2(r - 2), S4(r) + S4(r - 4)
template <>
struct BandColumns<8> {
    static constexpr int kPeriod = 4;
    BandSum last, s2[2], s4[4];
    __device__ __forceinline__ BandSum push(const BandSum& p, int q)
    {
        const BandSum n = p + last, m = n + s2[q % 2], s = m + s4[q % 4];
        last = p;
        s2[q % 2] = n;
        s4[q % 4] = m;
        return s;
    }
};

// columns of a band of `threads` threads that hold whole windows, and its LDS
__host__ __device__ inline int coherence_band_cols(int threads, int win_rg)
{
    const int t = (CB_PER_THREAD * threads - CB_PER_THREAD + 1 - win_rg) / CB_PER_THREAD + 1;
    return CB_PER_THREAD * t;
}
inline size_t coherence_band_lds(int threads)
{
    // two row buffers of 4 running sums and a mask word per thread (and one
    // word past the last)
    return 2 * (size_t)threads * (4 * sizeof(float4) + sizeof(int)) + sizeof(int);
}

// a value the compiler takes as new: what is computed from it is formed where
// it is used instead of being held in registers across a loop
__device__ __forceinline__ int afresh(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

struct BandRaw {
    BandI4 m;
    BandF4 s0, s1;
};

// the thread's 4 samples of row gr, zero outside the raster; whole: all 4
// columns are inside
__device__ __forceinline__ void band_fetch(const tops_ci16* M, const tops_cf32* S, int w, int h,
                                           int gr, int ci, bool whole, BandRaw& raw)
{
    raw.m = BandI4{0, 0, 0, 0};
    raw.s0 = raw.s1 = BandF4{0.f, 0.f, 0.f, 0.f};
    if (gr < 0 || gr >= h) return;   // uniform
    ci = afresh(ci);   // (the row's base stays scalar)
    const tops_ci16* mr = M + (size_t)gr * w;
    const tops_cf32* sr = S + (size_t)gr * w;
    if (whole) {   // a uniform base and a 32-bit offset (w <= CB_MAX_WIDTH)
        const char* mq = reinterpret_cast<const char*>(mr);
        const char* sq = reinterpret_cast<const char*>(sr);
        raw.m = *reinterpret_cast<const BandI4*>(mq + (unsigned)ci * 4u);
        raw.s0 = *reinterpret_cast<const BandF4*>(sq + (unsigned)ci * 8u);
        raw.s1 = *reinterpret_cast<const BandF4*>(sq + (unsigned)ci * 8u + 16u);
        return;
    }
#pragma unroll
    for (int j = 0; j < CB_PER_THREAD; j++) {
        if (ci + j < 0 || ci + j >= w) continue;
        raw.m[j] = reinterpret_cast<const int*>(mr)[ci + j];
        const tops_cf32 v = sr[ci + j];
        if (j < 2) {
            raw.s0[2 * j] = v.x;
            raw.s0[2 * j + 1] = v.y;
        } else {
            raw.s1[2 * j - 4] = v.x;
            raw.s1[2 * j - 3] = v.y;
        }
    }
}

__device__ __forceinline__ BandSum band_products(const BandRaw& raw)
{
    BandSum p;
#pragma unroll
    for (int j = 0; j < CB_PER_THREAD; j++) {
        const float mr = (float)(short)(raw.m[j] & 0xffff), mi = (float)(short)(raw.m[j] >> 16);
        const float sr = j < 2 ? raw.s0[2 * j] : raw.s1[2 * j - 4];
        const float si = j < 2 ? raw.s0[2 * j + 1] : raw.s1[2 * j - 3];
        p.v[j][0] = mr * sr + mi * si;
        p.v[j][1] = mi * sr - mr * si;
        p.v[j][2] = sr * sr + si * si;
        p.v[j][3] = mr * mr + mi * mi;
    }
    return p;
}

__device__ __forceinline__ float4 band_col(const BandSum& s, int j)
{
    return make_float4(s.v[j][0], s.v[j][1], s.v[j][2], s.v[j][3]);
}

// The range sums of the thread's 4 windows from its column sums V: a row
// buffer E (4 arrays of NT running sums) is written, the NT threads wait, and
// those whose windows lie in the band read it.  E may be written again after
// the next barrier but one.  t: the thread's number among the NT.  (Arrays at
// compile-time distances: their addresses are immediates of one register.)
template <int NT>
struct BandRange {
    int kmin, a, off[CB_PER_THREAD];
    __device__ __forceinline__ void init(int win_rg)
    {
        kmin = win_rg >> 2;
        a = win_rg & 3;
#pragma unroll
        for (int j = 0; j < CB_PER_THREAD; j++) {
            const int i = max(j + a - 1, 0);   // (j + a = 0: no tail)
            off[j] = (i & 3) * NT + kmin + (i >> 2);
        }
    }
    __device__ __forceinline__ void write(const BandSum& V, float4* E, int t) const
    {
        float4 e = band_col(V, 0);
        E[t] = e;
#pragma unroll
        for (int j = 1; j < CB_PER_THREAD; j++) {
            e = add4(e, band_col(V, j));
            E[j * NT + t] = e;
        }
    }
    // f(j, sums of the window at column j), j = 3 .. 0: one window at a time,
    // so that few sums are held at once.  The window's ends are added to each
    // other and only then to its middle, which is two chains: few of the sums
    // are rounded at the size of the whole.  (RMS error of the coherence against
    // 64 bits, 6 x 24 / 8 x 32 windows: 5.4e-8 / 5.5e-8; 5.9e-8 / 6.2e-8 with
    // one chain from left to right, 5.5e-8 / 5.7e-8 in the tiles.)
    template <class F>
    __device__ __forceinline__ void sums(const BandSum& V, const float4* E, int t, F&& f) const
    {
        const float4* T = E + 3 * NT + t;
        float4 mid = make_float4(0.f, 0.f, 0.f, 0.f), odd = mid;
        int k = 1;
#pragma unroll 2
        for (; k + 1 < kmin; k += 2) {
            mid = add4(mid, T[k]);
            odd = add4(odd, T[k + 1]);
        }
        if (k < kmin) mid = add4(mid, T[k]);   // (uniform)
        mid = add4(mid, odd);
        __builtin_amdgcn_sched_barrier(0);
        float4 tail[CB_PER_THREAD], x = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int j = 0; j < CB_PER_THREAD; j++) tail[j] = E[t + off[j]];
        if (a >= 2) x = T[kmin];
        float4 s = band_col(V, CB_PER_THREAD - 1);
#pragma unroll
        for (int j = CB_PER_THREAD - 1; j >= 0; j--) {
            if (j < CB_PER_THREAD - 1) s = add4(band_col(V, j), s);
            float4 o = s;
            // (uniform branches)
            if (j > 0 || a) o = add4(o, tail[j]);
            if (j == 3 && a >= 2) o = add4(o, x);
            if (j == 2 && a == 3) o = add4(o, x);
            f(j, add4(o, mid));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// Output rows r0 .. r1-1 of the band that starts at column cb (a multiple of
// 4): its coherence_band_cols(NT, win_rg) columns.  up: from the last
// row to the first.  Row blocks alternate, so that two neighbours read the
// WA - 1 rows they share at about the same time, the second from a cache.
template <int WA, int NT>
__device__ __forceinline__ void coherence_band(const tops_ci16* M, const tops_cf32* S, int w, int h,
                                               float* coh, int dx, int dy, int win_rg, int cb,
                                               int r0, int r1, bool up, float4* smem)
{
    const int t = (int)threadIdx.x;
    int* mask = reinterpret_cast<int*>(smem + 8 * NT);
    const int ci = cb - dx + CB_PER_THREAD * t, co = cb + CB_PER_THREAD * t;
    const bool whole = ci >= 0 && ci + CB_PER_THREAD <= w;
    const bool out = CB_PER_THREAD * t < coherence_band_cols(NT, win_rg) && co < w;
    BandRange<NT> rg;
    rg.init(win_rg);
    // step i reads row first + step * i; the last WA rows read are the window
    // of output row (row read) + to_out, whose mask bits are `age` steps back
    const int n = r1 - r0 + WA - 1;
    const int step = up ? -1 : 1, first = up ? r1 - 1 - dy + WA - 1 : r0 - dy;
    const int to_out = up ? dy : dy - (WA - 1), age = 4 * (up ? dy : WA - 1 - dy);
    using Columns = BandColumns<WA>;
    Columns az;
    unsigned seen = 0;
    BandRaw nxt;
    band_fetch(M, S, w, h, first, ci, whole, nxt);
    for (int base = 0; base < n; base += Columns::kPeriod) {
#pragma unroll
        for (int q = 0; q < Columns::kPeriod; q++) {
            const int i = base + q, gr = first + step * i;
            if (i >= n) break;   // uniform
            const BandRaw cur = nxt;
            if (i + 1 < n) band_fetch(M, S, w, h, gr + step, ci, whole, nxt);
            const BandSum p = band_products(cur);
            seen <<= 4;
#pragma unroll
            for (int j = 0; j < CB_PER_THREAD; j++)
                seen |= amplitude_ok(p.v[j][2]) ? 1u << j : 0u;
            const BandSum V = az.push(p, q);
            __builtin_amdgcn_sched_barrier(0);
            if (i < WA - 1) continue;
            const int b = i & 1;
            float4* E = smem + b * 4 * NT;
            const int u = afresh(t);
            rg.write(V, E, u);
            mask[b * NT + u] = (int)(seen >> age & 15u);
            __syncthreads();
            if (!out) continue;
            const int* mk = mask + b * NT + u + (dx >> 2);
            const unsigned ok = (unsigned)(mk[0] | mk[1] << 4) >> (dx & 3);
            float z[CB_PER_THREAD];
            rg.sums(V, E, u, [&](int j, const float4& o) {
                z[j] = ok >> j & 1u ? coherence_of(o.x, o.y, o.z, o.w) : 0.0f;
            });
            float* row = coh + (size_t)(gr + to_out) * w;   // uniform
            float* dst = reinterpret_cast<float*>(reinterpret_cast<char*>(row) + (unsigned)co * 4u);
            if (co + CB_PER_THREAD <= w) {
                const BandF4 v = {z[0], z[1], z[2], z[3]};
                __builtin_nontemporal_store(v, reinterpret_cast<BandF4*>(dst));
            } else {
#pragma unroll
                for (int j = 0; j < CB_PER_THREAD; j++)
                    if (co + j < w) dst[j] = z[j];
            }
        }
    }
}

// f(std::integral_constant<int, win_az>) for win_az 2 .. CB_MAX_AZ
template <class F>
inline void band_dispatch(int win_az, F&& f)
{
    switch (win_az) {
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 5: f(std::integral_constant<int, 5>()); break;
    case 6: f(std::integral_constant<int, 6>()); break;
    case 7: f(std::integral_constant<int, 7>()); break;
    default: f(std::integral_constant<int, CB_MAX_AZ>()); break;
    }
}

}  // namespace tops
