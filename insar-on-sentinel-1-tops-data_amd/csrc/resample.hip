// resample.hip -- deramp -> 12x12 truncated-sinc resample -> reramp of one
// slave burst onto the master grid (gfx950).
//
// Semantics follow DerampAndResample.cu:108-183 (GetIndexes,
// DerampDemod_Shared) and 348-520 (Interpolation_12p):
//   slave line  y = poly(CpmAz; Ln, Pn) + AzShift, pixel x = poly(CpmRg; Ln, Pn)
//   (Iy, fy) = (trunc(y), int(frac*2047 + 0.5)), same for x
//   outside the slave box            -> 0
//   within 5 / 7 samples of its edge -> the sample at (Iy, Ix) (deramp and
//                                       reramp with the same phase cancel)
//   interior -> S = sum_j kL_j sum_i kP_i D(Iy-5+j, Ix-5+i),
//               Phi = sum_j kL_j sum_i kP_i phi(Iy-5+j, Ix-5+i),
//               out = S * exp(-j Phi)
// with D = slave * exp(j phi), phi(y, x) = -pi kt (ta - tref)^2 - 2 pi fdc ta,
// ta = (y - firstLine) * dt.
//
// Two implementations:
//   resample_fp64_*  plain all-FP64 per-stage form (deramp kernel writing an
//                    FP64 deramped burst + phase to HBM, then one thread per
//                    output reading 144+144 taps from HBM): the baseline.
//   resample_fast    fused column walker: each 64-lane wave walks a strip
//                    of output rows in groups of 4; every lane deramps one
//                    slave column on the fly (FP64 phasor recurrence, FP32
//                    samples), the azimuth sums of a group's distinct keys
//                    come from FP32 matrix instructions and are shared
//                    through LDS, and each output does its 12 range taps
//                    over those sums (FP32 MACs), takes its phase from the
//                    moment identity below (FP64) and reramps.
//
// Moment identity: phi is quadratic in the burst-relative line y for a fixed
// column, phi(y, x) = a(x) + b(x) y + c(x) y^2 with
//   a = -pi kt tref^2, b = 2 pi dt (kt tref - fdc), c = -pi kt dt^2.
// With y_j = y0 + (j - 5) and Mk = sum_j kL_j (j-5)^k (float LUT values in
// FP64), sum_j kL_j phi(y_j, x) = M0 a + (y0 M0 + M1) b + (y0^2 M0 + 2 y0 M1
// + M2) c exactly, so Phi needs three 12-tap FP64 range dot products.
#include "stream_access.hpp"
#include "tops_internal.hpp"
#include "walker.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

namespace tops {

// ======================================================================
// Plain all-FP64 form
// ======================================================================
__global__ void __launch_bounds__(256) deramp_fp64_kernel(ResampleParams p, double2* dre, double* ph)
{
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    int y = blockIdx.y;
    if (x >= p.s_pixels) return;
    int xa = p.sb[0] + x, ya = p.sb[2] + y;
    double phi = deramp_phase_direct(p, ya, xa);
    double sn, cs;
    sincos(phi, &sn, &cs);
    size_t q = (size_t)y * p.s_pixels + x;
    tops_ci16 s = p.slave[q];
    dre[q] = make_double2(s.re * cs - s.im * sn, s.re * sn + s.im * cs);
    ph[q] = phi;
}

__global__ void __launch_bounds__(256) resample_fp64_kernel(ResampleParams p, const double2* dre, const double* ph)
{
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    int r = blockIdx.y;
    if (c >= p.m_pixels) return;
    int iy, fy, ix, fx;
    slave_pos(p, r, c, iy, fy, ix, fx);
    int reg = region_of(p, iy, ix);
    tops_cf32 o = {0.0f, 0.0f};
    if (reg == 1) {
        size_t q = (size_t)(iy - p.sb[2]) * p.s_pixels + (ix - p.sb[0]);
        double2 d = dre[q];
        double sn, cs;
        sincos(ph[q], &sn, &cs);
        o.x = (float)(d.x * cs + d.y * sn);
        o.y = (float)(d.y * cs - d.x * sn);
    } else if (reg == 2) {
        const float* kl = p.kaz + fy * kTaps;
        const float* kp = p.krg + fx * kTaps;
        size_t base = (size_t)(iy - kHalf - p.sb[2]) * p.s_pixels + (ix - kHalf - p.sb[0]);
        double sr = 0.0, si = 0.0, sp = 0.0;
        for (int j = 0; j < kTaps; j++) {
            double tr = 0.0, ti = 0.0, tp = 0.0;
            const double2* drow = dre + base + (size_t)j * p.s_pixels;
            const double* prow = ph + base + (size_t)j * p.s_pixels;
            for (int i = 0; i < kTaps; i++) {
                double k = (double)kp[i];
                double2 d = drow[i];
                tr = fma(k, d.x, tr);
                ti = fma(k, d.y, ti);
                tp = fma(k, prow[i], tp);
            }
            double l = (double)kl[j];
            sr = fma(l, tr, sr);
            si = fma(l, ti, si);
            sp = fma(l, tp, sp);
        }
        double sn, cs;
        sincos(sp, &sn, &cs);
        o.x = (float)(sr * cs + si * sn);
        o.y = (float)(si * cs - sr * sn);
    }
    p.out[(size_t)r * p.m_pixels + c] = o;
}

int launch_resample_fp64(tops_ctx* ctx, const ResampleParams& p, hipStream_t s)
{
    size_t n = (size_t)p.s_lines * p.s_pixels;
    size_t need = n * (sizeof(double2) + sizeof(double));
    int rc = ctx->scratch.ensure(need);
    if (rc) return rc;
    double2* dre = (double2*)ctx->scratch.ptr;
    double* ph = (double*)(dre + n);
    dim3 g1((p.s_pixels + 255) / 256, p.s_lines);
    hipLaunchKernelGGL(deramp_fp64_kernel, g1, dim3(256), 0, s, p, dre, (double*)ph);
    TOPS_HIP(hipGetLastError());
    dim3 g2((p.m_pixels + 255) / 256, p.m_lines);
    hipLaunchKernelGGL(resample_fp64_kernel, g2, dim3(256), 0, s, p, (const double2*)dre,
                       (const double*)ph);
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

// Fused fast form: column-walking waves
// ======================================================================
// One 64-lane workgroup owns a strip of output rows x WK_OUT output columns.
// Lane l is bound to slave column ucol0 + l for the whole strip and walks it
// in groups of output rows:
//   * it keeps the deramped slave samples of rows wbase..wbase+15 (+19 where
//     lines advance unevenly) of its column in registers; new rows are deramped on arrival with an FP64
//     phasor recurrence along the column (exp(j phi) is advanced by
//     exp(j (b + c (2y+1))), which is advanced by exp(j 2c)), anchored with
//     an FP64 sincos at the strip start and after a resync;
//   * the positions of all rows of the group come first, then their distinct
//     azimuth keys (Iy, fy): up to WK_SLOTS per row and round;
//   * per row and key it forms the 12-tap azimuth sum U of its column and
//     writes it to LDS;
//   * each output then needs only its own 12 range taps over U, and its
//     phase.
// Outputs that the shared pass cannot serve (a range window outside the strip's
// 64 columns, a key out of the window's reach at all its positions) are computed
// by interior_direct.
//
// Why groups: one row at a time is a chain of dependent latencies (position
// -> keys -> tap loads -> LDS exchange -> range sums) and of scalar loads that
// the resident waves do not cover; four rows go through it together, and four
// rows are what a 4x4x1 matrix instruction takes.
//
// What bounds it: vector issue, about three quarters of the time (one IW
// burst, 1500 x 21000, moves 0.38 GB: 60 us of memory time).  Measured there,
// on one GPU: 233 us, against 292-335 for the row-at-a-time walker with scalar
// tap loads and 12 FP64 phases an output (265-273 before the launch ended in low
// strips and the azimuth shift was a scalar load).  3 waves per SIMD (161
// VGPRs): 2 take 238 us; at 4 the registers spill into the row loop (266); at 6
// to 9, with a wave pair sharing a strip, 307 to 608 at the 265 us stage.
//
// The phase.  Phi is the 12 x 12 tap sum of phi(y, x) = a(x) + b(x) y +
// c(x) y^2.  Over a strip's 64 columns a, b and c are cubics of the column to
// their own FP64 rounding (they come from quadratic Doppler centroid and FM rate
// polynomials), so the range sum collapses to the tap moments of the output's
// LUT row as the azimuth sum does (walk kSmooth): 10 FP64 operations an output
// instead of 24 and 12 LDS reads (a quadratic fit leaves out up to 1e-8 rad at
// 2000 columns a burst and 5e-7 at 320; it took 231 us here, and bursts below 700
// columns the column sums: 1500 x 500 60 us, now 35).  The strip checks its own
// arrays: on every
// slave line every column's residual from the cubic through four of its columns
// must stay below a bound of the order of the FP64 sum's rounding (fit_phase);
// otherwise it sums the 12 columns' FP64 phases.

constexpr int WK_GROUP = 4;           // output rows per group (one matrix-instruction block)
constexpr int WK_SLOTS = 2;           // azimuth keys per row and round
constexpr int WK_LONG = 20;           // lines of the window where lines do not advance evenly
// What the fitted phase may leave out: 2^-32 rad and 2^-47 of the size of the
// phase's terms, a few roundings of the FP64 sum it takes the place of, and
// never more than half an ulp of an FP32 sample of magnitude 1
constexpr double kSmoothTol = 0x1p-32, kSmoothRel = 0x1p-47, kSmoothMax = 0x1p-25;

struct WalkLds {
    // azimuth sums U: [row * WK_SLOTS + slot][column]; the general form holds
    // one slot per row in the first half and the azimuth-interpolated phases
    // in the second
    float2 u[WK_GROUP * WK_SLOTS][64];
    double rowt[32][6];         // row-uniform position terms of 32 rows
    double pos[5][64];          // per lane: Pn, c2 Pn and c5 Pn Pn of both polynomials
    double ph[WK_GROUP][WK_SLOTS][6];  // smooth: the row's phase per key as a cubic of the column
    double abc[3][64];          // per lane: the column's phase coefficients a, b, c
    double fit[3][4];           // smooth: a(x), b(x), c(x) in revolutions, cubics of t, the
                                // column less that of the 6th tap of the first servable window
};
static_assert(sizeof(WalkLds) <= 10240, "16 workgroups per CU");

__device__ __forceinline__ double lane_value(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// 1 / n from the hardware's estimate (23 bits) in two Newton steps
__device__ __forceinline__ double recip(int n)
{
    const double x = (double)n;
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// Fits the strip's phase coefficients into sm.fit, each the cubic through its
// values at four columns near the Chebyshev places (false: not smooth enough on
// the slave box's lines, which hold every interior output's).
__device__ __forceinline__ bool fit_phase(const ResampleParams& p, WalkLds& sm, int ucol0)
{
    const int lane = threadIdx.x;
    const int l0 = max(0, p.sb[0] - ucol0), l1 = min(63, p.sb[1] - ucol0);
    const int span = l1 - l0;
    if (span < 3 || !p.krg_unit) return false;
    const int out = (span * 5 + 64) >> 7, in = (span * 79 + 128) >> 8;
    const int t0 = l0 + out, t1 = l0 + in, t2 = l1 - in, t3 = l1 - out;
    const double x0 = (double)(lane - t0), x1 = (double)(lane - t1), x2 = (double)(lane - t2);
    // the column of t = 0, from the places
    const double a0 = (double)(l0 + kHalf - t0), a1 = (double)(l0 + kHalf - t1);
    const double a2 = (double)(l0 + kHalf - t2);
    const double ro = recip(t1 - t0), ri = recip(t2 - t1), r2 = recip(t2 - t0), r3 = recip(t3 - t0);
    // What the fit leaves out of the phase is a quadratic of the line: its values
    // at the ends and the middle of the box bound it within a factor 1.25 in
    // between.  It is each lane's residual, and the third moment of the taps
    // (below 1) times the cubic's leading coefficient and the rounding of their
    // second, which are the strip's: a lane takes them at one of the three lines.
    const double y0 = (double)p.sb[2] - (double)p.first_line;
    const double y2 = (double)p.sb[3] - (double)p.first_line, y1 = 0.5 * (y0 + y2);
    const double ym = fmax(fabs(y0), fabs(y2)), yl = lane & 2 ? y2 : lane & 1 ? y1 : y0;
    double e0 = 0.0, e1 = 0.0, e2 = 0.0, third = 0.0, second = 0.0, size = 0.0;
    double s0 = 1.0, s1 = 1.0, s2 = 1.0, sl = 1.0, sz = 1.0;
#pragma unroll 1
    for (int k = 0; k < 3; k++) {
        const double v = sm.abc[k][lane];
        const double f0 = lane_value(v, t0), f1 = lane_value(v, t1), f2 = lane_value(v, t2);
        const double d01 = (f1 - f0) * ro, d12 = (f2 - f1) * ri, d23 = (lane_value(v, t3) - f2) * ro;
        const double d02 = (d12 - d01) * r2, d3 = ((d23 - d12) * r2 - d02) * r3;
        // f0 + (x - t0)(d01 + (x - t1)(d02 + (x - t2) d3)) about t = 0
        const double u = fma(a2, d3, d02), w = fma(a1, d3, u), c2 = fma(a0, d3, w);
        const double z = fma(a1, u, d01);
        sm.fit[k][0] = fma(a0, z, f0) * kInvTwoPi;
        sm.fit[k][1] = fma(a0, w, z) * kInvTwoPi;
        sm.fit[k][2] = c2 * kInvTwoPi;
        sm.fit[k][3] = d3 * kInvTwoPi;
        const double res = v - fma(x0, fma(x1, fma(x2, d3, d02), d01), f0);
        e0 = fma(s0, res, e0);
        e1 = fma(s1, res, e1);
        e2 = fma(s2, res, e2);
        third = fma(sl, d3, third);
        second = fma(sl, c2, second);
        size = fma(sz, fabs(v), size);
        s0 *= y0;
        s1 *= y1;
        s2 *= y2;
        sl *= yl;
        sz *= ym;
    }
    const double tol = fmin(kSmoothTol + kSmoothRel * size, kSmoothMax);
    const double r = 2.5 * fmax(fmax(fabs(e0), fmax(fabs(e1), fabs(e2))),
                                fma(0x1p-24, fabs(second), fabs(third)));
    // (fmax drops a NaN: the sum keeps it, and a NaN fails the comparison)
    const double nan = 0.0 * (e0 + e1 + e2 + third + second);
    return __ballot(lane >= l0 && lane <= l1 && !(r + nan <= tol)) == 0ull;
}

// The mark of an interior output left to the direct path, in its place in the
// output until the strip ends.  (Any output that holds these bits is formed
// by the direct path, so an equal result would only be formed twice.)
__device__ __forceinline__ tops_cf32 unserved()
{
    return {__uint_as_float(0x7fc5a17eu), __uint_as_float(0x7fc0de1au)};
}
__device__ __forceinline__ bool is_unserved(const tops_cf32& v)
{
    return __float_as_uint(v.x) == 0x7fc5a17eu && __float_as_uint(v.y) == 0x7fc0de1au;
}

typedef float MfmaAcc __attribute__((ext_vector_type(4)));

// U of 4 output rows in every column: acc[i] += sum_k wt(row i, line k)
// win[k].  The taps of all four rows sit in one register (lane 4 k + i: row
// i, window line k); the 4x4x1 matrix instruction broadcasts block k of it to
// all 16 blocks (cbsz 4, abid k) and multiplies it with the window line held
// one column per lane, which is the walker's own layout.  Each step is an
// FP32 fused multiply-add per element in line order, bit-equal to the
// scalar-tap chain fmaf(tap, win, acc).
// (lines 16 on of a longer window in a second register)
template <int K, int S, int N, int T>
struct AzStep {
    __device__ __forceinline__ static void run(const WinRow (&win)[N], const float (&wt)[T][WK_SLOTS],
                                               MfmaAcc (&re)[S], MfmaAcc (&im)[S])
    {
        AzStep<K - 1, S, N, T>::run(win, wt, re, im);
#pragma unroll
        for (int s = 0; s < S; s++) {
            re[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(wt[K / 16][s], win_re(win[K]), re[s], 4, K % 16, 0);
            im[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(wt[K / 16][s], win_im(win[K]), im[s], 4, K % 16, 0);
        }
    }
};
template <int S, int N, int T>
struct AzStep<-1, S, N, T> {
    __device__ __forceinline__ static void run(const WinRow (&)[N], const float (&)[T][WK_SLOTS],
                                               MfmaAcc (&)[S], MfmaAcc (&)[S]) {}
};

// v truncated toward zero, saturated (the conversion instruction's own
// result; a NaN gives 0)
__device__ __forceinline__ int trunc_i32(double v)
{
    int r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// the largest value of the wave (uniform; values 0 .. INT_MAX): 0 is what a
// lane without a source reads
__device__ __forceinline__ int wave_max(int v)
{
    unsigned u = (unsigned)v;
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x111, 0xf, 0xf, true));    // row_shr:1
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x112, 0xf, 0xf, true));    // row_shr:2
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x114, 0xf, 0xf, true));    // row_shr:4
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x118, 0xf, 0xf, true));    // row_shr:8
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x142, 0xa, 0xf, false));   // row_bcast:15
    u = max(u, (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x143, 0xc, 0xf, false));   // row_bcast:31
    return __builtin_amdgcn_readlane((int)u, 63);
}
__device__ __forceinline__ int wave_min(int v) { return wave_max(v ^ INT_MAX) ^ INT_MAX; }

// value k[lane & 3] of four uniform values
__device__ __forceinline__ int by_row(int k0, int k1, int k2, int k3, bool b0, bool b1)
{
    const int lo = b0 ? k1 : k0, hi = b0 ? k3 : k2;
    return b1 ? hi : lo;
}

// Output rows r0 .. r1-1 of the strip whose lane 0 is output column c0 and
// slave column ucol0, in groups of 4.  kSmooth: the fitted phase; otherwise
// FP64 phases per column.  kEven: the slave line advances by about one a row
// and hardly along it, so that the window slides by 4 lines from group to group
// and reaches all of a group's keys; the few outputs it does not reach are left
// to the direct path.  Otherwise the window is 4 lines longer, slides by any
// number of lines, and to further positions for keys it does not reach: that
// would cost even rows 8 % (1500 x 12000: 164 us and 177).
template <bool kSmooth, bool kEven>
__device__ __forceinline__ void walk_rows(const ResampleParams& p, int c0, int r0, int r1,
                                          int ucol0, ColumnWalker& w, WalkLds& sm)
{
    constexpr int G = WK_GROUP;
    constexpr int S = kSmooth ? WK_SLOTS : 1;   // azimuth keys per row and round
    constexpr int N = kEven ? WK_WIN : WK_LONG;  // lines of the window
    constexpr int kReach = N - kTaps;           // lines past the window's first a key may start at
    static_assert(kAzShifts == WK_WIN - kTaps + 1, "the table's tap offsets");
    constexpr int kWaveShr1 = 0x138;            // DPP: the value of the lane to the left
    constexpr int kMaxSlide = 20;               // lines the window slides rather than start anew
    constexpr int kMaxMoves = 16;               // window positions after a group's first
    static_assert(32 % G == 0, "the row table is refreshed between groups");
    const int lane = threadIdx.x;
    const int c = c0 + lane;
    const unsigned long long out_mask = __builtin_amdgcn_ballot_w64(lane < WK_OUT && c < p.m_pixels);
    double (*pu)[64] = reinterpret_cast<double (*)[64]>(sm.u[WK_GROUP]);   // general form
    const double azs = az_shift_of(p);
    const bool b0 = lane & 1, b1 = lane & 2;
    // lines interior to the slave box (region_of): ylo .. ylo + yn.  Columns
    // interior to it whose 12 taps are lanes of the strip: xlo .. xlo + xn, the
    // first tap on lane xlo - kHalf - ucol0.  (none: no output can be served)
    const int ylo = p.sb[2] + kHalf, yn = p.sb[3] - kHalf - 2 - ylo;
    const int xlo = max(ucol0, p.sb[0]) + kHalf;
    const int xn = min(ucol0 + 64 - kTaps + kHalf, p.sb[1] - kHalf - 2) - xlo;
    const bool none = yn < 0 || xn < 0;
    const float2* u0 = &sm.u[0][none ? 0 : xlo - kHalf - ucol0];
    WinRow win[N];
    int wbase = INT_MIN;           // absolute slave line held in win[0]
    bool late = false;             // outputs are marked for the direct path (uniform)
    // A group takes one round of up to S keys per row, or further rounds
    // (again) where a row segment holds more, or its keys are further apart than
    // the window reaches; a round keeps the positions.
    // key: line * 2048 + LUT row of an output the shared pass may serve
    // (INT_MAX: none); fxo: byte offset of its range LUT row; xt: its first
    // tap's lane, from u0; heads: the lanes that list the row's keys not yet
    // taken; need: outputs not formed yet.
    int key[G], fxo[G], xt[G], line0 = 0;
    unsigned long long heads[G], need[G];
    bool again = false;
    bool place = true;   // !kEven: the window is to be placed
    int moves = 0;       // and its positions since the group's first
    for (int r = r0; r < r1;) {
        if (!again) {
            // ---- row-uniform position terms, 32 rows at a time (one per lane)
            const int rr = (r - r0) & 31;
            if (__builtin_expect(rr == 0, 0)) {
                __syncthreads();
                const int rl = r + lane;
                if (lane < 32) {
#pragma clang fp contract(off)
                    const double ln = norm_warp((double)(p.mb[2] + rl), (double)p.mb[2],
                                                (double)p.mb[3]);
                    sm.rowt[lane][0] = p.cpm_az[0] + p.cpm_az[1] * ln;
                    sm.rowt[lane][1] = p.cpm_az[3] * ln * ln;
                    sm.rowt[lane][2] = p.cpm_az[4] * ln;
                    sm.rowt[lane][3] = p.cpm_rg[0] + p.cpm_rg[1] * ln;
                    sm.rowt[lane][4] = p.cpm_rg[3] * ln * ln;
                    sm.rowt[lane][5] = p.cpm_rg[4] * ln;
                }
                __syncthreads();
            }

            // ---- this lane's output positions.  An interior position is
            // positive, so its fraction is v - floor(v), exactly v - (int)v.
            {
#pragma clang fp contract(off)
                const double pn = sm.pos[0][lane], q1 = sm.pos[1][lane], q2 = sm.pos[2][lane];
                const double q3 = sm.pos[3][lane], q4 = sm.pos[4][lane];
#pragma unroll
                for (int i = 0; i < G; i++) {
                    const double2* t2 = reinterpret_cast<const double2*>(sm.rowt[rr + i]);
                    const double2 ta = t2[0], tb = t2[1], td = t2[2];
                    const double ys = ta.x + q1 + ta.y + tb.x * pn + q2 + azs;
                    const double xs = tb.y + q3 + td.x + td.y * pn + q4;
                    const int iy = trunc_i32(ys), dx = trunc_i32(xs) - xlo;
                    const int fy = trunc_i32(__builtin_amdgcn_fract(ys) * kInterval + 0.5);
                    const int fx = trunc_i32(__builtin_amdgcn_fract(xs) * kInterval + 0.5);
                    need[i] = r + i < r1 ? out_mask : 0ull;
                    const bool servable = __builtin_amdgcn_inverse_ballot_w64(
                        (none ? 0ull : need[i]) &
                        __builtin_amdgcn_ballot_w64((unsigned)(iy - ylo) <= (unsigned)yn) &
                        __builtin_amdgcn_ballot_w64((unsigned)dx <= (unsigned)xn));
                    static_assert(kLutRows == 2048, "key packing");
                    key[i] = servable ? iy * kLutRows + fy : INT_MAX;
                    fxo[i] = fx * (int)(kKrgxRow * sizeof(float));
                    xt[i] = servable ? dx : 0;
                    // formed here, not where they are used
                    asm volatile("" : "+v"(key[i]), "+v"(fxo[i]), "+v"(xt[i]));
                    if (i & 1) __builtin_amdgcn_sched_barrier(0);
                }
            }
            // ---- distinct azimuth keys of each row.  Keys change slowly
            // along a row, so a key is listed at each lane where it differs
            // from the lane to its left.  Keys have 0 <= line < 2^20
            // (interior rows of a slave box checked at launch).
#pragma unroll
            for (int i = 0; i < G; i++) {
                const int kleft = __builtin_amdgcn_update_dpp(~key[i], key[i], kWaveShr1, 0xf, 0xf,
                                                              false);
                heads[i] = __builtin_amdgcn_ballot_w64(key[i] != INT_MAX) &
                           __builtin_amdgcn_ballot_w64(kleft != key[i]);
            }
            // the group's first line among its keys
            line0 = wave_min(min(min(key[0], key[1]), min(key[2], key[3]))) >> 11;
        }
        if (line0 != INT_MAX >> 11) {
            int wline = line0;   // the first line a key may start at
            int slide = 0, steps = 0;
            if constexpr (!kEven) {
                // the window is to hold lines line0-5 onwards: it slides by
                // fours (-1: starts anew), and by single lines too where that
                // reaches further keys
                if (place) {
                    slide = wbase == INT_MIN ? -1 : line0 - kHalf - wbase;
                    if (slide >= 0 && slide <= kMaxSlide) {
                        int last = 0;
#pragma unroll
                        for (int i = 0; i < G; i++)
                            last = max(last, key[i] == INT_MAX ? 0 : key[i]);
                        if ((wave_max(last) >> 11) - line0 + (slide & 3) > kReach) steps = slide & 3;
                        wbase = line0 - kHalf - (slide & 3) + steps;
                        slide >>= 2;
                    } else {
                        slide = -1;
                        wbase = line0 - kHalf;
                    }
                    place = false;
                }
                wline = wbase + kHalf;
            }
            // ---- this round's keys (uniform; -1: none).  A key whose
            // lines lie beyond the window's reach is left to its next position
            // (kEven: to the direct path).  A key that reappears further along the
            // row is served by its first slot.
            // (no head left reads lane 63, which owns no output)
            int kq[G][S];
            // (no line reaches kMaxSlaveLine)
            const int lim = min(wline + kReach, kMaxSlaveLine - 1) << 11 | (kLutRows - 1);
#pragma unroll
            for (int i = 0; i < G; i++) {
#pragma unroll
                for (int s = 0; s < S; s++) {
                    const unsigned long long h = heads[i];
                    const int k = __builtin_amdgcn_readlane(key[i], __builtin_ctzll(h | 1ull << 63));
                    kq[i][s] = k <= lim ? k : -1;
                    heads[i] = h & (h - 1);
                }
            }
            bool second = false;
            if (S == 2)
                second = (kq[0][S - 1] & kq[1][S - 1] & kq[2][S - 1] & kq[3][S - 1]) != -1;
            // the round's table loads first, so that the window's slide
            // covers their latency.  wt: lane 4 k + i holds row i's tap at
            // window line k (the key's 12 taps pre-shifted by its line
            // offset, zeros elsewhere)
            int kr[S];
            float wt[kEven ? 1 : 2][WK_SLOTS];
#pragma unroll
            for (int s = 0; s < S; s++) {
                kr[s] = by_row(kq[0][s], kq[1][s], kq[2][s], kq[3][s], b0, b1);
                if (kr[s] < 0) kr[s] = wline << 11;
                const int o = (kr[s] >> 11) - wline, row = kr[s] & (kLutRows - 1);
                if constexpr (kEven) {
                    wt[0][s] = p.kaz_sh[(o * kLutRows + row) * kAzShiftTaps + (lane >> 2)];
                } else {
                    const int k0 = (lane >> 2) - o, k1 = k0 + 16;
                    wt[0][s] = (unsigned)k0 < (unsigned)kTaps ? p.kaz[row * kTaps + k0] : 0.0f;
                    wt[1][s] = (unsigned)k1 < (unsigned)kTaps ? p.kaz[row * kTaps + k1] : 0.0f;
                }
            }
            float4 tap[2][4];
            auto load_range = [&](int i) {
                const float4* q = reinterpret_cast<const float4*>(
                    reinterpret_cast<const char*>(p.krgx) + (unsigned)fxo[i]);
#pragma unroll
                for (int k = 0; k < 4; k++) tap[i & 1][k] = q[k];
            };
            if (lane < WK_OUT) load_range(0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!kEven) {
                if (__builtin_expect(slide < 0, 0)) {
                    w.anchor(p, wbase, sm.abc[0][lane], sm.abc[1][lane], sm.abc[2][lane]);
                    int raw[N];
#pragma unroll
                    for (int k = 0; k < N; k++) raw[k] = w.fetch(p, wbase + k);
#pragma unroll
                    for (int k = 0; k < N; k++) win[k] = win_pack(w.deramp(raw[k]));
                    w.prefetch(p);
                } else {
                    for (; slide > 0; slide--) slide4(win, w, p);
                    for (; steps > 0; steps--) slide1(win, w, p);
                }
            } else if (!again) {
                // the window holds lines wbase .. wbase+15; lines line0-5
                // onwards are wanted.  It slides by 4 lines, which is what 4
                // output rows advance by; positions that advance otherwise (a
                // whole-line contour of the offset field, once per crossing)
                // start it anew.
                const int o = wbase == INT_MIN ? -1 : line0 - kHalf - wbase;
                if (o == 4) {
                    slide4(win, w, p);
                } else if (__builtin_expect(o != 0, 0)) {
                    w.anchor(p, line0 - kHalf, sm.abc[0][lane], sm.abc[1][lane], sm.abc[2][lane]);
                    int raw[WK_WIN];
#pragma unroll
                    for (int k = 0; k < WK_WIN; k++) raw[k] = w.fetch(p, line0 - kHalf + k);
#pragma unroll
                    for (int k = 0; k < WK_WIN; k++) win[k] = win_pack(w.deramp(raw[k]));
                    w.prefetch(p);
                }
                wbase = line0 - kHalf;
            }
            if (kSmooth && second) {
                // (four independent chains: no wait between dependent steps)
                MfmaAcc re[2] = {}, im[2] = {};
                AzStep<N - 1, 2, N, kEven ? 1 : 2>::run(win, wt, re, im);
#pragma unroll
                for (int i = 0; i < G; i++) {
                    sm.u[i * S][lane] = make_float2(re[0][i], im[0][i]);
                    sm.u[i * S + S - 1][lane] = make_float2(re[1][i], im[1][i]);
                }
            } else {
                MfmaAcc re[1] = {}, im[1] = {};
                AzStep<N - 1, 1, N, kEven ? 1 : 2>::run(win, wt, re, im);
#pragma unroll
                for (int i = 0; i < G; i++) sm.u[i * S][lane] = make_float2(re[0][i], im[0][i]);
            }
            if (!kSmooth) {
#pragma unroll 1
                for (int i = 0; i < G; i++) {
                    const int kk = __builtin_amdgcn_readlane(kr[0], i);
                    CDouble* mq = (CDouble*)(p.mom + 4 * (kk & (kLutRows - 1)));
                    const double m0 = mq[0], m1 = mq[1], m2 = mq[2];
                    const double y0 = (double)((kk >> 11) - p.first_line);
                    const double bq = fma(y0, m0, m1);
                    const double cq = y0 * y0 * m0 + 2.0 * y0 * m1 + m2;
                    pu[i][lane] = fma(m0, sm.abc[0][lane],
                                      fma(bq, sm.abc[1][lane], cq * sm.abc[2][lane]));
                }
            }
            if (kSmooth) {
                // lane 4 s + i: the phase of row i and slot s, P0 + P1 t + P2
                // t^2 + P3 t^3 over t = column of the 6th tap less the one of
                // xt = 0, in revolutions, and 3 P3
                const int kl = lane < G ? kr[0] : kr[S - 1];
                if (lane < G * S) {
                    const double4 m = reinterpret_cast<const double4*>(p.mom)[kl & (kLutRows - 1)];
                    const double y0 = (double)((kl >> 11) - p.first_line);
                    const double n1 = fma(y0, m.x, m.y);
                    const double n2 = y0 * y0 * m.x + 2.0 * y0 * m.y + m.z;
                    double* q = sm.ph[lane & 3][lane >> 2];
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        q[k] = fma(m.x, sm.fit[0][k], fma(n1, sm.fit[1][k], n2 * sm.fit[2][k]));
                    q[4] = 3.0 * q[3];
                }
            }
            __syncthreads();
            // ---- each output's 12 range taps over U, its phase, the reramp:
            // formed for every output lane, stored for the outputs served.
            // The stores come last: memory operations complete in order, so a
            // table load behind a store would wait for the store too
            tops_cf32 z[G];
            unsigned long long mine[G];
#pragma unroll
            for (int i = 0; i < G; i++) {
                mine[i] = need[i] & (__builtin_amdgcn_ballot_w64(key[i] == kq[i][0]) |
                                     __builtin_amdgcn_ballot_w64(key[i] == kq[i][S - 1]));
                need[i] &= ~mine[i];
            }
            if (lane < WK_OUT) {
#pragma unroll
            for (int i = 0; i < G; i++) {
                const bool s1 = S == 2 && key[i] == kq[i][S - 1];
                if (i + 1 < G) load_range(i + 1);   // the next row's taps
                __builtin_amdgcn_sched_barrier(0);
                if (!kEven && mine[i] == 0ull) continue;   // (uniform)
                const float4 k0 = tap[i & 1][0], k1 = tap[i & 1][1], k2 = tap[i & 1][2];
                const float4 km = tap[i & 1][3];
                const float kp[kTaps] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y,
                                         k1.z, k1.w, k2.x, k2.y, k2.z, k2.w};
                const float2* u = u0 + i * S * 64 + xt[i] + (s1 ? 64 : 0);
                float sr = 0.f, si = 0.f;
                // (the LDS reads of 6 taps are issued together before their
                // sums; all 12 at once would spill)
                static_assert(kTaps % 6 == 0, "tap groups of 6");
#pragma unroll
                for (int h = 0; h < kTaps; h += 6) {
                    float2 v[6];
#pragma unroll
                    for (int k = 0; k < 6; k++) v[k] = u[h + k];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 6; k++) {
                        sr = fmaf(kp[h + k], v[k].x, sr);
                        si = fmaf(kp[h + k], v[k].y, si);
                    }
                }
                double ph;
                if (kSmooth) {
                    // sum_k kp P(t + k - 5): with the LUT row's sum 1 + e0, mean
                    // offset mu and second moment about it, v, this is
                    // (1 + e0) P(x) + v P''(x) / 2 at x = t + mu (the third
                    // moment is left out: fit_phase)
                    const double* q = sm.ph[i][s1 ? 1 : 0];
                    const double P0 = q[0], P1 = q[1], P2 = q[2], P3 = q[3], P3x3 = q[4];
                    const double x = (double)xt[i] +
                                     __hiloint2double(__float_as_int(km.y), __float_as_int(km.x));
                    const double Q = fma(x, fma(x, fma(x, P3, P2), P1), P0);
                    ph = fma((double)km.w, fma(x, P3x3, P2), fma((double)km.z, Q, Q));
                } else {
                    const double* pl = reinterpret_cast<const double*>(u0) + (WK_GROUP + i) * 64 + xt[i];
                    ph = 0.0;
#pragma unroll
                    for (int k = 0; k < kTaps; k++) ph = fma((double)kp[k], pl[k], ph);
                    ph *= kInvTwoPi;
                }
                z[i] = reramp_rev(sr, si, ph);
                asm volatile("" : "+v"(z[i].x), "+v"(z[i].y));
                __builtin_amdgcn_sched_barrier(0);
            }
            }
            // written once: nontemporal stores
#pragma unroll
            for (int i = 0; i < G; i++)
                if (__builtin_amdgcn_inverse_ballot_w64(mine[i]))
                    stream_store_float2(p.out + (size_t)(r + i) * p.m_pixels + (unsigned)c, z[i].x,
                                        z[i].y);
            __syncthreads();   // LDS is rewritten by the next round or group
            again = (heads[0] | heads[1] | heads[2] | heads[3]) != 0ull;
        }
        if (__builtin_expect(again, 0)) continue;
        if constexpr (!kEven) place = true;

        // ---- the outputs no round served: outside the box (0), in its edge
        // band (the sample itself), or marked for the direct path.  The four
        // rows together: edge strips would otherwise wait for one load a row
        // and end long after the others
        if (__builtin_expect((need[0] | need[1] | need[2] | need[3]) != 0ull, 0)) {
            if constexpr (!kEven) {
                // keys beyond the window's reach first: rounds at its next position
                unsigned long long far[G];
#pragma unroll
                for (int i = 0; i < G; i++)
                    far[i] = need[i] & __builtin_amdgcn_ballot_w64(key[i] != INT_MAX);
                if ((far[0] | far[1] | far[2] | far[3]) != 0ull && moves < kMaxMoves) {
                    int first = INT_MAX;
#pragma unroll
                    for (int i = 0; i < G; i++) {
                        first = min(first,
                                    __builtin_amdgcn_inverse_ballot_w64(far[i]) ? key[i] : INT_MAX);
                        const int kleft = __builtin_amdgcn_update_dpp(~key[i], key[i], kWaveShr1,
                                                                      0xf, 0xf, false);
                        heads[i] = far[i] & __builtin_amdgcn_ballot_w64(kleft != key[i]);
                    }
                    line0 = wave_min(first) >> 11;
                    again = place = true;
                    moves++;
                    continue;
                }
            }
            int reg[G];
            tops_ci16 v[G];
#pragma unroll
            for (int i = 0; i < G; i++) {
                int iy, fy, ix, fx;
                slave_pos(p, r + i, c, iy, fy, ix, fx);
                reg[i] = need[i] >> lane & 1 ? region_of(p, iy, ix) : -1;
                v[i] = {0, 0};
                if (reg[i] == 1)
                    v[i] = p.slave[(size_t)(iy - p.sb[2]) * p.s_pixels + (ix - p.sb[0])];
            }
#pragma unroll
            for (int i = 0; i < G; i++) {
                if (__builtin_amdgcn_ballot_w64(reg[i] == 2) != 0ull) late = true;
                tops_cf32 o = {(float)v[i].re, (float)v[i].im};
                if (reg[i] == 2) o = unserved();
                if (reg[i] >= 0)
                    stream_store_float2(p.out + (size_t)(r + i) * p.m_pixels + (unsigned)c, o.x, o.y);
            }
        }
        if constexpr (!kEven) moves = 0;
        r += G;
    }

    // ---- the direct path (outside the row loop: its registers would spill)
    if (__builtin_expect(late, 0)) {
        __threadfence();
        for (int r = r0; r < r1; r++) {
            if (!__builtin_amdgcn_inverse_ballot_w64(out_mask)) continue;
            tops_cf32* q = p.out + (size_t)r * p.m_pixels + (unsigned)c;
            if (!is_unserved(*q)) continue;
            int iy, fy, ix, fx;
            slave_pos(p, r, c, iy, fy, ix, fx);
            if (region_of(p, iy, ix) != 2) continue;
            const tops_cf32 o = interior_direct(p.slave, p.kt, p.tref, p.fdc, p.mom, p.kaz, p.krg,
                                                p.s_pixels, p.sb[0], p.sb[2], p.first_line, p.dt,
                                                iy, fy, ix, fx);
            stream_store_float2(q, o.x, o.y);
        }
    }
}

// One strip of one burst: output columns sx*WK_OUT .. +WK_OUT-1, output rows
// r0 .. r1-1 of the master box.  p may live in global memory (batched
// launches): its fields are wave-uniform.
template <bool kEven>
__device__ __forceinline__ void resample_strip(const ResampleParams& p, int sx, int r0, int r1,
                                               WalkLds& sm)
{
    const int lane = threadIdx.x;
    const int c0 = sx * WK_OUT;
    const int c = c0 + lane;

    // Position polynomial (polyval6 order, contraction off), split into
    //   ys = ((((A + c2 Pn) + B) + D Pn) + c5 Pn Pn) + AzShift
    // with A = c0 + c1 Ln, B = c3 Ln Ln, D = c4 Ln uniform over a row and
    // c2 Pn, c5 Pn Pn fixed per lane: the same operations in the same order.
    // (kept in LDS, read once per group: registers are the walker's limit)
    {
#pragma clang fp contract(off)
        const double pn = norm_warp((double)(p.mb[0] + min(c, p.m_pixels - 1)),
                                    (double)p.mb[0], (double)p.mb[1]);
        sm.pos[0][lane] = pn;
        sm.pos[1][lane] = p.cpm_az[2] * pn;
        sm.pos[2][lane] = p.cpm_az[5] * pn * pn;
        sm.pos[3][lane] = p.cpm_rg[2] * pn;
        sm.pos[4][lane] = p.cpm_rg[5] * pn * pn;
    }

    // slave column of lane 0.  Output j (lane j) takes its range taps from
    // lanes ix_j - 5 - ucol0 .. +11, which must lie in 0 .. 63.  With
    // rel_j = ix_j - j over the strip within [lo, hi] (its corners: the
    // offset fields are smooth), ucol0 = lo - 5 serves every output when
    // hi - lo <= 1 (the slave column drifts by at most one column along the
    // strip's 52 outputs and rows); any other output takes the direct path.
    int ucol0;
    {
        const int cl = min(c0 + WK_OUT - 1, p.m_pixels - 1);
        const int cc = (lane & 2) ? cl : c0;
        int iyc, fyc, ixc, fxc;
        slave_pos(p, (lane & 1) ? r1 - 1 : r0, cc, iyc, fyc, ixc, fxc);
        const int rel = ixc - (cc - c0);
        int lo = __builtin_amdgcn_readlane(rel, 0);
        for (int k = 1; k < 4; k++) lo = min(lo, __builtin_amdgcn_readlane(rel, k));
        ucol0 = lo - kHalf;
    }
    ColumnWalker w;
    w.init(p, ucol0 + lane);
    {
        double a = 0.0, b = 0.0, cc = 0.0;
        if (w.in_box) phase_coeffs(p, w.xcol, a, b, cc);
        sm.abc[0][lane] = a;
        sm.abc[1][lane] = b;
        sm.abc[2][lane] = cc;
        phasor(2.0 * cc, w.qr, w.qi);
    }
    if (fit_phase(p, sm, ucol0))
        walk_rows<true, kEven>(p, c0, r0, r1, ucol0, w, sm);
    else
        walk_rows<false, kEven>(p, c0, r0, r1, ucol0, w, sm);
}

// The strip of workgroup b of n: the first n_tall strips, then the others, each
// dealt to the XCDs in contiguous ranges (strips whose slave columns overlap
// run on one XCD)
__device__ __forceinline__ int strip_remap(int b, int n_tall, int n)
{
    return b < n_tall ? xcd_remap(b, n_tall) : n_tall + xcd_remap(b - n_tall, n - n_tall);
}

// Batched form: one workgroup per entry of a strip table covering many
// bursts (work[i] = {burst, strip x, first row, rows}; the first n_tall entries
// are the tall strips).
template <bool kEven>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWalkWavesPerSimd)))
resample_batch_kernel(const ResampleParams* items, const int4* work, int n_tall)
{
    __shared__ WalkLds sm;
    // the table and the parameter blocks are read-only and read with
    // wave-uniform indices: through the constant address space they become
    // scalar loads, as the single-burst kernel's argument block is
    typedef __attribute__((address_space(4))) const int CInt;
    typedef __attribute__((address_space(4))) const ResampleParams CParams;
    const CInt* w = (const CInt*)work + 4 * strip_remap((int)blockIdx.x, n_tall, (int)gridDim.x);
    const int item = w[0], sx = w[1], r0 = w[2], rows = w[3];
    CParams* it = (CParams*)items + item;
    resample_strip<kEven>(*(const ResampleParams*)it, sx, r0, min(r0 + rows, it->m_lines), sm);
}

// Row ranges of up to kItems bursts in one launch, the parameter blocks in the
// kernel arguments: nothing is uploaded, so the launch can be captured.
// seg[i]: rows row0 .. row0+rows-1 of item `item` in strips of `height` rows,
// numbered from `first` on, row strips fastest, the first tall_strips of them
// tall.
template <int kItems>
struct ResampleSet {
    ResampleParams item[kItems];
    struct Seg { int item, row0, rows, height, first; } seg[4 * kItems];
    int n_seg, tall_strips;
};
static_assert(sizeof(ResampleSet<kResampleSetItems>) <= 4096, "kernel argument segment");

template <int kItems, bool kEven>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWalkWavesPerSimd)))
resample_fast_kernel(ResampleSet<kItems> set)
{
    __shared__ WalkLds sm;
    // the arguments read in place in the kernel-argument segment: their fields
    // become scalar loads where they are used, as in the batched kernel,
    // instead of SGPRs held for the whole kernel (which spill to VGPR lanes
    // inside the row loop)
    typedef __attribute__((address_space(4))) const ResampleSet<kItems> CSet;
    CSet* k = (CSet*)__builtin_amdgcn_kernarg_segment_ptr();
    (void)set;
    int t = strip_remap((int)blockIdx.x, k->tall_strips, (int)gridDim.x);
    int i = 0;
    while (i + 1 < k->n_seg && k->seg[i + 1].first <= t) i++;
    t -= k->seg[i].first;
    const int h = k->seg[i].height, rows = k->seg[i].rows, ny = (rows + h - 1) / h;
    const int sx = t / ny, sy = t - sx * ny;
    const int r0 = k->seg[i].row0 + sy * h;
    const int r1 = min(r0 + h, k->seg[i].row0 + rows);
    resample_strip<kEven>(*(const ResampleParams*)&k->item[k->seg[i].item], sx, r0, r1, sm);
}

int resample_strip_columns(int m_pixels) { return (m_pixels + WK_OUT - 1) / WK_OUT; }

// Walker waves the GPU holds at once: CUs x 4 SIMDs x the kernel's waves per
// SIMD (kWalkWavesPerSimd)
int resample_wave_slots() { return device_cus() * 4 * kWalkWavesPerSimd; }

// Strip height whose strips (each one wave) fill `rounds` rounds of the
// GPU's wave slots without a partial extra round: the smallest height with
// sum_i nx_i * ceil(lines_i / h) <= rounds * slots.
int resample_rows_for_rounds(const int* lines, const int* pixels, int n, int rounds)
{
    const long cap = (long)rounds * resample_wave_slots();
    int lo = 8, hi = 8;
    for (int i = 0; i < n; i++) hi = std::max(hi, lines[i]);
    auto strips = [&](int h) {
        long t = 0;
        for (int i = 0; i < n; i++)
            t += (long)((pixels[i] + WK_OUT - 1) / WK_OUT) * ((lines[i] + h - 1) / h);
        return t;
    };
    if (strips(hi) > cap) return hi;
    while (lo < hi) {
        int mid = (lo + hi) / 2;
        if (strips(mid) <= cap) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

static int whole_groups(int rows) { return (rows + WK_GROUP - 1) / WK_GROUP * WK_GROUP; }

// Tall strips of `tall` rows, and low ones for the last rows of every range:
// the GPU stays full until the last strips, which end within a low strip's
// time of each other.  The low ones cover 0.6 tall strips' time of every wave
// slot (0.4 to 0.9 measured the same within 2 %), none where that is under a
// twentieth of the launch.
StripHeights resample_heights_of(int tall, const int* lines, const int* pixels, int n)
{
    double rows = 0;
    for (int i = 0; i < n; i++) rows += (double)lines[i] * resample_strip_columns(pixels[i]);
    const double r = rows / resample_wave_slots();
    const int low = std::max(8, whole_groups(tall / 4));
    const int pct = (int)std::min(25.0, 60.0 * tall / std::max(r, 1.0));
    return {tall, low, low < tall && pct >= 5 ? pct : 0};
}

// Strip heights of a launch of n row ranges.  With R rows of strips per wave
// slot, strips of h rows that each cost about 8 rows more to start, and a last
// round that is half empty, the time goes as R (1 + 8 / h) + c h: least at a
// height proportional to sqrt(R), measured 56 to 64 rows at R = 200, 48 at
// 113, 32 at 39, 20 to 24 at 19; in launches of many rows 50 to 56 were best
// (9 bursts 1500 x 21000 in the subswath flow 3.62 ms, 3.68 at 64, 3.79 at 96).
// A launch whose tall strips spill a little into another round takes the next
// height that does not (700 x 9000: 69 us at 28, 60 at 32).  Few rows fill the
// slots once, in strips of 8 rows (512 x 2048: 24 us at 8, 26 at 12), or of 4,
// one group, where those all run at once: a wave is a chain of its groups (130 x
// 1000: 13.9 us, 21.0 at 8; 300 x 2000 17.8, 20.4).
// One height for 6 rounds against this: 1500 x 21000 250 us -> 234, 1487 x
// 24491 289 -> 267, 1200 x 15000 152 -> 145, 700 x 9000 75 -> 60, 300 x 20000
// 73 -> 62, 100 x 21000 32 -> 29.
static StripHeights resample_heights(const int* lines, const int* pixels, int n)
{
    const double slots = resample_wave_slots();
    double rows = 0;
    for (int i = 0; i < n; i++) rows += (double)lines[i] * resample_strip_columns(pixels[i]);
    const double r = rows / slots;
    if (r <= 4) return {4, 4, 0};
    if (r <= 8) return {8, 8, 0};
    int h = std::min(WK_GROUP * (int)std::lround(1.13 * std::sqrt(r)), 56);
    for (int k = 0; k < 3; k++, h += WK_GROUP) {
        const StripHeights sh = resample_heights_of(h, lines, pixels, n);
        double tall = 0, low = 0;
        for (int i = 0; i < n; i++) {
            const int nx = resample_strip_columns(pixels[i]), nl = sh.low_rows(lines[i]);
            tall += (double)nx * ((lines[i] - nl + h - 1) / h);
            low += (double)nx * (nl / sh.low);
        }
        // the tall strips' rounds against the average end of all strips
        constexpr double kStart = 8;
        const double all = (tall * (h + kStart) + low * (sh.low + kStart)) / slots;
        if (std::ceil(tall / slots) * (h + kStart) <= all + 0.5 * (sh.low + kStart)) return sh;
    }
    return resample_heights_of(h - 3 * WK_GROUP, lines, pixels, n);
}

// Whether the walker's form for even positions serves an item: over the whole
// box the slave line advances by 1 within 1/16 a row, so that the window starts
// anew at most every fourth group, and 4 rows of a strip spread over at most 4
// lines.  Both slopes are linear: their extremes are at the box's corners.  A
// false comparison, as of NaN, takes the other form, which serves everything.
// (1500 x 12000, this form against the other, us: 1 line a row 164 / 177, 0.95 164
// / 167, 1.05 150 / 155, 0.9 169 / 162, 0.8 183 / 157, 0.5 188 / 150, 2 2570 / 166;
// lines a column 0.018 2263 / 2526, 0.025 3211 / 2523.  The walker of one row at a
// time: 202 at 1, 168 at 0.5, 192 at 2, and 206 at 3 lines a row, where the other
// form takes two window positions a group, 245.)
bool resample_even(const ResampleParams& p)
{
    const double per_row = 4.0 / (p.mb[3] - p.mb[2]), per_col = 4.0 / (p.mb[1] - p.mb[0]);
    for (int k = 0; k < 4; k++) {
        const double ln = k & 1 ? 2.0 : -2.0, pn = k & 2 ? 2.0 : -2.0;
        const double* c = p.cpm_az;
        const double rate = (c[1] + 2.0 * c[3] * ln + c[4] * pn) * per_row;
        const double shear = (c[2] + c[4] * ln + 2.0 * c[5] * pn) * per_col;
        if (!(std::fabs(rate - 1.0) <= 1.0 / 16 &&
              (WK_GROUP - 1) * rate + WK_OUT * std::fabs(shear) <= kAzShifts - 1))
            return false;
    }
    return true;
}

static int check_slave_bytes(const ResampleParams& p)
{
    if ((long long)p.s_lines * p.s_pixels * 4 > kMaxSlaveBytes)
        return set_error(TOPS_ERR_ARG, "resample: slave box of %d x %d samples over 2^31 bytes",
                         p.s_lines, p.s_pixels);
    return TOPS_OK;
}

// Ranges i0 .. i1-1 of items[base ..] in one launch.
template <int kItems>
static int launch_set(const ResampleParams* items, int base, const int (*range)[3], int i0, int i1,
                      const StripHeights& sh, hipStream_t s)
{
    ResampleSet<kItems> set;
    set.n_seg = 0;
    int strips = 0;
    auto add = [&](int item, int row0, int rows, int h) {
        if (rows <= 0) return;
        // (no runt: the strips of a range are of one height)
        h = whole_groups((rows + (rows + h - 1) / h - 1) / ((rows + h - 1) / h));
        set.seg[set.n_seg++] = {item, row0, rows, h, strips};
        strips += resample_strip_columns(set.item[item].m_pixels) * ((rows + h - 1) / h);
    };
    for (int i = i0; i < i1; i++) {
        const int k = range[i][0] - base;
        set.item[k] = items[range[i][0]];
        add(k, range[i][1], range[i][2] - sh.low_rows(range[i][2]), sh.tall);
    }
    set.tall_strips = strips;
    for (int i = i0; i < i1; i++) {
        const int n = sh.low_rows(range[i][2]);
        add(range[i][0] - base, range[i][1] + range[i][2] - n, n, sh.low);
    }
    if (strips == 0) return TOPS_OK;
    bool even = true;
    for (int i = i0; i < i1; i++) even = even && resample_even(items[range[i][0]]);
    if (even)
        hipLaunchKernelGGL((resample_fast_kernel<kItems, true>), dim3(strips), dim3(64), 0, s, set);
    else
        hipLaunchKernelGGL((resample_fast_kernel<kItems, false>), dim3(strips), dim3(64), 0, s, set);
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

int launch_resample_fast(const ResampleParams& p, hipStream_t s, int strip_rows)
{
    if (int rc = check_slave_bytes(p)) return rc;
    StripHeights sh = {strip_rows, strip_rows, 0};
    if (strip_rows <= 0) sh = resample_heights(&p.m_lines, &p.m_pixels, 1);
    const int range[1][3] = {{0, 0, p.m_lines}};
    return launch_set<1>(&p, 0, range, 0, 1, sh, s);
}

// Row ranges range[i] = {item, first row, rows} (in item order, at most two an
// item) of n_items bursts.
int launch_resample_set(const ResampleParams* items, int n_items, const int (*range)[3],
                        int n_range, hipStream_t s)
{
    std::vector<int> lines(n_range), pixels(n_range);
    for (int i = 0; i < n_range; i++) {
        const int it = range[i][0];
        if (it < 0 || it >= n_items || (i > 1 && range[i - 2][0] >= it) ||
            (i > 0 && range[i - 1][0] > it))
            return set_error(TOPS_ERR_ARG, "resample: row ranges out of order");
        const ResampleParams& p = items[it];
        if (range[i][1] < 0 || range[i][2] < 0 || range[i][1] + range[i][2] > p.m_lines)
            return set_error(TOPS_ERR_ARG, "resample: rows %d .. %d outside the box's %d lines",
                             range[i][1], range[i][1] + range[i][2] - 1, p.m_lines);
        if (int rc = check_slave_bytes(p)) return rc;
        lines[i] = range[i][2];
        pixels[i] = p.m_pixels;
    }
    if (n_range == 0) return TOPS_OK;
    const StripHeights sh = resample_heights(lines.data(), pixels.data(), n_range);
    for (int i = 0; i < n_range;) {
        // as many items as the arguments hold
        const int i0 = i, base = range[i][0];
        while (i < n_range && range[i][0] < base + kResampleSetItems) i++;
        if (int rc = launch_set<kResampleSetItems>(items, base, range, i0, i, sh, s)) return rc;
    }
    return TOPS_OK;
}

int launch_resample_batch(const ResampleParams* d_items, const int4* d_work, int n_work,
                          int n_tall, bool even, hipStream_t s)
{
    if (n_work <= 0) return TOPS_OK;
    if (even)
        hipLaunchKernelGGL(resample_batch_kernel<true>, dim3(n_work), dim3(64), 0, s, d_items,
                           d_work, n_tall);
    else
        hipLaunchKernelGGL(resample_batch_kernel<false>, dim3(n_work), dim3(64), 0, s, d_items,
                           d_work, n_tall);
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

}  // namespace tops
