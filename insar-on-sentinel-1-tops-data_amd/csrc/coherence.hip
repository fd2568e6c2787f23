// coherence.hip -- boxcar interferometric coherence (gfx950).
//
// Semantics of EstCoh.cu:101-139 (CohMatSet, short2 master) and 413-456
// (Cohbasic): per output (r, c) the window covers rows r-dy .. r-dy+winAz-1
// and columns c-dx .. c-dx+winRg-1 of the burst, zero outside it (the
// reference leaves that padding uninitialised, EstCoh.cu:581-583);
//   coh = |sum M conj(S)| / sqrt(sum|S|^2 * sum|M|^2)  (0 when the product
//   is not positive), and coh = 0 where |S(r, c)| < 0.001.
//
// Fast forms: windows of 2 to 8 lines and 4 to 64 samples walk down bands of
// columns (coherence_band.hpp); other windows, and rasters too small to fill
// the GPU with bands, stage the products (M conj S, |S|^2, |M|^2) of a 16x64
// output tile's (16+winAz-1) x (64+winRg-1) window in LDS and form plain FP32
// range sums, then short azimuth sums.  Each window sum is a direct sum of its
// own terms in both (tile_window.hpp).
// FP64 form: one thread per output, direct FP64 window sums from HBM.
#include "tops_internal.hpp"
#include "tile_window.hpp"
#include "coherence_band.hpp"

#include <algorithm>
#include <type_traits>

namespace tops {

__global__ void __launch_bounds__(256) coherence_fp64_kernel(const tops_ci16* M, const tops_cf32* S, int w,
                                      int h, int dx, int dy, int win_rg, int win_az,
                                      float* coh)
{
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    int r = blockIdx.y;
    if (c >= w) return;
    size_t q0 = (size_t)r * w + c;
    tops_cf32 sc = S[q0];
    double mag = sqrt((double)sc.x * sc.x + (double)sc.y * sc.y);
    if (mag < 0.001) { coh[q0] = 0.0f; return; }
    double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
    for (int j = 0; j < win_az; j++) {
        int rr = r - dy + j;
        if (rr < 0 || rr >= h) continue;
        for (int k = 0; k < win_rg; k++) {
            int cc = c - dx + k;
            if (cc < 0 || cc >= w) continue;
            size_t q = (size_t)rr * w + cc;
            tops_ci16 m = M[q];
            tops_cf32 s = S[q];
            double mr = m.re, mi = m.im, sr = s.x, si = s.y;
            a0 += mr * sr + mi * si;
            a1 += mi * sr - mr * si;
            a2 += sr * sr + si * si;
            a3 += mr * mr + mi * mi;
        }
    }
    double pp = a2 * a3;
    coh[q0] = pp > 0.0 ? (float)(sqrt(a0 * a0 + a1 * a1) / sqrt(pp)) : 0.0f;
}

// CWR x CWA: a window fixed at compile time (0 x 0: win_rg x win_az)
template <int CWR = 0, int CWA = 0>
__device__ __forceinline__ void coherence_tile(const tops_ci16* M, const tops_cf32* S, int w,
                                               int h, int dx, int dy, int win_rg, int win_az,
                                               float* coh, int tx, int ty, float4* smem)
{
    const int r0 = ty * TW_ROWS, c0 = tx * TW_COLS;
    WindowSums ws[4];
    // (uniform branch; the launch's LDS is tile_window_launch_lds for it)
    if (CWR ? true : tile_window_shared_ok(win_rg, win_az))
        tile_window_sums_shared<CWR, CWA>(M, S, w, h, r0, c0, dx, dy, win_rg, win_az, smem, ws,
                                          nullptr);
    else
        tile_window_sums(M, S, w, h, r0, c0, dx, dy, win_rg, win_az, smem, ws, nullptr);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int c = c0 + lane;
    if (c >= w) return;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int r = r0 + wv * 4 + k;
        if (r >= h) break;
        size_t q = (size_t)r * w + c;
        tops_cf32 s = S[q];
        float out = 0.0f;
        if (amplitude_ok(s.x * s.x + s.y * s.y)) out = ws[k].coherence();
        coh[q] = out;
    }
}

template <int CWR = 0, int CWA = 0>
__global__ void __launch_bounds__(256) coherence_fast_kernel(const tops_ci16* M, const tops_cf32* S, int w,
                                      int h, int dx, int dy, int win_rg, int win_az,
                                      float* coh)
{
    extern __shared__ float4 smem[];
    coherence_tile<CWR, CWA>(M, S, w, h, dx, dy, win_rg, win_az, coh, blockIdx.x, blockIdx.y,
                             smem);
}

// Batched form: work[i] = {item, tile x, tile y, 0}.
template <int CWR = 0, int CWA = 0>
__global__ void __launch_bounds__(256) coherence_batch_kernel(const CohItem* items, const int4* work,
                                                              int dx, int dy, int win_rg, int win_az)
{
    extern __shared__ float4 smem[];
    const int4 wk = work[blockIdx.x];
    const CohItem& it = items[wk.x];
    coherence_tile<CWR, CWA>(it.m, it.s, it.w, it.h, dx, dy, win_rg, win_az, it.coh, wk.y, wk.z,
                             smem);
}

// ---- band form (coherence_band.hpp) --------------------------------------
// Workgroups of 256 threads, as many per CU as the registers allow (waves per
// SIMD): 4 for 2 and 3 lines (82 and 97 VGPRs), 3 for 4 to 7 (113 to 161; 4
// lines at 4 waves 123 us against 114 on 1487 x 24491, 7 x 20 at 2 waves 125 us
// against 110 on 1500 x 21000), 2 above (205).
__host__ __device__ constexpr int band_waves(int win_az)
{
    return win_az <= 3 ? 4 : win_az <= 7 ? 3 : 2;
}
constexpr int CB_THREADS = 256;

template <int WA>
__global__ void __launch_bounds__(CB_THREADS)
__attribute__((amdgpu_waves_per_eu(band_waves(WA))))
coherence_band_kernel(const tops_ci16* M, const tops_cf32* S, int w, int h, int dx, int dy,
                      int win_rg, float* coh, int rows, size_t stride)
{
    extern __shared__ float4 smem[];
    // blocks numbered bands fastest and dealt to the XCDs in contiguous
    // ranges; raster blockIdx.z
    const int t = xcd_remap((int)(blockIdx.x + blockIdx.y * gridDim.x),
                            (int)(gridDim.x * gridDim.y));
    const int by = t / (int)gridDim.x, bx = t - by * (int)gridDim.x;
    const int r0 = by * rows;
    M += blockIdx.z * stride;
    S += blockIdx.z * stride;
    coh += blockIdx.z * stride;
    coherence_band<WA, CB_THREADS>(M, S, w, h, coh, dx, dy, win_rg,
                       bx * coherence_band_cols(CB_THREADS, win_rg), r0, min(r0 + rows, h),
                       by & 1, smem);
}

// Batched form: work[i] = {item, band, row block, 0}, `rows` rows per block;
// table and items through the constant address space (scalar loads).
template <int WA>
__global__ void __launch_bounds__(CB_THREADS)
__attribute__((amdgpu_waves_per_eu(band_waves(WA))))
coherence_band_batch_kernel(const CohItem* items, const int4* work, int dx, int dy, int win_rg,
                            int rows)
{
    extern __shared__ float4 smem[];
    typedef __attribute__((address_space(4))) const int CInt;
    typedef __attribute__((address_space(4))) const CohItem CCohItem;
    const CInt* wk = (const CInt*)work + 4 * xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int item = wk[0], bx = wk[1], by = wk[2];
    CCohItem* it = (CCohItem*)items + item;
    const int h = it->h, r0 = by * rows;
    coherence_band<WA, CB_THREADS>(it->m, it->s, it->w, h, it->coh, dx, dy, win_rg,
                       bx * coherence_band_cols(CB_THREADS, win_rg), r0, min(r0 + rows, h),
                       by & 1, smem);
}

// The form of a launch over n rasters of one window (sizes w[i * step], h[i *
// step]; step 0: all of one size).  A band's workgroup is a
// chain of its rows and the window's, so rasters whose tiles all run at once
// stay with them: up to 4 tiles per CU for windows of up to 5 lines, 8 above
// (us, tiles against bands, 256 CUs: 3 x 10 window 6.6 / 7.3 on 512 x 2048,
// 8.2 / 7.7 on 600 x 2000, 13.5 / 9.1 on 700 x 3000; 6 x 24 window 11.9 / 14.5
// on 1500 x 1100, 14.6 / 13.5 on 700 x 3000, 153 / 102 on 1500 x 21000).
CohForm coherence_form(const int* w, const int* h, int n, int step, int dx, int dy, int win_rg,
                       int win_az)
{
    const bool tile_ok = tile_window_launch_lds(win_rg, win_az) != 0;
    bool band_ok = win_az >= 2 && win_az <= CB_MAX_AZ && win_rg >= CB_PER_THREAD &&
                   win_rg <= CB_MAX_RG && dx >= 0 && dx < win_rg && dy >= 0 && dy < win_az;
    long tiles = 0;
    for (int i = 0; i < n; i++) {
        int nx, ny;
        tiles += coherence_tile_count(w[i * step], h[i * step], &nx, &ny);
        band_ok = band_ok && w[i * step] <= CB_MAX_WIDTH;
    }
    if (band_ok && (!tile_ok || tiles > (long)device_cus() * (win_az <= 5 ? 4 : 8)))
        return CohForm::kBand;
    return tile_ok ? CohForm::kTile : CohForm::kDirect;
}

int coherence_band_count(int w, int h, int win_rg, int rows, int* nx, int* ny)
{
    const int cols = coherence_band_cols(CB_THREADS, win_rg);
    *nx = (w + cols - 1) / cols;
    *ny = (h + rows - 1) / rows;
    return *nx * *ny;
}

// Rows per workgroup: the fewest with which all workgroups run at once, 3 per
// CU for 3 to 7 lines (a fourth fits beside 3 lines but reads more halo rows:
// 101 us instead of 99 on 1500 x 21000), else as many as fit (2 lines: 103 us
// with 4, 114 with 3).  Launches of many rasters take further rounds rather
// than more than 96 rows, up to the 65535 row blocks a grid has.
static int coherence_band_rows(int w, int h, int n, int win_rg, int win_az)
{
    const long slots = (long)device_cus() * (win_az == 3 ? 3 : band_waves(win_az));
    const int least = (int)((h + 65534l) / 65535);
    for (long round = 1;; round++) {
        int lo = 1, hi = h;   // the smallest height within `round` rounds
        auto blocks = [&](int rows) {
            int nx, ny;
            return (long)n * coherence_band_count(w, h, win_rg, rows, &nx, &ny);
        };
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (blocks(mid) <= round * slots) hi = mid;
            else lo = mid + 1;
        }
        if (lo <= 96 && blocks(lo) <= round * slots) return std::max(lo, least);
    }
}

int coherence_tile_count(int w, int h, int* nx, int* ny)
{
    *nx = (w + TW_COLS - 1) / TW_COLS;
    *ny = (h + TW_ROWS - 1) / TW_ROWS;
    return *nx * *ny;
}

int launch_coherence_batch(const CohItem* d_items, const int4* d_work, int n_work, CohForm form,
                           int dx, int dy, int win_rg, int win_az, int band_rows, hipStream_t st)
{
    if (n_work <= 0) return TOPS_OK;
    if (form == CohForm::kBand) {
        if (band_rows <= 0)
            return set_error(TOPS_ERR_ARG, "batched coherence: %d rows per block", band_rows);
        band_dispatch(win_az, [&](auto wa) {
            hipLaunchKernelGGL(coherence_band_batch_kernel<decltype(wa)::value>, dim3(n_work),
                               dim3(CB_THREADS), coherence_band_lds(CB_THREADS), st, d_items,
                               d_work, dx, dy, win_rg, band_rows);
        });
        TOPS_HIP(hipGetLastError());
        return TOPS_OK;
    }
    const size_t lds = tile_window_launch_lds(win_rg, win_az);
    if (lds == 0 || form != CohForm::kTile)
        return set_error(TOPS_ERR_ARG, "batched coherence: window %dx%d exceeds the LDS tile",
                         win_az, win_rg);
    if (reference_window(win_rg, win_az))
        hipLaunchKernelGGL((coherence_batch_kernel<24, 6>), dim3(n_work), dim3(256), lds, st,
                           d_items, d_work, dx, dy, win_rg, win_az);
    else
        hipLaunchKernelGGL(coherence_batch_kernel, dim3(n_work), dim3(256), lds, st, d_items,
                           d_work, dx, dy, win_rg, win_az);
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

static int launch_band(const tops_ci16* m, const tops_cf32* s, int w, int h, int n, size_t stride,
                       int dx, int dy, int win_rg, int win_az, float* coh, hipStream_t st)
{
    const int rows = coherence_band_rows(w, h, n, win_rg, win_az);
    int nx, ny;
    coherence_band_count(w, h, win_rg, rows, &nx, &ny);
    band_dispatch(win_az, [&](auto wa) {
        hipLaunchKernelGGL(coherence_band_kernel<decltype(wa)::value>, dim3(nx, ny, n),
                           dim3(CB_THREADS), coherence_band_lds(CB_THREADS), st, m, s, w, h, dx,
                           dy, win_rg, coh, rows, stride);
    });
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

int launch_coherence_stack(const tops_ci16* m, const tops_cf32* s, int w, int h, int n,
                           size_t stride, int dx, int dy, int win_rg, int win_az, float* coh,
                           hipStream_t st)
{
    // bands of all rasters in one launch (9 of 1500 x 23500, 6 x 24: 1.01 ms
    // against 1.08 one by one)
    if (coherence_form(&w, &h, n, 0, dx, dy, win_rg, win_az) == CohForm::kBand && n <= 65535)
        return launch_band(m, s, w, h, n, stride, dx, dy, win_rg, win_az, coh, st);
    int rc = TOPS_OK;
    for (int i = 0; i < n && !rc; i++)
        rc = launch_coherence(m + i * stride, s + i * stride, w, h, dx, dy, win_rg, win_az,
                              coh + i * stride, TOPS_MODE_FAST, st);
    return rc;
}

int launch_coherence(const tops_ci16* m, const tops_cf32* s, int w, int h, int dx,
                     int dy, int win_rg, int win_az, float* coh, int mode, hipStream_t st)
{
    const CohForm form = mode == TOPS_MODE_FP64
                             ? CohForm::kDirect
                             : coherence_form(&w, &h, 1, 0, dx, dy, win_rg, win_az);
    if (form == CohForm::kBand)
        return launch_band(m, s, w, h, 1, 0, dx, dy, win_rg, win_az, coh, st);
    if (form == CohForm::kDirect) {
        dim3 g((w + 255) / 256, h);
        hipLaunchKernelGGL(coherence_fp64_kernel, g, dim3(256), 0, st, m, s, w, h, dx, dy,
                           win_rg, win_az, coh);
    } else {
        dim3 g((w + TW_COLS - 1) / TW_COLS, (h + TW_ROWS - 1) / TW_ROWS);
        if (reference_window(win_rg, win_az))
            hipLaunchKernelGGL((coherence_fast_kernel<24, 6>), g, dim3(256),
                               tile_window_launch_lds(win_rg, win_az), st, m, s, w, h, dx, dy,
                               win_rg, win_az, coh);
        else
            hipLaunchKernelGGL(coherence_fast_kernel, g, dim3(256),
                               tile_window_launch_lds(win_rg, win_az), st, m, s, w, h, dx, dy,
                               win_rg, win_az, coh);
    }
    TOPS_HIP(hipGetLastError());
    return TOPS_OK;
}

}  // namespace tops
