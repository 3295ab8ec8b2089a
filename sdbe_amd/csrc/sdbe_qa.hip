// FX cross-correlation checker behind include/sdbe_qa.h: the GPU form of
// corr_Xt_search / corr_Xt (software/verification/cross_corr.py:23-116).
//
// Kernels (32768-sample windows, 16384-point complex FFTs in LDS):
//   k_xc_r2c    one workgroup per window of either series: packed R2C, bins
//               0..16383 (numpy fft scale), and the window's auto-power,
//               weighted for its lag-0 value
//   k_xc_cross  per (bin block, tile of offsets): mean cross-power S_0x1
//   k_xc_c2r    one workgroup per offset: packed C2R of S_0x1 (numpy irfft
//               scale, bin 16384 zero) divided by sqrt(s_0x0[0] s_1x1[0]),
//               with the peak |s| and the standard deviation of s
// The maximum of an autocorrelation (the inverse real DFT of a non-negative
// power spectrum) is its lag-0 value, (P[0] + 2 sum_{k>0} P[k]) / 32768.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <new>
#include <vector>

#include "sdbe_device.hpp"
#include "../../include/sdbe_qa.h"

using namespace sdbe;

namespace {

constexpr int LW = SDBE_XCORR_WINDOW;     // 32768
constexpr int NHW = LW / 2;               // 16384
constexpr int KB = NHW / 256;             // bin blocks of k_xc_cross
// Offsets per wide k_xc_cross tile; what is left over goes to 4-wide tiles, and
// below XC_TILE_MIN offsets all tiles are 4 wide.  12 is what three waves per SIMD
// hold (168 registers; 16 takes 256).  257 offsets of 256 windows, a whole call: 283
// us with 8, 254 with 12, 274 with 16; 201 of 100: 115, 108, 122.  Three wide tiles
// are 768 waves for 1024 SIMDs and win already: 37 of 256 104 us, all 4 wide 114;
// 49 of 256 116 and 145; 63 of 128 81 and 92.  Two do not: 25 of 256 104 and 104.
constexpr int XC_OT = 12, XC_TILE_MIN = 3 * XC_OT;
static_assert(NHW == NCH, "the correlator reuses the 16384-point FFT");

// Sum over the 1024 threads of a workgroup, in every thread (red: 16 doubles).
__device__ __forceinline__ double block_sum_1024(double a, double *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += red[i];
    return s;
}

// Workgroups 0 .. avg - 1 take the x0 windows, the others the x1 windows, so one
// launch spreads both over the CUs.  pw[w] = sum over bins of (k ? 2 : 1) |X[w][k]|^2,
// the window's share of the lag-0 autocorrelation: a mean over any windows is a
// mean of these, so no later pass reads the spectra for it.
__global__ void __launch_bounds__(1024)
k_xc_r2c(const float *__restrict__ x0, int first0, const float *__restrict__ x1, int first1, int avg,
         float2 *__restrict__ X0, float2 *__restrict__ X1, double *__restrict__ pw0, double *__restrict__ pw1,
         const float2 *__restrict__ fft_img, const float2 *__restrict__ tw32k) {
    __shared__ float lds[LDS_FFT_N];
    __shared__ FftTw ftw;
    __shared__ double red[16];
    fft_tw_load(&ftw, fft_img);
    const int t = threadIdx.x;
    const bool second = (int)blockIdx.x >= avg;
    const int w = second ? (int)blockIdx.x - avg : (int)blockIdx.x;
    const float2 *xb = reinterpret_cast<const float2 *>(second ? x1 + (size_t)(first1 + w) * LW
                                                               : x0 + (size_t)(first0 + w) * LW);
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = xb[t + 1024 * q];
    fft16k<-1>(v, lds, &ftw);
    __syncthreads();    // the FFT's last LDS reads are done
#pragma unroll
    for (int q = 0; q < 16; ++q) lds_put(lds, lds_re(t + 1024 * q), v[q]);
    __syncthreads();
    float2 *out = (second ? X1 : X0) + (size_t)w * NHW;
    double p = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int k = t + 1024 * q;
        const int km = (NHW - k) & (NHW - 1);
        const float2 zm = cconj(lds_get(lds, lds_re(km)));   // conj Z[N - k]
        const float2 E = cscale(cadd(v[q], zm), 0.5f);
        const float2 D = cscale(csub(v[q], zm), 0.5f);
        const float2 X = cadd(E, mul_si<-1>(cmul(cconj(tw32k[k]), D)));
        out[k] = X;
        p += (k == 0 ? 1.0 : 2.0) * ((double)X.x * X.x + (double)X.y * X.y);
    }
    const double s = block_sum_1024(p, red);
    if (t == 0) (second ? pw1 : pw0)[w] = s;
}

// Offsets o0 .. o0 + OT - 1 of bin k: S[o][k] = mean_w X0[w][k] conj(X1[o + w][k]),
// FP64 sums.  One thread keeps OT sums and the OT windows of x1 that the current
// w meets, in a ring that takes one new window per step (unrolled, so its
// indices are constants): one load of each series and two conversions per OT
// offsets, where a thread per (bin, offset) loaded and converted both for every
// offset.  The FP64 FMAs bound it, so a complex product is three of them and not
// four (ax bx, ay by, (ax + ay)(bx - by); the second factor comes once per window):
// the factors are FP32 values and their sums, which FP64 holds with room to spare, and
// the rounding of the three sums is 1e-16 of the powers.  82 us for 257 offsets of 256
// windows at one wave instruction per CU and cycle; a whole call 254 us, with four
// products and 16 offsets a thread 290, with a thread per (bin, offset) 1165.
// Bin blocks are the fastest grid dimension, 64 of them, so the tiles of a bin
// block run on one XCD and read the same windows through its L2 at about the
// same time.
template <int OT>
__device__ __forceinline__ void cross_tile(const float2 *__restrict__ X0, const float2 *__restrict__ X1, int avg,
                                           int n_off, int o0, int k, float2 *__restrict__ S) {
    const int last = n_off + avg - 2;          // last x1 window; a tile past n_off loads it again
    // sums of ax bx, ay by and (ax + ay)(bx - by); a conj(b) = pr + pi + i (pd - pr + pi)
    double pr[OT], pi[OT], pd[OT], bx[OT], by[OT], bd[OT];
#pragma unroll
    for (int j = 0; j < OT; ++j) {
        const float2 b = X1[(size_t)min(o0 + j, last) * NHW + k];
        pr[j] = pi[j] = pd[j] = 0.0;
        bx[j] = b.x;       // slot OT - 1 is replaced by the first step
        by[j] = b.y;
        bd[j] = bx[j] - by[j];
    }
    // step i of a block of OT: window o0 + w + j of x1 is in slot (i + j) % OT
    auto step = [&](int i, float2 a, float2 b) {
        const double ax = a.x, ay = a.y, as = ax + ay;
        constexpr int N1 = OT - 1;
        bx[(i + N1) % OT] = b.x;
        by[(i + N1) % OT] = b.y;
        bd[(i + N1) % OT] = bx[(i + N1) % OT] - by[(i + N1) % OT];
#pragma unroll
        for (int j = 0; j < OT; ++j) {
            pr[j] = fma(ax, bx[(i + j) % OT], pr[j]);
            pi[j] = fma(ay, by[(i + j) % OT], pi[j]);
            pd[j] = fma(as, bd[(i + j) % OT], pd[j]);
        }
    };
    int w = 0;
    for (; w + OT <= avg; w += OT) {
        float2 a[OT], b[OT];
#pragma unroll
        for (int i = 0; i < OT; ++i) {
            a[i] = X0[(size_t)(w + i) * NHW + k];
            b[i] = X1[(size_t)min(o0 + w + i + OT - 1, last) * NHW + k];
        }
#pragma unroll
        for (int i = 0; i < OT; ++i) step(i, a[i], b[i]);
    }
#pragma unroll
    for (int i = 0; i < OT; ++i)
        if (w + i < avg)
            step(i, X0[(size_t)(w + i) * NHW + k], X1[(size_t)min(o0 + w + i + OT - 1, last) * NHW + k]);
#pragma unroll
    for (int j = 0; j < OT; ++j)
        if (o0 + j < n_off)
            S[(size_t)(o0 + j) * NHW + k] =
                make_float2((float)((pr[j] + pi[j]) / avg), (float)((pd[j] - pr[j] + pi[j]) / avg));
}

// n_wide tiles of OT offsets, then tiles of 4 for the rest
template <int OT>
__global__ void __launch_bounds__(256)
k_xc_cross(const float2 *__restrict__ X0, const float2 *__restrict__ X1, int avg, int n_off, int n_wide,
           float2 *__restrict__ S) {
    const int k = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
    if (y < n_wide)
        cross_tile<OT>(X0, X1, avg, n_off, y * OT, k, S);
    else
        cross_tile<4>(X0, X1, avg, n_off, n_wide * OT + 4 * (y - n_wide), k, S);
}

__global__ void __launch_bounds__(1024)
k_xc_c2r(const float2 *__restrict__ S, const double *__restrict__ pw0, const double *__restrict__ pw1, int avg,
         float *__restrict__ s_out, float *__restrict__ peak, float *__restrict__ sdev,
         const float2 *__restrict__ fft_img, const float2 *__restrict__ tw32k) {
    __shared__ float lds[LDS_FFT_N];
    __shared__ FftTw ftw;
    __shared__ double red[3][16];
    fft_tw_load(&ftw, fft_img);
    const int o = blockIdx.x, t = threadIdx.x;
    // mean lag-0 powers of the offset's windows
    double n0 = 0.0, n1 = 0.0;
    for (int i = t; i < avg; i += 1024) {
        n0 += pw0[i];
        n1 += pw1[o + i];
    }
    n0 = block_sum_1024(n0, red[0]) / avg;
    n1 = block_sum_1024(n1, red[1]) / avg;
    __syncthreads();    // red is used again below
    // irfft scale 1 / 32768 and the normalisation by the lag-0 autocorrelations
    const float sc = (float)(1.0 / ((double)LW * sqrt((n0 / LW) * (n1 / LW))));
    const float2 *Xo = S + (size_t)o * NHW;
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int k = t + 1024 * q;
        float2 a = Xo[k];
        float2 b = k == 0 ? make_float2(0.f, 0.f) : Xo[NHW - k];    // bin 16384 is zero
        if (k == 0) a.y = 0.f;                                      // bin 0: real part only
        const float2 sum = cadd(a, cconj(b)), dif = csub(a, cconj(b));
        v[q] = cadd(sum, mul_si<+1>(cmul(tw32k[k], dif)));
    }
    fft16k<+1>(v, lds, &ftw);
    float2 *dst = reinterpret_cast<float2 *>(s_out + (size_t)o * LW);
    double s1 = 0.0, s2 = 0.0;
    float mx = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const float2 y = cscale(v[q], sc);
        dst[t + 1024 * q] = y;
        s1 += (double)y.x + (double)y.y;
        s2 += (double)y.x * y.x + (double)y.y * y.y;
        mx = fmaxf(mx, fmaxf(fabsf(y.x), fabsf(y.y)));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
        mx = fmaxf(mx, __shfl_xor(mx, off));
    }
    if ((t & 63) == 0) {
        red[0][t >> 6] = s1;
        red[1][t >> 6] = s2;
        red[2][t >> 6] = (double)mx;
    }
    __syncthreads();
    if (t == 0) {
        double a = 0.0, b = 0.0, m = 0.0;
        for (int i = 0; i < 16; ++i) {
            a += red[0][i];
            b += red[1][i];
            m = fmax(m, red[2][i]);
        }
        const double mean = a / LW;
        double var = b / LW - mean * mean;
        if (var < 0.0) var = 0.0;
        peak[o] = (float)m;
        sdev[o] = (float)sqrt(var);
    }
}

}  // namespace

struct sdbe_xcorr {
    int device = 0;
    int max_win = 0, max_off = 0;
    int last_hip_err = 0;
    float2 *fft_img = nullptr;
    float2 *tw32k = nullptr;      // e^{2 pi i k / 32768}, k < 16384
    float2 *X0 = nullptr;         // [max_win][16384]
    float2 *X1 = nullptr;         // [max_win][16384]
    float2 *S = nullptr;          // [max_off][16384]
    double *pw0 = nullptr;        // [max_win] lag-0 power of each window
    double *pw1 = nullptr;        // [max_win]
};

namespace {
int xc_fail(sdbe_xcorr_t *x, hipError_t e) {
    if (x) x->last_hip_err = (int)e;
    return SDBE_ERR_HIP;
}
#define XC_TRY(x, expr)                               \
    do {                                              \
        hipError_t _e = (expr);                       \
        if (_e != hipSuccess) return xc_fail((x), _e); \
    } while (0)
}  // namespace

extern "C" {

void sdbe_xcorr_destroy(sdbe_xcorr_t *x) {
    if (!x) return;
    (void)hipSetDevice(x->device);
    (void)hipDeviceSynchronize();
    (void)hipFree(x->fft_img);
    (void)hipFree(x->tw32k);
    (void)hipFree(x->X0);
    (void)hipFree(x->X1);
    (void)hipFree(x->S);
    (void)hipFree(x->pw0);
    (void)hipFree(x->pw1);
    delete x;
}

int sdbe_xcorr_last_hip_error(const sdbe_xcorr_t *x) { return x ? x->last_hip_err : 0; }

int sdbe_xcorr_create(int device, int32_t max_windows, int32_t max_offsets, sdbe_xcorr_t **out) {
    if (!out) return SDBE_ERR_ARG;
    *out = nullptr;
    if (max_windows < 1 || max_windows > 65536 || max_offsets < 1 || max_offsets > 65535) return SDBE_ERR_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return SDBE_ERR_NODEV;
    if (hipSetDevice(device) != hipSuccess) return SDBE_ERR_NODEV;
    sdbe_xcorr_t *x = new (std::nothrow) sdbe_xcorr();
    if (!x) return SDBE_ERR_NOMEM;
    x->device = device;
    x->max_win = max_windows;
    x->max_off = max_offsets;
    int rc = SDBE_OK;
    std::vector<float2> img(FFT_TW_N), tw(NHW);
    const double two_pi = 6.283185307179586476925286766559;
    fft_tw_fill(img.data());
    for (int k = 0; k < NHW; ++k) {
        const double ang = two_pi * (double)k / (double)LW;
        tw[k] = make_float2((float)cos(ang), (float)sin(ang));
    }
#define XALLOC(ptr, bytes)                                              \
    do {                                                                \
        if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess) {        \
            rc = SDBE_ERR_NOMEM;                                        \
            goto fail;                                                  \
        }                                                               \
    } while (0)
    XALLOC(x->fft_img, FFT_TW_N * sizeof(float2));
    XALLOC(x->tw32k, NHW * sizeof(float2));
    XALLOC(x->X0, (size_t)max_windows * NHW * sizeof(float2));
    XALLOC(x->X1, (size_t)max_windows * NHW * sizeof(float2));
    XALLOC(x->S, (size_t)max_offsets * NHW * sizeof(float2));
    XALLOC(x->pw0, (size_t)max_windows * sizeof(double));
    XALLOC(x->pw1, (size_t)max_windows * sizeof(double));
#undef XALLOC
    if (hipMemcpy(x->fft_img, img.data(), FFT_TW_N * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(x->tw32k, tw.data(), NHW * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    *out = x;
    return SDBE_OK;
fail:
    sdbe_xcorr_destroy(x);
    return rc;
}

int sdbe_xcorr_search(sdbe_xcorr_t *x, const float *d_x0, int32_t n0_windows, const float *d_x1,
                      int32_t n1_windows, int32_t first_offset, int32_t n_offsets, int32_t avg, float *d_s,
                      float *d_peak, float *d_std, void *stream) {
    if (!x || !d_x0 || !d_x1 || !d_s || !d_peak || !d_std) return SDBE_ERR_ARG;
    if (avg < 1 || n_offsets < 1 || n0_windows < 1 || n1_windows < 1) return SDBE_ERR_ARG;
    const int64_t c = n0_windows / 2 - avg / 2;                 // cross_corr.py:97
    const int64_t lo = c + first_offset, hi = c + first_offset + (int64_t)n_offsets - 1 + avg;
    if (c < 0 || c + avg > n0_windows || lo < 0 || hi > n1_windows) return SDBE_ERR_ARG;
    if (n_offsets > x->max_off || avg > x->max_win || (int64_t)n_offsets + avg - 1 > x->max_win)
        return SDBE_ERR_CAPACITY;
    XC_TRY(x, hipSetDevice(x->device));
    hipStream_t s = (hipStream_t)stream;
    // spectra of the windows the search uses: x0[c, c + avg), x1[lo, lo + n_offsets + avg - 1)
    hipLaunchKernelGGL(k_xc_r2c, dim3(avg + n_offsets + avg - 1), dim3(1024), 0, s, d_x0, (int)c, d_x1, (int)lo,
                       (int)avg, x->X0, x->X1, x->pw0, x->pw1, (const float2 *)x->fft_img, (const float2 *)x->tw32k);
    const int n_wide = n_offsets >= XC_TILE_MIN ? n_offsets / XC_OT : 0;
    const int n_tiles = n_wide + (n_offsets - n_wide * XC_OT + 3) / 4;
    hipLaunchKernelGGL(k_xc_cross<XC_OT>, dim3(KB, n_tiles), dim3(256), 0, s, (const float2 *)x->X0,
                       (const float2 *)x->X1, (int)avg, (int)n_offsets, n_wide, x->S);
    hipLaunchKernelGGL(k_xc_c2r, dim3(n_offsets), dim3(1024), 0, s, (const float2 *)x->S,
                       (const double *)x->pw0, (const double *)x->pw1, (int)avg, d_s, d_peak, d_std,
                       (const float2 *)x->fft_img, (const float2 *)x->tw32k);
    XC_TRY(x, hipGetLastError());
    return SDBE_OK;
}

}  // extern "C"
