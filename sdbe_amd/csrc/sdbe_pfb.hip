// gfx950 polyphase filterbank (PFB) and its least-squares inverse behind the
// C-ABI of include/sdbe_pfb.h.
//
// Geometry: blocks of L = 32768 real samples, 16385 bins, 4 taps.
//   forward  spec_i = rfft_L( sum_p w[p L + n] x[(i + p) L + n] )
//            (equal to every 4th bin of the rfft of the windowed 4 L samples,
//            software/prototyping/cuda/pfb_inverse.cu:172-208)
//   inverse  yh_i = irfft_L(spec_i); per branch n, with P[i][j] = w[n + L (j - i)]
//            (0 <= j - i < 4): solve (P P^T) z = yh[., n], x[., n] = P^T z
//            (the minimum-norm least-squares solution; pfb_inverse.cu:213-488
//            sets up the same band matrices, its solve is compiled out)
//
// Kernels:
//   k_pfb_fold_r2c  one workgroup per spectrum: 4-tap fold, packed R2C
//                   (16384-point complex FFT in LDS + split post-processing)
//   k_pfb_fold2_r2c the same for calls of more spectra than CUs, two at a time
//   k_pfb_c2r       packed C2R of each spectrum to the pseudo-timestream
// The solve, for any prototype without zeros together on the unit circle:
//   k_pfb_spectral  once per plan, one thread per branch: the constant
//                   minimum-phase factor of P P^T and the tables built on it
//   k_pfb_span, k_pfb_join, k_pfb_solve
//                   two recursive filters, block-parallel over the rows
//   k_pfb_corner    calls of up to 256 rows: their tables, then k_pfb_solve alone
// and for the others the factor-row kernels:
//   k_pfb_factor    once per plan, one thread per branch: banded Cholesky of
//                   P P^T (bandwidth 3, Toeplitz per branch), FP64; the factor's
//                   state is checkpointed every 16 rows
//   k_pfb_fspan, k_pfb_scan, k_pfb_ffin
//                   forward substitution, one thread per (branch, 256-row span):
//                   span transfers, a per-branch scan of the incoming states,
//                   the span from its true state
//   k_pfb_bspan, k_pfb_scan, k_pfb_bfin
//                   back substitution likewise (16-row chunks from the last, factor
//                   rows recomputed from the checkpoints), the final pass emitting
//                   the 4-tap projection x = P^T z
// The solve is FP64: P P^T is badly conditioned for the branches whose tap
// polynomial has a zero near z = -1 (condition ~ (nblock / pi)^2 for a
// symmetric prototype near the middle branch).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <new>
#include <vector>

#include "sdbe_device.hpp"
#include "../../include/sdbe_pfb.h"
#include "../../include/sdbe_stage.h"

using namespace sdbe;

namespace {

constexpr int LB = SDBE_PFB_LBLOCK;       // 32768
constexpr int NH = LB / 2;                // 16384-point complex FFT
constexpr int NBIN = SDBE_PFB_NBINS;      // 16385
constexpr int NT = SDBE_PFB_NTAP;         // 4
constexpr int SEG = 16;                   // factor checkpoint spacing, backward chunk
constexpr int SPAN = 256;                 // rows per thread in the span-parallel solves
constexpr int CKW = 6;                    // doubles per factor checkpoint
constexpr int SOLVE_WG = 64;

static_assert(NH == NCH, "the PFB reuses the 16384-point FFT");

// s + S i w d, in four fused multiply-adds (two roundings a component)
template <int S> __device__ __forceinline__ float2 add_i_mul(float2 s, float2 w, float2 d) {
    constexpr float f = (float)S;
    return make_float2(fmaf(-f * w.x, d.y, fmaf(-f * w.y, d.x, s.x)), fmaf(f * w.x, d.x, fmaf(-f * w.y, d.y, s.y)));
}

// e^{2 pi i (t + 1024 q)/L} from T = e^{2 pi i t/L}: the product in FP64, which this
// chip issues at FP32's rate, so that its one rounding is a table entry's (the
// product of two FP32 factors raised the error of the whole transform by 3 to 4%).
__device__ __forceinline__ float2 split_tw(double2 T, int q) {
    const double c = __builtin_cos(6.283185307179586476925286766559 * q / 32),
                 s = __builtin_sin(6.283185307179586476925286766559 * q / 32);
    return make_float2((float)fma(T.x, c, -T.y * s), (float)fma(T.x, s, T.y * c));
}

// The split of a packed transform, Z (element t + 1024 q in v[q]) to bins k = t +
// 1024 q of out: X[k] = 1/2 (Z[k] + conj Z[N-k]) - 1/2 i e^{-2 pi i k/L} (Z[k] - conj Z[N-k]),
// the mirror bins through LDS.
__device__ __forceinline__ void r2c_split(float2 (&v)[16], float *lds, int t, const double2 *__restrict__ tw1k,
                                          float2 *__restrict__ out) {
    const double2 T = tw1k[t];
    __syncthreads();                         // the FFT's last LDS reads are done
    const int rd = lds_re(t);
#pragma unroll
    for (int q = 0; q < 16; ++q) lds_put(lds, rd + 2048 * q, v[q]);
    __syncthreads();
    // mirror of t + 1024 q: (1024 - t) + 1024 (15 - q); t = 0: 1024 ((16 - q) & 15)
    const int rm = lds_re((1024 - t) & 1023);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int mq = t == 0 ? (16 - q) & 15 : 15 - q;
        const float2 zm = cconj(lds_get(lds, rm + 2048 * mq));   // conj Z[N - k]
        const float2 E = cscale(cadd(v[q], zm), 0.5f);
        const float2 D = cscale(csub(v[q], zm), 0.5f);
        // streamed out: ordinary stores evict the blocks the neighbours read again
        __builtin_nontemporal_store(
            __builtin_bit_cast(uint64_t, add_i_mul<-1>(E, cconj(split_tw(T, q)), D)),
            reinterpret_cast<uint64_t *>(out + t + 1024 * q));
    }
    if (t == 0) out[NH] = make_float2(v[0].x - v[0].y, 0.f);
}

// Forward PFB of spectrum i.  z[m] = y[2m] + i y[2m+1] of the folded block;
// Z = FFT_16384(z); X[k] = 1/2 (Z[k] + conj Z[N-k]) - 1/2 i e^{-2 pi i k/L} (Z[k] - conj Z[N-k]),
// X[N] = Re Z[0] - Im Z[0].
// Spectra are contiguous per XCD (xcd_contig): the workgroups in flight on an
// XCD fold neighbouring spectra, whose 4-block input windows overlap by 3
// blocks, so most block reads are hits in that XCD's L2.
__global__ void __launch_bounds__(1024)
k_pfb_fold_r2c(const float *__restrict__ x, const float *__restrict__ win, float2 *__restrict__ spec,
               const float2 *__restrict__ fft_img, const double2 *__restrict__ tw1k) {
    __shared__ float lds[LDS_FFT_N];
    __shared__ FftTw ftw;
    fft_tw_load(&ftw, fft_img);
    const int i = xcd_contig((int)blockIdx.x, (int)gridDim.x), t = threadIdx.x;
    const float2 *xb = reinterpret_cast<const float2 *>(x + (size_t)i * LB);
    const float2 *wb = reinterpret_cast<const float2 *>(win);
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int m = t + 1024 * q;
        float2 acc = make_float2(0.f, 0.f);
#pragma unroll
        for (int p = 0; p < NT; ++p) {
            const float2 xv = xb[(size_t)p * NH + m];
            const float2 wv = wb[(size_t)p * NH + m];
            acc.x = fmaf(wv.x, xv.x, acc.x);
            acc.y = fmaf(wv.y, xv.y, acc.y);
        }
        v[q] = acc;
    }
    fft16k<-1>(v, lds, &ftw);
    r2c_split(v, lds, t, tw1k, spec + (size_t)i * NBIN);
}

// The forward transform of calls of more spectra than CUs: persistent, two
// consecutive spectra at a time.  Folding one spectrum reads 4 blocks and 4 blocks
// of taps, 1 MB through the CU's L1 (7 us at its 64 bytes a clock, beside 9 us of
// transform); two read 5 and 4 together, and the second's folded samples wait in
// 32 registers while the first is transformed (one copy of the transform's code,
// looped: with two the allocator spills 200 registers).  The pairs of an XCD are
// neighbours, whose blocks overlap.  4096 spectra: 383 us (424 with ordinary
// stores); one spectrum per workgroup 567; a fold pass of its own and a
// persistent transform 186 + 247.  400 spectra: 42 and 53 us.
__global__ void __launch_bounds__(1024)
k_pfb_fold2_r2c(const float *__restrict__ x, int n, const float *__restrict__ win, float2 *__restrict__ spec,
                const float2 *__restrict__ fft_img, const double2 *__restrict__ tw1k) {
    __shared__ float lds[LDS_FFT_N];
    __shared__ FftTw ftw;
    fft_tw_load(&ftw, fft_img);
    const int pairs = (n + 1) >> 1;
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc((void *)win, 0, NT * LB * (int)sizeof(float), 0x00020000);
    for (int p = xcd_contig((int)blockIdx.x, (int)gridDim.x); p < pairs; p += (int)gridDim.x) {
        const int i = 2 * p;
        const int blocks = min(NT + 1, n + NT - 1 - i);       // 4 when spectrum i + 1 does not exist
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(x + (size_t)i * LB), 0, blocks * LB * (int)sizeof(float), 0x00020000);
        const int last = 4 * LB * (blocks - 1);
        float2 a[16], b[16], w[2][NT], v[2][NT + 1];
        const int t0 = row_tid();
        // one q ahead: with more in flight the sums spill (2 ahead 462 us, 3 475)
        auto fetch = [&](int q) {
#pragma unroll
            for (int k = 0; k < NT; ++k)
                w[q & 1][k] = __builtin_bit_cast(
                    float2, __builtin_amdgcn_raw_buffer_load_b64(rw, 8 * t0, 4 * LB * k + 8192 * q, 0));
#pragma unroll
            for (int k = 0; k <= NT; ++k)
                v[q & 1][k] = __builtin_bit_cast(
                    float2, __builtin_amdgcn_raw_buffer_load_b64(rx, 8 * t0, (k < NT ? 4 * LB * k : last) + 8192 * q, 0));
        };
        fetch(0);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            if (q < 15) fetch(q + 1);
            __builtin_amdgcn_sched_barrier(0);
            a[q] = b[q] = make_float2(0.f, 0.f);
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                const float2 wk = w[q & 1][k], va = v[q & 1][k], vb = v[q & 1][k + 1];
                a[q].x = fmaf(wk.x, va.x, a[q].x);
                a[q].y = fmaf(wk.y, va.y, a[q].y);
                b[q].x = fmaf(wk.x, vb.x, b[q].x);
                b[q].y = fmaf(wk.y, vb.y, b[q].y);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll 1
        for (int h = 0; h < 2 && i + h < n; ++h) {            // workgroup-uniform
            const int t = row_tid();
            fft16k_p123<-1>(a, lds, &ftw, t);
            fft16k_p4<-1>(a, &ftw, t);
            r2c_split(a, lds, t, tw1k, spec + (size_t)(i + h) * NBIN);
#pragma unroll
            for (int q = 0; q < 16; ++q) a[q] = b[q];
        }
    }
}

// Pseudo-timestream of spectrum i: Z[k] = (X[k] + conj X[N-k]) + i e^{2 pi i k/L} (X[k] - conj X[N-k])
// (imaginary parts of X[0], X[N] dropped), z = IFFT_16384(Z) / L, samples (2m, 2m+1) = (Re, Im) z[m]
// -- numpy's irfft.  Persistent, one workgroup per CU: the next spectrum's bins
// and mirror bins (64 registers) load while the last pass and the stores of the
// current one run (LOOP false: a workgroup per spectrum, nothing to load ahead).
// 4096 spectra: 262 us, 4.1 TB/s of the 1.07 GB it must move (not persistent, the
// twiddles from memory: 330).
template <bool LOOP>
__global__ void __launch_bounds__(1024)
k_pfb_c2r(const float2 *__restrict__ spec, int n, float *__restrict__ yh, const float2 *__restrict__ fft_img,
          const double2 *__restrict__ tw1k) {
    __shared__ float lds[LDS_FFT_N];
    __shared__ FftTw ftw;
    fft_tw_load(&ftw, fft_img);
    const int t = threadIdx.x;
    const float sc = 1.0f / (float)LB;
    auto rsrc = [&](int row) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(spec + (size_t)row * NBIN), 0, NBIN * (int)sizeof(float2),
                                                 0x00020000);
    };
    // bin k = t + 1024 q, and N - k = (1024 - t) + 1024 (15 - q); k = 0 pairs with bin N
    auto bin = [&](__amdgpu_buffer_rsrc_t rs, int q) {
        return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, 8 * t, 8192 * q, 0));
    };
    auto mirror = [&](__amdgpu_buffer_rsrc_t rs, int q) {
        return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, 8 * (1024 - t), 8192 * (15 - q), 0));
    };
    float2 a[16], b[16];
    int row = blockIdx.x;
    __amdgpu_buffer_rsrc_t rs = rsrc(row);
#pragma unroll
    for (int q = 0; q < 16; ++q) a[q] = bin(rs, q);
#pragma unroll
    for (int q = 0; q < 16; ++q) b[q] = mirror(rs, q);
    for (;;) {
        const int next = row + (int)gridDim.x, tr = row_tid();
        const double2 T = tw1k[tr];
        float2 v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            if (q == 0 && tr == 0) a[0].y = b[0].y = 0.f;
            const float2 sum = cadd(a[q], cconj(b[q])), dif = csub(a[q], cconj(b[q]));
            v[q] = add_i_mul<+1>(sum, split_tw(T, q), dif);
        }
        fft16k_p12<+1>(v, lds, &ftw, tr);
        fft16k_p3w<+1>(v, lds, &ftw, tr);
        if (LOOP) {
            // the bins before the last pass, the mirror bins as its outputs leave
            // their registers; the last spectrum loads itself again
            rs = rsrc(next < n ? next : row);
#pragma unroll
            for (int q = 0; q < 16; ++q) a[q] = bin(rs, q);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int T0 = fft16k_tord(tr);            // z[T0 + 1024 q] in v[q]
        float2 *dst = reinterpret_cast<float2 *>(yh + (size_t)row * LB) + T0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            fft16k_p4_one<+1>(v, &ftw, T0, g);
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[1024 * (g + 4 * r)] = cscale(v[g + 4 * r], sc);
            if (LOOP) {
#pragma unroll
                for (int r = 0; r < 4; ++r) b[4 * g + r] = mirror(rs, 4 * g + r);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!LOOP || next >= n) break;
        row = next;
    }
}

// One row of the banded Cholesky factor of the Toeplitz band (a0, a1, a2, a3):
// inv0 = 1 / L(i, i), dk = L(i, i - k).  r1, r2, r3 are rows i - 1, i - 2,
// i - 3 ({1, 0, 0, 0} before the first row).  Keeping the reciprocal of the
// diagonal makes a row one reciprocal square root and fused multiply-adds: the
// rows form a dependent chain, and FP64 division and square root are
// multi-instruction sequences that would sit on it four times per row.
struct Row {
    double inv0, d1, d2, d3;
};

template <bool EDGE = true>
__device__ __forceinline__ Row chol_row(int i, double a0, double a1, double a2, double a3, const Row &r1,
                                        const Row &r2, const Row &r3) {
    // rows 0..2 see fewer band entries; EDGE false is for rows i >= 3
    const double e1 = !EDGE || i >= 1 ? a1 : 0.0, e2 = !EDGE || i >= 2 ? a2 : 0.0, e3 = !EDGE || i >= 3 ? a3 : 0.0;
    Row r;
    r.d3 = e3 * r3.inv0;
    r.d2 = (e2 - r.d3 * r2.d1) * r2.inv0;
    r.d1 = (e1 - r.d3 * r1.d2 - r.d2 * r1.d1) * r1.inv0;
    r.inv0 = rsqrt(a0 - r.d1 * r.d1 - r.d2 * r.d2 - r.d3 * r.d3);
    return r;
}

// The banded solves run span-parallel: thread (branch n, span s) covers rows
// s0 = 256 s .. s1 - 1 (s1 = min(s0 + 256, nblock)).  A substitution is a
// linear recurrence of order 3, so a span's output is its particular solution
// (zero incoming state) plus a 3 x 3 transfer of the incoming state; per branch,
// a scan over the spans composes the transfers into each span's true incoming
// state, and a final pass recomputes the span from it.  The factor rows are
// data-independent: the factor's state at every 16th row is checkpointed once,
// at plan creation (k_pfb_factor), and rows are recomputed from it.  Span and
// checkpoint layouts put the branch index innermost, [s][k][32768], so every
// access is coalesced.

// A factor row needs, of the three rows before it, r1 = {inv0, d1, d2},
// r2 = {inv0, d1} and r3 = {inv0}: ckpt[c][6][LB] holds them for rows
// 16 c - 1, 16 c - 2, 16 c - 3.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_factor(int nck, const double *__restrict__ a, double *__restrict__ ckpt) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    const double a0 = a[n], a1 = a[LB + n], a2 = a[2 * LB + n], a3 = a[3 * LB + n];
    Row r1 = {1.0, 0.0, 0.0, 0.0}, r2 = r1, r3 = r1;
    for (int c = 0; c < nck; ++c) {
        double *ck = ckpt + (size_t)c * CKW * LB + n;
        const double st[CKW] = {r1.inv0, r1.d1, r1.d2, r2.inv0, r2.d1, r3.inv0};
#pragma unroll
        for (int k = 0; k < CKW; ++k) ck[(size_t)k * LB] = st[k];
        for (int k = 0; k < SEG; ++k) {
            const Row r = chol_row(c * SEG + k, a0, a1, a2, a3, r1, r2, r3);
            r3 = r2;
            r2 = r1;
            r1 = r;
        }
    }
}

// The six checkpoint doubles of chunk c, and the three rows before it.
struct Ckpt {
    double v[CKW];
};

__device__ __forceinline__ Ckpt load_ckpt(const double *__restrict__ ckpt, int c, int n) {
    const double *ck = ckpt + (size_t)c * CKW * LB + n;
    Ckpt r;
#pragma unroll
    for (int k = 0; k < CKW; ++k) r.v[k] = ck[(size_t)k * LB];
    return r;
}

__device__ __forceinline__ void ckpt_rows(const Ckpt &c, Row &r1, Row &r2, Row &r3) {
    r1 = Row{c.v[0], c.v[1], c.v[2], 0.0};
    r2 = Row{c.v[3], c.v[4], 0.0, 0.0};
    r3 = Row{c.v[5], 0.0, 0.0, 0.0};
}

__device__ __forceinline__ void load_band(const double *__restrict__ a, int n, double &a0, double &a1,
                                          double &a2, double &a3) {
    a0 = a[n];
    a1 = a[LB + n];
    a2 = a[2 * LB + n];
    a3 = a[3 * LB + n];
}

// A span pass runs either the particular solution (one chain, zero incoming
// state, the data as right-hand side) or the three responses to unit incoming
// states (no data).  The responses are data-independent and, for every span
// that is full, independent of the number of rows: they are computed once per
// plan for full spans.  The last span of a call may be partial, and its
// transfer is never used (forward: its outgoing state ends the scan; backward:
// its incoming state is zero).  Output [s][3 NC][LB], index 3 j + c = state
// component c of chain j.
template <int NC>
__device__ __forceinline__ void chains_init(double (&st)[NC][3]) {
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c) st[j][c] = (NC == 3 && j == c) ? 1.0 : 0.0;
}

template <int NC>
__device__ __forceinline__ void chains_store(double *__restrict__ out, int sp, int n, const double (&st)[NC][3]) {
    double *o = out + (size_t)sp * 3 * NC * LB + n;
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c) o[(size_t)(3 * j + c) * LB] = st[j][c];
}

// Chunks are 16 rows from a multiple of 16.  GEN handles the general chunk
// (the first rows of the matrix, a partial last chunk); the others take the
// path with no row tests.
template <bool GEN, int NC, bool HOM>
__device__ __forceinline__ void fchunk(int c0, int s1, const float (&y)[SEG], double a0, double a1, double a2,
                                       double a3, Row &r1, Row &r2, Row &r3, double (&st)[NC][3]) {
#pragma unroll
    for (int k = 0; k < SEG; ++k) {
        if (!GEN || c0 + k < s1) {
            const Row r = chol_row<GEN>(c0 + k, a0, a1, a2, a3, r1, r2, r3);
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const double rhs = HOM ? 0.0 : (double)y[k];
                const double ui = (rhs - r.d1 * st[j][0] - r.d2 * st[j][1] - r.d3 * st[j][2]) * r.inv0;
                st[j][2] = st[j][1];
                st[j][1] = st[j][0];
                st[j][0] = ui;
            }
            r3 = r2;
            r2 = r1;
            r1 = r;
        }
    }
}

// Forward L u = yh[., n]: per span the final state (u[s1-1], u[s1-2], u[s1-3])
// of the particular solution (HOM false, out = p[s][3][LB]) or of the
// responses to (u[s0-1], u[s0-2], u[s0-3]) = e_j (HOM true, out = M[s][9][LB]).
template <bool HOM>
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_fspan(const float *__restrict__ yh, int nblock, const double *__restrict__ a,
            const double *__restrict__ ckpt, double *__restrict__ out) {
    constexpr int NC = HOM ? 3 : 1;
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, sp = blockIdx.y, s0 = sp * SPAN;
    const int s1 = min(s0 + SPAN, nblock);
    double a0, a1, a2, a3;
    load_band(a, n, a0, a1, a2, a3);
    Row r1, r2, r3;
    ckpt_rows(load_ckpt(ckpt, s0 / SEG, n), r1, r2, r3);
    double st[NC][3];
    chains_init<NC>(st);
    for (int c0 = s0; c0 < s1; c0 += SEG) {
        float y[SEG];
#pragma unroll
        for (int k = 0; k < SEG; ++k) y[k] = HOM ? 0.f : yh[(size_t)min(c0 + k, nblock - 1) * LB + n];
        if (c0 >= SEG && c0 + SEG <= s1)
            fchunk<false, NC, HOM>(c0, s1, y, a0, a1, a2, a3, r1, r2, r3, st);
        else
            fchunk<true, NC, HOM>(c0, s1, y, a0, a1, a2, a3, r1, r2, r3, st);
    }
    chains_store<NC>(out, sp, n, st);
}

// Per branch: the incoming state of every span, state[s][3][LB], from the
// particular states p[s][3][LB] and the transfers M[s][9][LB].
// Forward (dir +1): state_0 = 0, state_{s+1} = M_s state_s + p_s;
// backward (dir -1): from the last span down.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_scan(const double *__restrict__ pst, const double *__restrict__ mt, int nspan, int dir,
           double *__restrict__ state) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    double x0 = 0.0, x1 = 0.0, x2 = 0.0;
    for (int i = 0; i < nspan; ++i) {
        const int sp = dir > 0 ? i : nspan - 1 - i;
        double *st = state + (size_t)sp * 3 * LB + n;
        st[0] = x0;
        st[(size_t)LB] = x1;
        st[(size_t)2 * LB] = x2;
        const double *pp = pst + (size_t)sp * 3 * LB + n;
        const double *t = mt + (size_t)sp * 9 * LB + n;
        double m[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) m[k] = t[(size_t)k * LB];
        const double y0 = pp[0] + m[0] * x0 + m[3] * x1 + m[6] * x2;
        const double y1 = pp[(size_t)LB] + m[1] * x0 + m[4] * x1 + m[7] * x2;
        const double y2 = pp[(size_t)2 * LB] + m[2] * x0 + m[5] * x1 + m[8] * x2;
        x0 = y0;
        x1 = y1;
        x2 = y2;
    }
}

template <bool GEN>
__device__ __forceinline__ void ffchunk(int c0, int s1, const float (&y)[SEG], double a0, double a1, double a2,
                                        double a3, Row &r1, Row &r2, Row &r3, double (&st)[3]) {
#pragma unroll
    for (int k = 0; k < SEG; ++k) {
        if (!GEN || c0 + k < s1) {
            const Row r = chol_row<GEN>(c0 + k, a0, a1, a2, a3, r1, r2, r3);
            const double ui = ((double)y[k] - r.d1 * st[0] - r.d2 * st[1] - r.d3 * st[2]) * r.inv0;
            st[2] = st[1];
            st[1] = st[0];
            st[0] = ui;
            r3 = r2;
            r2 = r1;
            r1 = r;
        }
    }
}

// Forward, final pass: the span from its true incoming state.  u itself is not
// stored: the state entering every 16-row chunk, uck[c][3][LB] = (u[16c-1],
// u[16c-2], u[16c-3]), is, and the backward passes recompute a chunk's u from it
// and yh along with the chunk's factor rows.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_ffin(const float *__restrict__ yh, int nblock, const double *__restrict__ a,
           const double *__restrict__ ckpt, const double *__restrict__ state, double *__restrict__ uck) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, sp = blockIdx.y, s0 = sp * SPAN;
    const int s1 = min(s0 + SPAN, nblock);
    double a0, a1, a2, a3;
    load_band(a, n, a0, a1, a2, a3);
    Row r1, r2, r3;
    ckpt_rows(load_ckpt(ckpt, s0 / SEG, n), r1, r2, r3);
    const double *st = state + (size_t)sp * 3 * LB + n;
    double st3[3] = {st[0], st[(size_t)LB], st[(size_t)2 * LB]};   // u[i-1], u[i-2], u[i-3]
    for (int c0 = s0;; c0 += SEG) {
        double *uc = uck + (size_t)(c0 / SEG) * 3 * LB + n;
        uc[0] = st3[0];
        uc[(size_t)LB] = st3[1];
        uc[(size_t)2 * LB] = st3[2];
        if (c0 + SEG >= s1) break;   // the span's last chunk feeds no later chunk
        float y[SEG];
#pragma unroll
        for (int k = 0; k < SEG; ++k) y[k] = yh[(size_t)(c0 + k) * LB + n];
        if (c0 >= SEG)
            ffchunk<false>(c0, s1, y, a0, a1, a2, a3, r1, r2, r3, st3);
        else
            ffchunk<true>(c0, s1, y, a0, a1, a2, a3, r1, r2, r3, st3);
    }
}

// Factor rows 16 c + k0 .. 16 c + k0 + K - 1 into Lx[k0 ..] from checkpoint
// c's rows (k0 = 0, K = 16: the chunk; rows after it are the next chunk's first).
template <int K, bool GEN = true>
__device__ __forceinline__ void chunk_rows(const Ckpt &ck, int row0, double a0, double a1, double a2, double a3,
                                           Row *Lx) {
    Row r1, r2, r3;
    ckpt_rows(ck, r1, r2, r3);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        Lx[k] = chol_row<GEN>(row0 + k, a0, a1, a2, a3, r1, r2, r3);
        r3 = r2;
        r2 = r1;
        r1 = Lx[k];
    }
}

// The chunk's u (forward substitution from the state entering the chunk, with
// the factor rows just recomputed), for the backward passes.
__device__ __forceinline__ void chunk_u(const Row (&Lx)[SEG + 3], const float (&y)[SEG], const double (&us)[3],
                                        double (&uu)[SEG]) {
    double w1 = us[0], w2 = us[1], w3 = us[2];
#pragma unroll
    for (int k = 0; k < SEG; ++k) {
        const double ui = ((double)y[k] - Lx[k].d1 * w1 - Lx[k].d2 * w2 - Lx[k].d3 * w3) * Lx[k].inv0;
        uu[k] = ui;
        w3 = w2;
        w2 = w1;
        w1 = ui;
    }
}

template <bool GEN, int NC, bool HOM>
__device__ __forceinline__ void bchunk(const Ckpt &ck, int c0, int s1, const float (&y)[SEG], const double (&us)[3],
                                       double a0, double a1, double a2, double a3, Row (&Lx)[SEG + 3],
                                       double (&st)[NC][3]) {
    chunk_rows<SEG, GEN>(ck, c0, a0, a1, a2, a3, Lx);
    double uu[SEG];
    if constexpr (!HOM) chunk_u(Lx, y, us, uu);
#pragma unroll
    for (int k = SEG - 1; k >= 0; --k) {
        if (!GEN || c0 + k < s1) {
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                double rhs = 0.0;
                if constexpr (!HOM) rhs = uu[k];
                const double zi = (rhs - Lx[k + 1].d1 * st[j][0] - Lx[k + 2].d2 * st[j][1] -
                                   Lx[k + 3].d3 * st[j][2]) * Lx[k].inv0;
                st[j][2] = st[j][1];
                st[j][1] = st[j][0];
                st[j][0] = zi;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) Lx[SEG + k] = Lx[k];
}

// Backward L^T z = u: per span, in 16-row chunks from the last, the final state
// (z[s0], z[s0+1], z[s0+2]) of the particular solution (HOM false, out =
// p[s][3][LB]) or of the responses to (z[s1], z[s1+1], z[s1+2]) = e_j (HOM
// true, out = M[s][9][LB]).  Row i uses L(i+1, i), L(i+2, i), L(i+3, i):
// chunk c keeps its rows in Lx[0..15] and the three following rows in
// Lx[16..18].  The next chunk's checkpoint is loaded one chunk ahead.
template <bool HOM>
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_bspan(const float *__restrict__ yh, const double *__restrict__ uck, int nblock, const double *__restrict__ a,
            const double *__restrict__ ckpt, double *__restrict__ out) {
    constexpr int NC = HOM ? 3 : 1;
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, sp = blockIdx.y, s0 = sp * SPAN;
    const int s1 = min(s0 + SPAN, nblock);
    const int chi = (s1 - 1) / SEG, clo = s0 / SEG;
    double a0, a1, a2, a3;
    load_band(a, n, a0, a1, a2, a3);
    Row Lx[SEG + 3];
    chunk_rows<3>(load_ckpt(ckpt, chi + 1, n), (chi + 1) * SEG, a0, a1, a2, a3, Lx + SEG);
    Ckpt ck = load_ckpt(ckpt, chi, n);
    double st[NC][3];
    chains_init<NC>(st);
    for (int c = chi; c >= clo; --c) {
        const int c0 = c * SEG;
        float y[SEG];
        double us[3] = {0.0, 0.0, 0.0};
        if constexpr (!HOM) {
#pragma unroll
            for (int k = 0; k < SEG; ++k) y[k] = yh[(size_t)min(c0 + k, nblock - 1) * LB + n];
            const double *uc = uck + (size_t)c * 3 * LB + n;
            us[0] = uc[0];
            us[1] = uc[(size_t)LB];
            us[2] = uc[(size_t)2 * LB];
        }
        const Ckpt ckn = load_ckpt(ckpt, max(c - 1, clo), n);
        if (c0 >= SEG && c0 + SEG <= s1)
            bchunk<false, NC, HOM>(ck, c0, s1, y, us, a0, a1, a2, a3, Lx, st);
        else
            bchunk<true, NC, HOM>(ck, c0, s1, y, us, a0, a1, a2, a3, Lx, st);
        ck = ckn;
    }
    chains_store<NC>(out, sp, n, st);
}

template <bool GEN>
__device__ __forceinline__ void bfchunk(const Ckpt &ck, int c0, int s1, const float (&y)[SEG], const double (&us)[3],
                                        double a0, double a1, double a2, double a3, const double (&w)[4],
                                        Row (&Lx)[SEG + 3], double (&z)[3], float *__restrict__ xc) {
    chunk_rows<SEG, GEN>(ck, c0, a0, a1, a2, a3, Lx);
    double uu[SEG];
    chunk_u(Lx, y, us, uu);
#pragma unroll
    for (int k = SEG - 1; k >= 0; --k) {
        if (!GEN || c0 + k < s1) {
            const double zi = (uu[k] - Lx[k + 1].d1 * z[0] - Lx[k + 2].d2 * z[1] - Lx[k + 3].d3 * z[2]) * Lx[k].inv0;
            xc[(size_t)k * LB] = (float)(w[0] * z[2] + w[1] * z[1] + w[2] * z[0] + w[3] * zi);
            z[2] = z[1];
            z[1] = z[0];
            z[0] = zi;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) Lx[SEG + k] = Lx[k];
}

// Backward, final pass: z of the span from its true incoming state and the
// 4-tap projection x = P^T z: x[i + 3] = w0 z[i+3] + w1 z[i+2] + w2 z[i+1] + w3 z[i]
// for the span's rows i; span 0 also emits x[0..2] (z[i] = 0 for i < 0).
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_bfin(const float *__restrict__ yh, const double *__restrict__ uck, int nblock, const double *__restrict__ a,
           const double *__restrict__ ckpt, const double *__restrict__ state, const float *__restrict__ win,
           float *__restrict__ x) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, sp = blockIdx.y, s0 = sp * SPAN;
    const int s1 = min(s0 + SPAN, nblock);
    const int chi = (s1 - 1) / SEG, clo = s0 / SEG;
    double a0, a1, a2, a3;
    load_band(a, n, a0, a1, a2, a3);
    const double w[4] = {win[n], win[LB + n], win[2 * LB + n], win[3 * LB + n]};
    Row Lx[SEG + 3];
    chunk_rows<3>(load_ckpt(ckpt, chi + 1, n), (chi + 1) * SEG, a0, a1, a2, a3, Lx + SEG);
    Ckpt ck = load_ckpt(ckpt, chi, n);
    const double *st = state + (size_t)sp * 3 * LB + n;
    double z[3] = {st[0], st[(size_t)LB], st[(size_t)2 * LB]};   // z[i+1], z[i+2], z[i+3]
    for (int c = chi; c >= clo; --c) {
        const int c0 = c * SEG;
        float y[SEG];
#pragma unroll
        for (int k = 0; k < SEG; ++k) y[k] = yh[(size_t)min(c0 + k, nblock - 1) * LB + n];
        const double *uc = uck + (size_t)c * 3 * LB + n;
        const double us[3] = {uc[0], uc[(size_t)LB], uc[(size_t)2 * LB]};
        const Ckpt ckn = load_ckpt(ckpt, max(c - 1, clo), n);
        float *xc = x + (size_t)(c0 + 3) * LB + n;
        if (c0 >= SEG && c0 + SEG <= s1)
            bfchunk<false>(ck, c0, s1, y, us, a0, a1, a2, a3, w, Lx, z, xc);
        else
            bfchunk<true>(ck, c0, s1, y, us, a0, a1, a2, a3, w, Lx, z, xc);
        ck = ckn;
    }
    if (sp == 0) {
        x[(size_t)2 * LB + n] = (float)(w[0] * z[2] + w[1] * z[1] + w[2] * z[0]);
        x[(size_t)LB + n] = (float)(w[0] * z[1] + w[1] * z[0]);
        x[n] = (float)(w[0] * z[0]);
    }
}

// --------------------------------------------- constant-coefficient solve
// P P^T is Toeplitz per branch, so it has a constant minimum-phase factor b:
// b(q) = b0 + b1 q + b2 q^2 + b3 q^3 with the taps' autocorrelation and no zero
// inside the unit circle (the taps' polynomial with its zeros inside reflected),
// and with B the lower-triangular Toeplitz matrix of b
//   P P^T = B B^T + E H H^T E^T,   H[i][m] = b_{i+m+1}  (E: the first three rows).
// B B^T is two recursive filters with three constant coefficients beta = b_k / b0
// (no factor rows to recompute or checkpoint), and the corner is a rank-3
// correction: with z0 the filters' solution, g = W z0[0..2] is taken off the
// first three right-hand sides, W = H (I + H^T G H)^-1 H^T, G the first 3 x 3
// block of (B B^T)^-1.  In scaled units v = b0 B^-1 y, zeta = b0^2 z:
//   v_i = y_i - beta1 v_{i-1} - beta2 v_{i-2} - beta3 v_{i-3},
//   zeta_i = v_i - beta1 zeta_{i+1} - beta2 zeta_{i+2} - beta3 zeta_{i+3}.
// Rounding: the tables are computed in double-double and the corner takes one
// refinement step, so the FP32 rounding of yh is all that is left in the result.
// Against an 80-bit solve, over the 280 worst branches of a Hamming prototype
// (double zeros near -0.995): 1.65e-7 to 1.79e-7 at 256 to 4096 rows, where the
// FP64 factor rows are themselves off by up to 3.0e-7 (4096 rows).  The exception is
// two zeros together on the unit circle: taps 1, 2, 1 lose 5e-5 in 1000 rows here
// and 1e-8 by factor rows.
// k_pfb_spectral counts such branches, and a plan that has any takes those.
//
// Thread (branch, span of 32 rows) keeps its rows' v in registers; a workgroup
// holds 64 branches x 8 spans and scans the spans' boundary states through LDS.
// Up to 256 rows that is the whole problem.  Above, k_pfb_span takes every
// 256-row block's outgoing states in both directions (from zero incoming ones) in
// one read of yh, k_pfb_join composes them per branch into the blocks' true
// incoming states with the corner, and k_pfb_solve finishes the blocks: two
// reads of yh and one write of x, all in 256-byte runs.  4096 spectra: span 130 us
// (4.1 TB/s), join 27, solve 225 (4.8 TB/s, the rate of a large copy); the
// factor-row kernels, which read yh four times beside 0.8 GB of checkpoints and
// recompute every factor row four times, take 890.  (Tiles of 8 branches over
// all 4096 rows read yh once, but in 32-byte runs: 700 us.)
constexpr int SR = 32, SWV = 8, SBLK = SR * SWV;     // rows per thread, waves and rows per workgroup
// table rows, [row][LB] doubles
constexpr int TB_BETA = 0;                // beta1..3
constexpr int TB_WZ = 3;                  // taps / b0^2
constexpr int TB_CS = 7;                  // C^32: the state after a span of no input
constexpr int TB_CB = 16;                 // C^256
constexpr int TB_RS = 25;                 // a span's head zeta per unit incoming state
constexpr int TB_HS = 34;                 // its impulse response h27..h31
constexpr int TB_RB = 39;                 // the same of a block: head zeta
constexpr int TB_HB = 48;                 // ... h251..h255
constexpr int TB_GB = 53;                 // ... first 3 x 3 block of (B B^T)^-1
constexpr int TB_N = 62;
// ... and of a call
constexpr int TC_W = 0;                   // corner matrix W (scaled)
constexpr int TC_RS = 9;                  // TB_RS of the partial last span
constexpr int TC_G = 18;                  // more than one block: g
constexpr int TC_N = 21;

// 3 x 3 matrices, m[3 r + c]
__device__ __forceinline__ void mat_mul(double (&o)[9], const double (&a)[9], const double (&b)[9]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) o[3 * r + c] = a[3 * r] * b[c] + a[3 * r + 1] * b[3 + c] + a[3 * r + 2] * b[6 + c];
}

// Double-double: h + l, |l| at most half an ulp of h.
struct Dd {
    double h = 0.0, l = 0.0;
};
__device__ __forceinline__ Dd dd_norm(double h, double l) {
    const double s = h + l;
    return Dd{s, l - (s - h)};
}
__device__ __forceinline__ Dd dd_add(Dd a, Dd b) {
    const double s = a.h + b.h, t = s - a.h;
    return dd_norm(s, (a.h - (s - t)) + (b.h - t) + (a.l + b.l));
}
__device__ __forceinline__ Dd dd_mul(Dd a, Dd b) {
    const double p = a.h * b.h;
    return dd_norm(p, fma(a.h, b.h, -p) + fma(a.h, b.l, a.l * b.h));
}
// a - b c
__device__ __forceinline__ Dd dd_sub_mul(Dd a, Dd b, double c) { return dd_add(a, dd_mul(b, Dd{-c, 0.0})); }

// sum_{k < n} C^k X (C^k)^T (TR) or sum_{k < n} C^k X C^k, by doubling over the
// bits of n.
template <bool TR>
__device__ __forceinline__ void power_sum(int n, const double (&C)[9], const double (&X)[9], double (&S)[9]) {
    double P[9], t[9], u[9];
    auto add = [&](const double (&m)[9], const double (&x)[9]) {   // S = x + m S m(^T)
        mat_mul(t, m, S);
        if (TR) {
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    u[3 * r + c] = t[3 * r] * m[3 * c] + t[3 * r + 1] * m[3 * c + 1] + t[3 * r + 2] * m[3 * c + 2];
        } else {
            mat_mul(u, t, m);
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) S[i] = x[i] + u[i];
    };
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        P[i] = C[i];
        S[i] = n > 0 ? X[i] : 0.0;
    }
    for (int bit = n > 0 ? 30 - __builtin_clz(n) : -1; bit >= 0; --bit) {     // below n's leading bit
        add(P, S);
        mat_mul(t, P, P);
#pragma unroll
        for (int i = 0; i < 9; ++i) P[i] = t[i];
        if ((n >> bit) & 1) {
            add(C, X);
            mat_mul(t, C, P);
#pragma unroll
            for (int i = 0; i < 9; ++i) P[i] = t[i];
        }
    }
}

// Head zeta (rows 0..2, nothing incoming from below) of n rows whose v is the
// response to the incoming state e_c, in column c: v_k = (C^(k+1))[0][c], and
// zeta_r = sum_k v_k h_{k-r} with (h_k, h_{k-1}, h_{k-2}) = C^k e_0.
__device__ __forceinline__ void head_response(int n, double be1, double be2, double be3, double (&rm)[9]) {
    const double C[9] = {-be1, -be2, -be3, 1.0, 0.0, 0.0, 0.0, 1.0, 0.0};
    const double X[9] = {-be1, -be2, -be3, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    power_sum<false>(n, C, X, rm);
}

// Per plan, one thread per branch: the minimum-phase factor and the tables.
// The cubic's real zero by Cardano's formula and Newton steps, deflated from the
// end that keeps the remaining coefficients accurate, then the quadratic.
// *clustered counts the branches with two zeros together on the unit circle.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_spectral(const float *__restrict__ win, double *__restrict__ tab, int *__restrict__ clustered) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    const double w[4] = {win[n], win[LB + n], win[2 * LB + n], win[3 * LB + n]};
    const double sc = fmax(fmax(fabs(w[0]), fabs(w[1])), fmax(fabs(w[2]), fabs(w[3])));
    // c0 x^3 + c1 x^2 + c2 x + c3, |c0| >= |c3| (either order has the autocorrelation),
    // zeros wanted in |x| <= 1
    const bool rev = fabs(w[3]) > fabs(w[0]);
    double c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = (rev ? w[3 - i] : w[i]) / sc;
    double b[4];
    bool close = false;
    if (fabs(c[0]) <= 1e-15) {      // both ends vanish: two taps
        const bool f = fabs(c[1]) >= fabs(c[2]);
        b[0] = f ? c[1] : c[2];
        b[1] = f ? c[2] : c[1];
        b[2] = b[3] = 0.0;
    } else {
        const double A = c[1] / c[0], B = c[2] / c[0], C = c[3] / c[0];
        const double Q = (A * A - 3.0 * B) / 9.0, R = (2.0 * A * A * A - 9.0 * A * B + 27.0 * C) / 54.0;
        double r;
        if (R * R < Q * Q * Q) {    // three real zeros: the largest
            const double th = acos(fmax(-1.0, fmin(1.0, R / sqrt(Q * Q * Q))));
            const double m = -2.0 * sqrt(Q), tau = 6.283185307179586476925286766559;
            r = m * cos(th / 3.0) - A / 3.0;
            for (int k = 1; k < 3; ++k) {
                const double x = m * cos((th + k * tau) / 3.0) - A / 3.0;
                if (fabs(x) > fabs(r)) r = x;
            }
        } else {
            const double s = -copysign(cbrt(fabs(R) + sqrt(fmax(R * R - Q * Q * Q, 0.0))), R);
            r = s + (s != 0.0 ? Q / s : 0.0) - A / 3.0;
        }
        for (int k = 0; k < 4; ++k) {
            const double f = ((r + A) * r + B) * r + C, d = (3.0 * r + 2.0 * A) * r + B;
            if (d == 0.0) break;
            const double x = r - f / d;
            if (!(fabs(((x + A) * x + B) * x + C) < fabs(f))) break;
            r = x;
        }
        // x^2 + d1 x + d0: coefficients above the largest of the terms |C|, |B r|,
        // |A r^2|, |r^3| from the top, those below it from the bottom
        double d1 = A + r, d0 = B + d1 * r;
        if (r != 0.0) {
            const double t0 = fabs(C), t1 = fabs(B * r), t2 = fabs(A * r * r), t3 = fabs(r * r * r);
            if (fmax(t2, t3) > fmax(t0, t1) || t1 > t0) d0 = -C / r;
            if (fmax(t2, t3) > fmax(t0, t1)) d1 = (d0 - B) / r;
        }
        double pol[4] = {c[0], 0.0, 0.0, 0.0};
        auto times = [&](double x) {        // times (x' - x), or reflected: (1 - x x')
            const double u = fabs(x) > 1.0 ? -x : 1.0, v = fabs(x) > 1.0 ? 1.0 : -x;
#pragma unroll
            for (int i = 3; i >= 1; --i) pol[i] = pol[i] * u + pol[i - 1] * v;
            pol[0] *= u;
        };
        auto inside = [](double x) { return fabs(x) > 1.0 ? 1.0 / x : x; };
        times(r);
        bool any = fabs(r) > 1.0;              // a zero was reflected
        const double disc = d1 * d1 - 4.0 * d0, ri = inside(r);
        constexpr double NEAR = 0.998, GAP = 0.02;
        if (disc >= 0.0) {
            const double s = -0.5 * (d1 + copysign(sqrt(disc), d1)), x2 = s != 0.0 ? d0 / s : 0.0;
            times(s);
            times(x2);
            any = any || fabs(s) > 1.0 || fabs(x2) > 1.0;
            const double si = inside(s), xi = inside(x2);
            close = (fmin(fabs(ri), fabs(si)) > NEAR && fabs(ri - si) < GAP) ||
                    (fmin(fabs(ri), fabs(xi)) > NEAR && fabs(ri - xi) < GAP) ||
                    (fmin(fabs(si), fabs(xi)) > NEAR && fabs(si - xi) < GAP);
        } else {
            const bool out = d0 > 1.0;
            any = any || out;
            const double e0 = out ? d0 : 1.0, e2 = out ? 1.0 : d0;
            const double p0 = pol[0], p1 = pol[1];
            pol[0] = p0 * e0;
            pol[1] = p0 * d1 + p1 * e0;
            pol[2] = p0 * e2 + p1 * d1;
            pol[3] = p1 * e2;
            const double re = -0.5 * d1 / e0, im = 0.5 * sqrt(-disc) / e0, mod = sqrt(fmin(d0, 1.0 / d0));
            close = mod > NEAR && (2.0 * im < GAP || (fabs(ri) > NEAR && hypot(ri - re, im) < GAP));
        }
        // taps that are minimum phase already (in either order) are the factor, exactly
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = any ? pol[i] : c[i];
    }
    if (close) atomicAdd(clustered, 1);
    const double be1 = b[1] / b[0], be2 = b[2] / b[0], be3 = b[3] / b[0], b0 = b[0] * sc;
    double *o = tab + n;
    o[(size_t)(TB_BETA + 0) * LB] = be1;
    o[(size_t)(TB_BETA + 1) * LB] = be2;
    o[(size_t)(TB_BETA + 2) * LB] = be3;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[(size_t)(TB_WZ + i) * LB] = w[i] / b0 / b0;
    // The span's and the block's responses, by recursion over their rows in
    // double-double: near-double zeros close to the unit circle (the Hamming
    // prototype has some around branches 4050 and 28720) amplify the tables'
    // rounding into the result, 3e-7 of it with powers by squaring in FP64.
    Dd v[3][3] = {{{1.0, 0.0}, {}, {}}, {{}, {1.0, 0.0}, {}}, {{}, {}, {1.0, 0.0}}};   // chain c: its last three values
    Dd h[3] = {}, rm[9] = {}, g[6] = {};
    for (int k = 0; k < SBLK; ++k) {
        const Dd in{k == 0 ? 1.0 : 0.0, 0.0};
        const Dd hk = dd_sub_mul(dd_sub_mul(dd_sub_mul(in, h[0], be1), h[1], be2), h[2], be3);
        h[2] = h[1];
        h[1] = h[0];
        h[0] = hk;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const Dd x = dd_sub_mul(dd_sub_mul(dd_sub_mul(Dd{}, v[c][0], be1), v[c][1], be2), v[c][2], be3);
            v[c][2] = v[c][1];
            v[c][1] = v[c][0];
            v[c][0] = x;
#pragma unroll
            for (int r = 0; r < 3; ++r) rm[3 * r + c] = dd_add(rm[3 * r + c], dd_mul(x, h[r]));
        }
#pragma unroll
        for (int r = 0, i = 0; r < 3; ++r)
#pragma unroll
            for (int c = r; c < 3; ++c, ++i) g[i] = dd_add(g[i], dd_mul(h[r], h[c]));
        if (k < SR && k >= SR - 5) o[(size_t)(TB_HS + k - (SR - 5)) * LB] = hk.h;
        if (k >= SBLK - 5) o[(size_t)(TB_HB + k - (SBLK - 5)) * LB] = hk.h;
        if (k == SR - 1 || k == SBLK - 1) {
            const int cr = k == SR - 1 ? TB_CS : TB_CB, rr = k == SR - 1 ? TB_RS : TB_RB;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    o[(size_t)(cr + 3 * r + c) * LB] = v[c][r].h;
                    o[(size_t)(rr + 3 * r + c) * LB] = rm[3 * r + c].h;
                }
        }
    }
#pragma unroll
    for (int r = 0, i = 0; r < 3; ++r)
#pragma unroll
        for (int c = r; c < 3; ++c, ++i) o[(size_t)(TB_GB + 3 * r + c) * LB] = o[(size_t)(TB_GB + 3 * c + r) * LB] = g[i].h;
}

// The corner matrix W of N rows, and G = sum_{i < N} s_i s_i^T with s_i = C^i e_0.
__device__ __forceinline__ void corner(int N, double be1, double be2, double be3, double (&W)[9], double (&G)[9]) {
    const double C[9] = {-be1, -be2, -be3, 1.0, 0.0, 0.0, 0.0, 1.0, 0.0};
    const double X[9] = {1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    double t[9];
    power_sum<true>(N, C, X, G);
    // H (scaled by 1 / b0), rows past N zero
    const double H[9] = {be1, be2, be3, N > 1 ? be2 : 0.0, N > 1 ? be3 : 0.0, 0.0, N > 2 ? be3 : 0.0, 0.0, 0.0};
    double S[9], K[9];
    mat_mul(t, G, H);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            S[3 * r + c] = (r == c ? 1.0 : 0.0) + H[r] * t[c] + H[3 + r] * t[3 + c] + H[6 + r] * t[6 + c];
    // S = L L^T (symmetric, eigenvalues >= 1); K = L^-1 H^T, W = K^T K
    const double l00 = 1.0 / sqrt(S[0]), l10 = S[3] * l00, l20 = S[6] * l00;
    const double l11 = 1.0 / sqrt(S[4] - l10 * l10), l21 = (S[7] - l20 * l10) * l11;
    const double l22 = 1.0 / sqrt(S[8] - l20 * l20 - l21 * l21);
#pragma unroll
    for (int c = 0; c < 3; ++c) {      // column c of H^T is row c of H
        K[c] = H[3 * c] * l00;
        K[3 + c] = (H[3 * c + 1] - l10 * K[c]) * l11;
        K[6 + c] = (H[3 * c + 2] - l20 * K[c] - l21 * K[3 + c]) * l22;
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) W[3 * r + c] = K[r] * K[c] + K[3 + r] * K[3 + c] + K[6 + r] * K[6 + c];
}

// Per call of at most one block, one thread per branch: its tables.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_corner(const double *__restrict__ tab, int N, double *__restrict__ tc) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    const double be1 = tab[n], be2 = tab[LB + n], be3 = tab[2 * LB + n];
    double W[9], G[9], rm[9];
    corner(N, be1, be2, be3, W, G);
    head_response(N & (SR - 1), be1, be2, be3, rm);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        tc[(size_t)(TC_W + i) * LB + n] = W[i];
        tc[(size_t)(TC_RS + i) * LB + n] = rm[i];
    }
}

struct V3 {
    double a, b, c;
};
__device__ __forceinline__ V3 v3_load(const double *__restrict__ p, int n) {
    return V3{p[n], p[LB + n], p[2 * LB + n]};
}
__device__ __forceinline__ void v3_store(double *__restrict__ p, int n, V3 v) {
    p[n] = v.a;
    p[LB + n] = v.b;
    p[2 * LB + n] = v.c;
}
// x + M y, M's element i at m[i * ST]
template <int ST>
__device__ __forceinline__ V3 mv_add(V3 x, const double *m, V3 y) {
    return V3{fma(m[0], y.a, fma(m[ST], y.b, fma(m[2 * ST], y.c, x.a))),
              fma(m[3 * ST], y.a, fma(m[4 * ST], y.b, fma(m[5 * ST], y.c, x.b))),
              fma(m[6 * ST], y.a, fma(m[7 * ST], y.b, fma(m[8 * ST], y.c, x.c)))};
}

// The filter's next value from its last three.
#define PFB_FILTER(in, s) fma(-be1, (s).a, fma(-be2, (s).b, fma(-be3, (s).c, (in))))

// Outgoing states of block blockIdx.y from zero incoming ones: P = its last three
// v, Q = its first three zeta.  Q is a sum over the rows, sum_k v_k h_{k-r}, so
// the rows are read once, in order, and none is kept.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_span(const float *__restrict__ yh, int N, const double *__restrict__ tab, double *__restrict__ P,
           double *__restrict__ Q) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, blk = blockIdx.y, r0 = blk * SBLK, r1 = min(r0 + SBLK, N);
    const double be1 = tab[n], be2 = tab[LB + n], be3 = tab[2 * LB + n];
    V3 st{0.0, 0.0, 0.0}, q = st, h{0.0, 0.0, 0.0};
    double in = 1.0;                       // h's input: an impulse at the block's first row
    constexpr int CH = 32;
    for (int c0 = r0; c0 < r1; c0 += CH) {
        float y[CH];
#pragma unroll
        for (int k = 0; k < CH; ++k) y[k] = yh[(size_t)min(c0 + k, N - 1) * LB + n];
        const bool full = c0 + CH <= r1;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            if (full || c0 + k < r1) {
                const double v = PFB_FILTER((double)y[k], st), hk = PFB_FILTER(in, h);
                in = 0.0;
                q = V3{fma(v, hk, q.a), fma(v, h.a, q.b), fma(v, h.b, q.c)};
                st = V3{v, st.a, st.b};
                h = V3{hk, h.a, h.b};
            }
        }
    }
    v3_store(P + (size_t)3 * blk * LB, n, st);
    v3_store(Q + (size_t)3 * blk * LB, n, q);
}

// Per branch: the blocks' true incoming states A (from above) and B (from below),
// the corner's g, and the partial last span's head response.  The walks over the
// blocks are short dependent chains on few waves (512), so up to JOIN_LDS blocks
// the states wait in LDS, all loaded at the start (IN_LDS); longer calls keep
// them in A and Q, which is overwritten.
constexpr int JOIN_LDS = 16;
template <bool IN_LDS>
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_join(const double *__restrict__ tab, int N, int nb, const double *__restrict__ P, double *Q, double *A,
           double *__restrict__ B, double *__restrict__ tc) {
    __shared__ V3 sh[IN_LDS ? 2 * JOIN_LDS * SOLVE_WG : 1];
    const int t = threadIdx.x, n = blockIdx.x * SOLVE_WG + t;
    constexpr size_t B3 = (size_t)3 * LB;
    // slot 0: P, then A; slot 1: Q
    auto get = [&](int slot, int k) {
        return IN_LDS ? sh[(2 * k + slot) * SOLVE_WG + t] : v3_load((slot ? Q : A) + B3 * k, n);
    };
    auto put = [&](int slot, int k, V3 v) {
        if (IN_LDS)
            sh[(2 * k + slot) * SOLVE_WG + t] = v;
        else
            v3_store((slot ? Q : A) + B3 * k, n, v);
    };
    if (IN_LDS) {
        constexpr int U = 8;
        for (int k0 = 0; k0 < nb; k0 += U) {
            V3 p[U], q[U];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                p[i] = v3_load(P + B3 * min(k0 + i, nb - 1), n);
                q[i] = v3_load(Q + B3 * min(k0 + i, nb - 1), n);
            }
#pragma unroll
            for (int i = 0; i < U; ++i)
                if (k0 + i < nb) {
                    put(0, k0 + i, p[i]);
                    put(1, k0 + i, q[i]);
                }
        }
    }
    const double be1 = tab[n], be2 = tab[LB + n], be3 = tab[2 * LB + n];
    double cb[9], rb[9], rl[9], W[9], G[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        cb[i] = tab[(size_t)(TB_CB + i) * LB + n];
        rb[i] = tab[(size_t)(TB_RB + i) * LB + n];
    }
    head_response(N & (SR - 1), be1, be2, be3, rl);
#pragma unroll
    for (int i = 0; i < 9; ++i) tc[(size_t)(TC_RS + i) * LB + n] = rl[i];
    head_response((N - 1) % SBLK + 1, be1, be2, be3, rl);     // the last block's
    corner(N, be1, be2, be3, W, G);
    const V3 zero{0.0, 0.0, 0.0};
    V3 a = zero;
    for (int k = 0; k < nb; ++k) {
        const V3 p = IN_LDS ? get(0, k) : v3_load(P + B3 * k, n), q = get(1, k);
        put(0, k, a);
        put(1, k, k == nb - 1 ? mv_add<1>(q, rl, a) : mv_add<1>(q, rb, a));
        a = mv_add<1>(p, cb, a);
    }
    V3 z = zero;                                               // zeta at the head of block k
    for (int k = nb - 1; k >= 0; --k) z = mv_add<1>(get(1, k), cb, z);
    const double *h = tab + (size_t)TB_HB * LB + n;
    const double h0 = h[0], h1 = h[LB], h2 = h[2 * LB], h3 = h[3 * LB], h4 = h[4 * LB];
    // -dg on the first three rows: the states it leaves after the first block, and on
    auto correct = [&](V3 dg) {
        V3 d{-(dg.a * h4 + dg.b * h3 + dg.c * h2), -(dg.a * h3 + dg.b * h2 + dg.c * h1),
             -(dg.a * h2 + dg.b * h1 + dg.c * h0)};
        for (int k = 1; k < nb; ++k) {
            const V3 p = get(0, k), q = get(1, k);
            put(0, k, V3{p.a + d.a, p.b + d.b, p.c + d.c});
            put(1, k, k == nb - 1 ? mv_add<1>(q, rl, d) : mv_add<1>(q, rb, d));
            d = mv_add<1>(zero, cb, d);
        }
    };
    V3 g = mv_add<1>(zero, W, z);
    correct(g);
    // One step of refinement: W comes from a Gram matrix, whose condition is that
    // of the corner squared.  With the head zeta of the corrected solution, g must
    // be H H^T zeta; the residual r is corrected by (I + H H^T G)^-1 r = r - W G r.
    z = zero;
    for (int k = nb - 1; k > 0; --k) z = mv_add<1>(get(1, k), cb, z);
    {
        const double *gb = tab + (size_t)TB_GB * LB + n;
        V3 q = get(1, 0);
        q = V3{q.a - (gb[0] * g.a + gb[LB] * g.b + gb[2 * LB] * g.c),
               q.b - (gb[3 * LB] * g.a + gb[4 * LB] * g.b + gb[5 * LB] * g.c),
               q.c - (gb[6 * LB] * g.a + gb[7 * LB] * g.b + gb[8 * LB] * g.c)};
        z = mv_add<1>(q, cb, z);
        const double H[9] = {be1, be2, be3, be2, be3, 0.0, be3, 0.0, 0.0};          // symmetric
        const V3 r = mv_add<1>(V3{-g.a, -g.b, -g.c}, H, mv_add<1>(zero, H, z));
        const V3 wgr = mv_add<1>(zero, W, mv_add<1>(zero, G, r));
        const V3 dg{r.a - wgr.a, r.b - wgr.b, r.c - wgr.c};
        correct(dg);
        g = V3{g.a + dg.a, g.b + dg.b, g.c + dg.c};
    }
    v3_store(tc + (size_t)TC_G * LB, n, g);
    if (IN_LDS)
        for (int k = 0; k < nb; ++k) v3_store(A + B3 * k, n, get(0, k));
    V3 b = zero;
    for (int k = nb - 1; k >= 0; --k) {
        v3_store(B + B3 * k, n, b);
        b = mv_add<1>(get(1, k), cb, b);
    }
}

// One block of 256 rows x 64 branches (a row of a wave: 256 contiguous bytes).
// ONE: the block is the whole problem, and the corner is solved here; else its
// incoming states and g come from k_pfb_join.  Rows past N read as zero and are
// not written (range-checked buffers).
template <bool ONE>
__global__ void __launch_bounds__(64 * SWV, 4)
k_pfb_solve(const float *__restrict__ yh, int N, const double *__restrict__ tab, const double *__restrict__ tc,
            const double *__restrict__ A, const double *__restrict__ B, float *__restrict__ x) {
    // rows of the workgroup's table in LDS
    constexpr int L_CS = 0, L_RS = 9, L_HS = 18, L_TC = 23, L_N = L_TC + TC_N;
    static_assert(TB_HS == TB_RS + 9, "a span's responses are contiguous");
    __shared__ double T[L_N * 64];
    __shared__ V3 tot[SWV][64], sg[64], sd[64];
    const int t = threadIdx.x, br = t & 63, wave = t >> 6, n0 = (int)blockIdx.x * 64, n = n0 + br;
    const int blk = ONE ? 0 : (int)blockIdx.y, r0 = SBLK * blk + SR * wave;
    const int nv = N - r0;                       // this span's rows: nv, at most 32 (none if <= 0)
    const __amdgpu_buffer_rsrc_t ry =
        __builtin_amdgcn_make_buffer_rsrc((void *)(yh + (size_t)SBLK * blk * LB), 0,
                                          min(N - SBLK * blk, SBLK) * LB * (int)sizeof(float), 0x00020000);
    double v[SR];
    const double be1 = tab[n], be2 = tab[LB + n], be3 = tab[2 * LB + n];
    V3 gin{0.0, 0.0, 0.0}, c0{0.0, 0.0, 0.0}, b0 = c0;
    if (!ONE) {
        if (blk == 0 && wave == 0) gin = v3_load(tc + (size_t)TC_G * LB, n);
        c0 = v3_load(A + (size_t)3 * blk * LB, n);
        b0 = v3_load(B + (size_t)3 * blk * LB, n);
    }
    {
        float y[SR];
        const int vo = 4 * (SR * wave * LB + n);
#pragma unroll
        for (int k = 0; k < SR; ++k) y[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ry, vo + 4 * LB * k, 0, 0));
        for (int e = t; e < L_N * 64; e += 64 * SWV) {
            const int r = e >> 6, c = n0 + (e & 63);
            T[e] = r < L_RS   ? tab[(size_t)(TB_CS + r) * LB + c]
                   : r < L_TC ? tab[(size_t)(TB_RS + r - L_RS) * LB + c]
                              : tc[(size_t)(r - L_TC) * LB + c];
        }
#pragma unroll
        for (int k = 0; k < SR; ++k) v[k] = (double)y[k];
    }
    if (!ONE) {
        v[0] -= gin.a;
        v[1] -= gin.b;
        v[2] -= gin.c;
    }
    const V3 zero{0.0, 0.0, 0.0};
    const double *cs = T + L_CS * 64 + br;
    // the span from zero states, both ways
    V3 p = zero, q = zero;
#pragma unroll
    for (int k = 0; k < SR; ++k) {
        v[k] = PFB_FILTER(v[k], p);
        p = V3{v[k], p.a, p.b};
    }
    const bool part = nv < SR;                   // the span ends early
    if (part) {
#pragma unroll
        for (int k = 0; k < SR; ++k)
            if (k >= nv) v[k] = 0.0;
    }
#pragma unroll
    for (int k = SR - 1; k >= 0; --k) q = V3{PFB_FILTER(v[k], q), q.a, q.b};
    // incoming state: a_j = C^(32 j) c0 + sum_{i < j} C^(32 (j - 1 - i)) p_i
    tot[wave][br] = p;
    __syncthreads();
    V3 a = c0;
    for (int i = 0; i < wave; ++i) a = mv_add<64>(tot[i][br], cs, a);
    __syncthreads();
    // from below: C^(32 (7 - j)) b0 + sum_{i > j} C^(32 (i - 1 - j)) q_i
    auto suffix = [&](V3 in) {
        tot[wave][br] = in;
        __syncthreads();
        V3 c = b0;
        for (int i = SWV - 1; i > wave; --i) c = mv_add<64>(tot[i][br], cs, c);
        return c;
    };
    // head response of this span (the partial last one has its own; none past it)
    const double *rm = T + (part ? L_TC + TC_RS : L_RS) * 64 + br;
    if (nv > 0) q = mv_add<64>(q, rm, a);
    V3 b = suffix(q);
    if (ONE) {
        if (wave == 0) {
            const double *h = T + L_HS * 64 + br;
            const V3 zh = mv_add<64>(q, cs, b);               // zeta[0..2] without the corner
            const V3 g = mv_add<64>(zero, T + (L_TC + TC_W) * 64 + br, zh);
            sg[br] = g;
            // state after the first span from -g on its first three rows
            sd[br] = V3{-(g.a * h[4 * 64] + g.b * h[3 * 64] + g.c * h[2 * 64]),
                        -(g.a * h[3 * 64] + g.b * h[2 * 64] + g.c * h[64]),
                        -(g.a * h[2 * 64] + g.b * h[64] + g.c * h[0])};
        }
        __syncthreads();
        if (wave > 0) {        // C^(32 (j - 1)) of it
            V3 d = sd[br];
            for (int i = 1; i < wave; ++i) d = mv_add<64>(zero, cs, d);
            a = V3{a.a + d.a, a.b + d.b, a.c + d.c};
            if (nv > 0) q = mv_add<64>(q, rm, d);
        } else {
            gin = sg[br];
        }
        b = suffix(q);
    }
    if (nv <= 0) return;
    // the rows from their true states
    {
        V3 d = a;
#pragma unroll
        for (int k = 0; k < SR; ++k) {
            const double dk = PFB_FILTER(!ONE ? 0.0 : k == 0 ? -gin.a : k == 1 ? -gin.b : k == 2 ? -gin.c : 0.0, d);
            v[k] += dk;
            d = V3{dk, d.a, d.b};
        }
    }
    if (part) {
#pragma unroll
        for (int k = 0; k < SR; ++k)
            if (k >= nv) v[k] = 0.0;
    }
    const double w0 = tab[(size_t)TB_WZ * LB + n], w1 = tab[(size_t)(TB_WZ + 1) * LB + n],
                 w2 = tab[(size_t)(TB_WZ + 2) * LB + n], w3 = tab[(size_t)(TB_WZ + 3) * LB + n];
    // x[i + 3] = w0 z[i+3] + w1 z[i+2] + w2 z[i+1] + w3 z[i]; the first span also x[0..2].
    // The buffer starts at the block's row i + 3 = SBLK blk + 3.
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void *)(x + (size_t)(SBLK * blk + 3) * LB), 0,
                                          min(N - SBLK * blk, SBLK) * LB * (int)sizeof(float), 0x00020000);
    const int vs = lds_opaque(4 * (SR * wave * LB + n));   // not the loads' offsets kept live until here
#pragma unroll
    for (int k = SR - 1; k >= 0; --k) {
        const double z = PFB_FILTER(v[k], b);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((float)(w0 * b.c + w1 * b.b + w2 * b.a + w3 * z)), rx,
                                              vs + 4 * LB * k, 0, 0);
        b = V3{z, b.a, b.b};
    }
    if (r0 == 0) {
        x[(size_t)2 * LB + n] = (float)(w0 * b.c + w1 * b.b + w2 * b.a);
        x[(size_t)LB + n] = (float)(w0 * b.b + w1 * b.a);
        x[n] = (float)(w0 * b.a);
    }
}
#undef PFB_FILTER

}  // namespace

struct sdbe_pfb {
    int device = 0;
    int max_spec = 0;
    int last_hip_err = 0;
    float2 *fft_img = nullptr;    // FftTw image
    double2 *tw1k = nullptr;      // e^{2 pi i k / 32768}, k < 1024
    float *win = nullptr;         // [4][32768]
    double *a = nullptr;          // [4][32768] band of P P^T per branch
    float *yh = nullptr;          // [max_spec][32768]
    double *uck = nullptr;        // [chunks][3][32768] forward state entering every 16-row chunk
    double *ckpt = nullptr;       // [chunks][6][32768] factor state at every 16th row
    double *pst = nullptr;        // [spans][3][32768] particular outgoing states
    double *mf = nullptr;         // [spans][9][32768] forward transfers of full spans
    double *mb = nullptr;         // [spans][9][32768] backward transfers of full spans
    double *state = nullptr;      // [spans][3][32768] incoming state of every span
    double *tab = nullptr;        // [TB_N][32768] constant-coefficient solve: tables
    double *tc = nullptr;         // [TC_N][32768] ... of the current call
    double *bst = nullptr;        // [4][nb][3][32768] ... its blocks' states, out and in, both ways
    int nb = 0;                   // blocks of max_spec rows
    int n_cu = 256;               // compute units of the device
    int constant = 0;             // no branch has zeros together on the unit circle
};

namespace {
int pfb_fail(sdbe_pfb_t *p, hipError_t e) {
    if (p) p->last_hip_err = (int)e;
    return SDBE_ERR_HIP;
}
#define PFB_TRY(p, expr)                               \
    do {                                               \
        hipError_t _e = (expr);                        \
        if (_e != hipSuccess) return pfb_fail((p), _e); \
    } while (0)
}  // namespace

extern "C" {

void sdbe_pfb_destroy(sdbe_pfb_t *p) {
    if (!p) return;
    (void)hipSetDevice(p->device);
    (void)hipDeviceSynchronize();
    (void)hipFree(p->fft_img);
    (void)hipFree(p->tw1k);
    (void)hipFree(p->win);
    (void)hipFree(p->a);
    (void)hipFree(p->yh);
    (void)hipFree(p->tab);
    (void)hipFree(p->tc);
    (void)hipFree(p->bst);
    (void)hipFree(p->uck);
    (void)hipFree(p->ckpt);
    (void)hipFree(p->pst);
    (void)hipFree(p->mf);
    (void)hipFree(p->mb);
    (void)hipFree(p->state);
    delete p;
}

int sdbe_pfb_last_hip_error(const sdbe_pfb_t *p) { return p ? p->last_hip_err : 0; }

int sdbe_pfb_create(int device, int32_t n_taps, const float *h_window, int32_t max_spectra, sdbe_pfb_t **out) {
    if (!out) return SDBE_ERR_ARG;
    *out = nullptr;
    if (n_taps != NT || !h_window || max_spectra < 1 || max_spectra > (1 << 16)) return SDBE_ERR_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return SDBE_ERR_NODEV;
    if (hipSetDevice(device) != hipSuccess) return SDBE_ERR_NODEV;
    sdbe_pfb_t *p = new (std::nothrow) sdbe_pfb();
    if (!p) return SDBE_ERR_NOMEM;
    p->device = device;
    p->max_spec = max_spectra;
    int rc = SDBE_OK, clustered = 0, *d_clustered = nullptr, ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && ncu > 0) p->n_cu = ncu;
    std::vector<float2> img(FFT_TW_N);
    std::vector<double2> tw(1024);
    const double two_pi = 6.283185307179586476925286766559;
    fft_tw_fill(img.data());
    for (int k = 0; k < 1024; ++k) {
        const double ang = two_pi * (double)k / (double)LB;
        tw[k] = make_double2(cos(ang), sin(ang));
    }
#define PALLOC(ptr, bytes)                                              \
    do {                                                                \
        if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess) {        \
            rc = SDBE_ERR_NOMEM;                                        \
            goto fail;                                                  \
        }                                                               \
    } while (0)
    PALLOC(p->fft_img, FFT_TW_N * sizeof(float2));
    PALLOC(p->tw1k, 1024 * sizeof(double2));
    PALLOC(p->win, (size_t)NT * LB * sizeof(float));
    PALLOC(p->yh, (size_t)max_spectra * LB * sizeof(float));
    PALLOC(p->tab, (size_t)TB_N * LB * sizeof(double));
    PALLOC(p->tc, (size_t)TC_N * LB * sizeof(double));
    d_clustered = reinterpret_cast<int *>(p->tc);    // until the first call writes its tables
    if (hipMemcpy(p->fft_img, img.data(), FFT_TW_N * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->tw1k, tw.data(), 1024 * sizeof(double2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->win, h_window, (size_t)NT * LB * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d_clustered, &clustered, sizeof(int), hipMemcpyHostToDevice) != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    hipLaunchKernelGGL(k_pfb_spectral, dim3(LB / SOLVE_WG), dim3(SOLVE_WG), 0, 0, (const float *)p->win, p->tab,
                       d_clustered);
    if (hipMemcpy(&clustered, d_clustered, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    p->constant = clustered == 0;
    if (p->constant) {
        p->nb = (max_spectra + SBLK - 1) / SBLK;
        PALLOC(p->bst, (size_t)4 * 3 * p->nb * LB * sizeof(double));
    } else {                                         // the factor-row kernels
        // one transfer per span; checkpoints up to the chunk after the last full span
        const size_t nspan = (size_t)(max_spectra + SPAN - 1) / SPAN;
        const size_t nck = nspan * (SPAN / SEG) + 1;
        std::vector<double> band((size_t)NT * LB);
        for (int n = 0; n < LB; ++n)
            for (int d = 0; d < NT; ++d) {
                double acc = 0.0;
                for (int k = 0; k + d < NT; ++k)
                    acc += (double)h_window[(size_t)(k + d) * LB + n] * (double)h_window[(size_t)k * LB + n];
                band[(size_t)d * LB + n] = acc;
            }
        PALLOC(p->a, (size_t)NT * LB * sizeof(double));
        PALLOC(p->uck, nck * 3 * LB * sizeof(double));
        PALLOC(p->ckpt, nck * CKW * LB * sizeof(double));
        PALLOC(p->pst, nspan * 3 * LB * sizeof(double));
        PALLOC(p->mf, nspan * 9 * LB * sizeof(double));
        PALLOC(p->mb, nspan * 9 * LB * sizeof(double));
        PALLOC(p->state, nspan * 3 * LB * sizeof(double));
        if (hipMemcpy(p->a, band.data(), (size_t)NT * LB * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
            rc = SDBE_ERR_HIP;
            goto fail;
        }
        // the factor's checkpoints and the full spans' transfers depend on the window only
        hipLaunchKernelGGL(k_pfb_factor, dim3(LB / SOLVE_WG), dim3(SOLVE_WG), 0, 0, (int)nck, (const double *)p->a,
                           p->ckpt);
        hipLaunchKernelGGL(k_pfb_fspan<true>, dim3(LB / SOLVE_WG, nspan), dim3(SOLVE_WG), 0, 0, (const float *)nullptr,
                           (int)(nspan * SPAN), (const double *)p->a, (const double *)p->ckpt, p->mf);
        hipLaunchKernelGGL(k_pfb_bspan<true>, dim3(LB / SOLVE_WG, nspan), dim3(SOLVE_WG), 0, 0, (const float *)nullptr,
                           (const double *)nullptr, (int)(nspan * SPAN), (const double *)p->a, (const double *)p->ckpt,
                           p->mb);
    }
#undef PALLOC
    if (hipDeviceSynchronize() != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    *out = p;
    return SDBE_OK;
fail:
    sdbe_pfb_destroy(p);
    return rc;
}

int sdbe_pfb_forward(sdbe_pfb_t *p, const float *d_x, int32_t n_spectra, void *d_spec, void *stream) {
    if (!p || !d_x || !d_spec || n_spectra < 1) return SDBE_ERR_ARG;
    if (n_spectra > p->max_spec) return SDBE_ERR_CAPACITY;
    PFB_TRY(p, hipSetDevice(p->device));
    hipStream_t s = (hipStream_t)stream;
    if (n_spectra <= p->n_cu) {          // pairs would leave CUs without work: one round either way, of one or of two spectra
        hipLaunchKernelGGL(k_pfb_fold_r2c, dim3(n_spectra), dim3(1024), 0, s, d_x, (const float *)p->win,
                           (float2 *)d_spec, (const float2 *)p->fft_img, (const double2 *)p->tw1k);
    } else {
        const int pairs = (n_spectra + 1) / 2;
        hipLaunchKernelGGL(k_pfb_fold2_r2c, dim3(pairs < p->n_cu ? pairs : p->n_cu), dim3(1024), 0, s, d_x,
                           (int)n_spectra, (const float *)p->win, (float2 *)d_spec, (const float2 *)p->fft_img,
                           (const double2 *)p->tw1k);
    }
    PFB_TRY(p, hipGetLastError());
    return SDBE_OK;
}

int sdbe_pfb_inverse(sdbe_pfb_t *p, const void *d_spec, int32_t n_spectra, float *d_x, void *stream) {
    if (!p || !d_spec || !d_x || n_spectra < 1) return SDBE_ERR_ARG;
    if (n_spectra > p->max_spec) return SDBE_ERR_CAPACITY;
    PFB_TRY(p, hipSetDevice(p->device));
    hipStream_t s = (hipStream_t)stream;
    const bool loop = n_spectra > p->n_cu;
    hipLaunchKernelGGL(loop ? k_pfb_c2r<true> : k_pfb_c2r<false>, dim3(loop ? p->n_cu : n_spectra), dim3(1024), 0, s,
                       (const float2 *)d_spec, (int)n_spectra, p->yh, (const float2 *)p->fft_img, (const double2 *)p->tw1k);
    if (p->constant) {
        const int N = n_spectra, nb = (N + SBLK - 1) / SBLK;
        const dim3 br(LB / SOLVE_WG), wg(SOLVE_WG);
        const double *tab = p->tab;
        const float *yh = p->yh;
        if (nb == 1) {
            hipLaunchKernelGGL(k_pfb_corner, br, wg, 0, s, tab, N, p->tc);
            hipLaunchKernelGGL(k_pfb_solve<true>, dim3(LB / 64), dim3(64 * SWV), 0, s, yh, N, tab, (const double *)p->tc,
                               (const double *)nullptr, (const double *)nullptr, d_x);
        } else {
            double *P = p->bst, *Q = P + (size_t)3 * p->nb * LB, *A = Q + (size_t)3 * p->nb * LB,
                   *B = A + (size_t)3 * p->nb * LB;
            hipLaunchKernelGGL(k_pfb_span, dim3(LB / SOLVE_WG, nb), wg, 0, s, yh, N, tab, P, Q);
            if (nb <= JOIN_LDS)
                hipLaunchKernelGGL(k_pfb_join<true>, br, wg, 0, s, tab, N, nb, (const double *)P, Q, A, B, p->tc);
            else
                hipLaunchKernelGGL(k_pfb_join<false>, br, wg, 0, s, tab, N, nb, (const double *)P, Q, A, B, p->tc);
            hipLaunchKernelGGL(k_pfb_solve<false>, dim3(LB / 64, nb), dim3(64 * SWV), 0, s, yh, N, tab,
                               (const double *)p->tc, (const double *)A, (const double *)B, d_x);
        }
        PFB_TRY(p, hipGetLastError());
        return SDBE_OK;
    }
    const int nspan = (n_spectra + SPAN - 1) / SPAN;
    const dim3 grid(LB / SOLVE_WG, nspan);
    const double *ck = p->ckpt, *a = p->a;
    hipLaunchKernelGGL(k_pfb_fspan<false>, grid, dim3(SOLVE_WG), 0, s, (const float *)p->yh, (int)n_spectra, a, ck,
                       p->pst);
    hipLaunchKernelGGL(k_pfb_scan, dim3(LB / SOLVE_WG), dim3(SOLVE_WG), 0, s, (const double *)p->pst, (const double *)p->mf, nspan, 1,
                       p->state);
    hipLaunchKernelGGL(k_pfb_ffin, grid, dim3(SOLVE_WG), 0, s, (const float *)p->yh, (int)n_spectra, a, ck,
                       (const double *)p->state, p->uck);
    hipLaunchKernelGGL(k_pfb_bspan<false>, grid, dim3(SOLVE_WG), 0, s, (const float *)p->yh,
                       (const double *)p->uck, (int)n_spectra, a, ck, p->pst);
    hipLaunchKernelGGL(k_pfb_scan, dim3(LB / SOLVE_WG), dim3(SOLVE_WG), 0, s, (const double *)p->pst, (const double *)p->mb, nspan, -1,
                       p->state);
    hipLaunchKernelGGL(k_pfb_bfin, grid, dim3(SOLVE_WG), 0, s, (const float *)p->yh, (const double *)p->uck,
                       (int)n_spectra, a, ck, (const double *)p->state, (const float *)p->win, d_x);
    PFB_TRY(p, hipGetLastError());
    return SDBE_OK;
}

}  // extern "C"
