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
// The solve, for prototypes that a constant factor loses nothing in
// (sdbe_pfb_solve.hpp: the rule and what it was measured over):
//   k_pfb_spectral  once per plan, one thread per branch: the constant
//                   minimum-phase factor of P P^T and the tables built on it
//   k_pfb_span, k_pfb_join, k_pfb_solve
//                   two recursive filters, block-parallel over the rows
//   k_pfb_corner    calls of up to 256 rows: their corner, then k_pfb_solve alone
// and for the others, if one branch is of that kind, the factor-row kernels:
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
#include "sdbe_pfb_solve.hpp"
#include "../../include/sdbe_pfb.h"
#include "../../include/sdbe_stage.h"

using namespace sdbe;
using namespace sdbe::pfb;

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
// The factor, its tables, the corner and the rule that admits a plan are in
// sdbe_pfb_solve.hpp; here they run block-parallel over the rows.
//
// Thread (branch, span of 32 rows) keeps its rows' v in registers; a workgroup
// holds 64 branches x 8 spans and scans the spans' boundary states through LDS, and
// each span's head zeta is taken from its true v (from the v of a zero incoming
// state it would lose the 32 rows' growth of both filters).
// Up to 256 rows that is the whole problem.  Above, k_pfb_span takes every
// 256-row block's outgoing states in both directions (from zero incoming ones) in
// one read of yh, k_pfb_join composes them per branch into the blocks' true
// incoming states with the corner, and k_pfb_solve finishes the blocks: two
// reads of yh and one write of x, all in 256-byte runs.  4096 spectra: span 128 us
// (4.2 TB/s), join 29, solve 247 (4.3 TB/s); the factor-row kernels, which read yh
// four times beside 0.8 GB of checkpoints and recompute every factor row four
// times, take 890.  A call of 256 rows: corner 13, solve 28.  (Tiles of 8 branches over
// all 4096 rows read yh once, but in 32-byte runs: 700 us.)

// Table rows of a call.
constexpr int TC_S = 0;                   // the corner's Cholesky factor
constexpr int TC_T = 6;                   // more than one block: t
constexpr int TC_N = 9;

// Per plan, one thread per branch.  *refused counts the branches that the
// constant-coefficient solve would lose more in than it may.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_spectral(const float *__restrict__ win, int blocks, double *__restrict__ tab, int *__restrict__ refused) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    const float w[4] = {win[n], win[LB + n], win[2 * LB + n], win[3 * LB + n]};
    if (!admitted(plan_tables(w, blocks, tab + n, LB))) atomicAdd(refused, 1);
}

__device__ __forceinline__ Beta beta_load(const double *__restrict__ tab, int n) {
    return Beta{tab[n], tab[LB + n], tab[2 * LB + n]};
}
__device__ __forceinline__ void corner_store(double *__restrict__ tc, int n, const Corner &c) {
    const double s[6] = {c.i0, c.l10, c.l20, c.i1, c.l21, c.i2};
#pragma unroll
    for (int i = 0; i < 6; ++i) tc[(size_t)(TC_S + i) * LB + n] = s[i];
}
__device__ __forceinline__ Corner corner_load(const double *__restrict__ tc, int n) {
    double s[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = tc[(size_t)(TC_S + i) * LB + n];
    return Corner{s[0], s[1], s[2], s[3], s[4], s[5]};
}

// Per call of at most one block, one thread per branch: its corner.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_corner(const double *__restrict__ tab, int N, double *__restrict__ tc) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x;
    const Beta be = beta_load(tab, n);
    double R[9], G[9];
    row_responses(N, be, R, G);
    corner_store(tc, n, corner(be, G));
}

__device__ __forceinline__ V3 v3_load(const double *__restrict__ p, int n) {
    return V3{p[n], p[LB + n], p[2 * LB + n]};
}
__device__ __forceinline__ void v3_store(double *__restrict__ p, int n, V3 v) {
    p[n] = v.a;
    p[LB + n] = v.b;
    p[2 * LB + n] = v.c;
}

// Outgoing states of block blockIdx.y from zero incoming ones: P = its last three
// v, Q = its first three zeta.  Q is a sum over the rows, sum_k v_k h_{k-r}, so
// the rows are read once, in order, and none is kept.
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_span(const float *__restrict__ yh, int N, const double *__restrict__ tab, double *__restrict__ P,
           double *__restrict__ Q) {
    const int n = blockIdx.x * SOLVE_WG + threadIdx.x, blk = blockIdx.y, r0 = blk * SBLK, r1 = min(r0 + SBLK, N);
    const Beta be = beta_load(tab, n);
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
                const double v = filter(be, (double)y[k], st), hk = filter(be, in, h);
                in = 0.0;
                q = V3{fma(v, hk, q.a), fma(v, h.a, q.b), fma(v, h.b, q.c)};
                st = shift(v, st);
                h = shift(hk, h);
            }
        }
    }
    v3_store(P + (size_t)3 * blk * LB, n, st);
    v3_store(Q + (size_t)3 * blk * LB, n, q);
}

// Per branch: the blocks' true incoming states A (from above) and B (from below),
// and the corner with its t.  Each step of t composes the blocks anew from the
// states of k_pfb_span, so that what t takes off the first block is taken off
// before it is carried on.  The walks over the blocks are short dependent chains on few
// waves (512), so up to JOIN_LDS blocks the states wait in LDS, all loaded at the
// start (IN_LDS: P, Q and the heads, 72 KB); longer calls read them again and keep
// the heads in B.  4096 spectra 29 us, 4097 57 (of 690 for the call).
constexpr int JOIN_LDS = 16;
template <bool IN_LDS>
__global__ void __launch_bounds__(SOLVE_WG)
k_pfb_join(const double *__restrict__ tab, int N, int nb, const double *__restrict__ P, const double *__restrict__ Q,
           double *__restrict__ A, double *B, double *__restrict__ tc) {
    __shared__ V3 sh[IN_LDS ? 3 * JOIN_LDS * SOLVE_WG : 1];
    const int t = threadIdx.x, n = blockIdx.x * SOLVE_WG + t;
    constexpr size_t B3 = (size_t)3 * LB;
    auto slot = [&](int i, int k) -> V3 & { return sh[(3 * k + i) * SOLVE_WG + t]; };
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
                    slot(0, k0 + i) = p[i];
                    slot(1, k0 + i) = q[i];
                }
        }
    }
    const Beta be = beta_load(tab, n);
    double cb[9], rb[9], gb[9], rl[9], G[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        cb[i] = tab[(size_t)(TB_CB + i) * LB + n];
        rb[i] = tab[(size_t)(TB_RB + i) * LB + n];
        gb[i] = tab[(size_t)(TB_GB + i) * LB + n];
        rl[i] = rb[i];
    }
    {
        const int rows = (N - 1) % SBLK + 1;               // the last block's
        double pw[9];
        block_gram(rows == SBLK ? nb : nb - 1, cb, gb, pw, G);
        if (rows != SBLK) {                                 // workgroup-uniform
            double gl[9], s[9], u[9];
            row_responses(rows, be, rl, gl);
            mat_mul(s, pw, gl);
            mat_mul_t(u, s, pw);
#pragma unroll
            for (int i = 0; i < 9; ++i) G[i] += u[i];
        }
    }
    const Corner cn = corner(be, G);
    corner_store(tc, n, cn);
    const double *hp = tab + (size_t)TB_HB * LB + n;
    const double h0 = hp[0], h1 = hp[LB], h2 = hp[2 * LB], h3 = hp[3 * LB], h4 = hp[4 * LB];
    const V3 zero{0.0, 0.0, 0.0};
    V3 tt = zero;
#pragma unroll 1
    for (int it = 0; it <= CORNER_STEPS; ++it) {
        const bool last = it == CORNER_STEPS;
        const V3 g = hankel(be, tt);
        V3 a = zero;
        for (int k = 0; k < nb; ++k) {
            V3 p = IN_LDS ? slot(0, k) : v3_load(P + B3 * k, n), q = IN_LDS ? slot(1, k) : v3_load(Q + B3 * k, n);
            if (k == 0) {      // the block's response to -g on its first three rows
                p = v3_sub(p, V3{fma(g.a, h4, fma(g.b, h3, g.c * h2)), fma(g.a, h3, fma(g.b, h2, g.c * h1)),
                                 fma(g.a, h2, fma(g.b, h1, g.c * h0))});
                q = mv_add<1>(q, gb, V3{-g.a, -g.b, -g.c});
            }
            q = mv_add<1>(q, k == nb - 1 ? rl : rb, a);
            if (IN_LDS)
                slot(2, k) = q;
            else
                v3_store(B + B3 * k, n, q);
            if (last) v3_store(A + B3 * k, n, a);
            a = mv_add<1>(p, cb, a);
        }
        V3 z = zero;                                        // zeta at the head of block k
        for (int k = nb - 1; k >= 0; --k) {
            const V3 q = IN_LDS ? slot(2, k) : v3_load(B + B3 * k, n);
            if (last) v3_store(B + B3 * k, n, z);
            z = mv_add<1>(q, cb, z);
        }
        if (!last) tt = v3_add(tt, corner_step(cn, be, z, tt));
    }
    v3_store(tc + (size_t)TC_T * LB, n, tt);
}

// One block of 256 rows x 64 branches (a row of a wave: 256 contiguous bytes).
// ONE: the block is the whole problem, and the corner is sought here; else its
// incoming states and t come from k_pfb_join.  Rows past N read as zero and are
// not written (range-checked buffers).
template <bool ONE>
__global__ void __launch_bounds__(64 * SWV, 4)
k_pfb_solve(const float *__restrict__ yh, int N, const double *__restrict__ tab, const double *__restrict__ tc,
            const double *__restrict__ A, const double *__restrict__ B, float *__restrict__ x) {
    __shared__ double cs[9 * 64];                // C^32
    __shared__ V3 tot[SWV][64], sd[64];
    // wave in a scalar register: v changes under branches on it, which must not be divergent
    const int t = threadIdx.x, br = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int n0 = (int)blockIdx.x * 64, n = n0 + br, blk = ONE ? 0 : (int)blockIdx.y, r0 = SBLK * blk + SR * wave;
    const int nv = N - r0;                       // this span's rows: nv, at most 32 (none if <= 0)
    const __amdgpu_buffer_rsrc_t ry =
        __builtin_amdgcn_make_buffer_rsrc((void *)(yh + (size_t)SBLK * blk * LB), 0,
                                          min(N - SBLK * blk, SBLK) * LB * (int)sizeof(float), 0x00020000);
    double v[SR];
    const Beta be = beta_load(tab, n);
    const V3 zero{0.0, 0.0, 0.0};
    V3 c0 = zero, tt = zero;
    if (!ONE) {
        if (blk == 0 && wave == 0) tt = v3_load(tc + (size_t)TC_T * LB, n);
        c0 = v3_load(A + (size_t)3 * blk * LB, n);
    }
    {
        float y[SR];
        const int vo = 4 * (SR * wave * LB + n);
#pragma unroll
        for (int k = 0; k < SR; ++k) y[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ry, vo + 4 * LB * k, 0, 0));
        for (int e = t; e < 9 * 64; e += 64 * SWV) cs[e] = tab[(size_t)(TB_CS + (e >> 6)) * LB + n0 + (e & 63)];
#pragma unroll
        for (int k = 0; k < SR; ++k) v[k] = (double)y[k];
    }
    if (!ONE) {                                  // tt is zero but in the block's first rows
        const V3 g = hankel(be, tt);
        v[0] -= g.a;
        v[1] -= g.b;
        v[2] -= g.c;
    }
    // x + C^32 y; the matrix is read where it is used (its 18 registers are v's)
    auto carry = [&](V3 x, V3 y) { return mv_add<64>(x, cs + lds_opaque(br), y); };
    // Spans past the last row stay out of the arithmetic and off the scans (their
    // states are zero): a call of few rows is one wave per workgroup.
    const bool mine = nv > 0;
    const int spans = min((N - SBLK * blk + SR - 1) / SR, SWV);
    V3 d = c0, b = zero;                         // b: the state from below
    if (mine) {                                  // the span from a zero state
        V3 p = zero;
#pragma unroll
        for (int k = 0; k < SR; ++k) {
            v[k] = filter(be, v[k], p);
            p = shift(v[k], p);
        }
        tot[wave][br] = p;
    }
    __syncthreads();
    // incoming state: C^(32 j) c0 + sum_{i < j} C^(32 (j - 1 - i)) p_i
    if (mine)
        for (int i = 0; i < wave; ++i) d = carry(tot[i][br], d);
    __syncthreads();
    V3 g = zero;
    const int steps = ONE ? CORNER_STEPS : blk == 0 ? CORNER_STEPS_BLOCK : 0;
#pragma unroll 1
    for (int it = 0;; ++it) {
        int m = n;                               // each step's own: the addresses below are not kept through the loop
        asm("" : "+v"(m) : "s"(it));
        V3 q = zero;                             // the span's head zeta with nothing incoming from below
        if (mine) {
            // v changes by the filter's response to -g on the span's first three
            // rows and to the incoming state d
#pragma unroll
            for (int k = 0; k < SR; ++k) {
                const double dk = filter(be, k == 0 ? -g.a : k == 1 ? -g.b : k == 2 ? -g.c : 0.0, d);
                v[k] += dk;
                d = shift(dk, d);
            }
            if (nv < SR) {                       // the span ends early
#pragma unroll
                for (int k = 0; k < SR; ++k)
                    if (k >= nv) v[k] = 0.0;
            }
#pragma unroll
            for (int k = SR - 1; k >= 0; --k) q = shift(filter(be, v[k], q), q);
            tot[wave][br] = q;
        }
        __syncthreads();
        if (mine) {                              // C^(32 (7 - j)) times the block's + sum_{i > j} C^(32 (i - 1 - j)) q_i
            b = ONE ? zero : v3_load(B + (size_t)3 * blk * LB, m);
            for (int i = spans - 1; i > wave; --i) b = carry(tot[i][br], b);
        }
        if (it == steps) break;
        d = zero;
        if (wave == 0) {
            const V3 dt = corner_step(corner_load(tc, m), be, carry(q, b), tt);
            tt = v3_add(tt, dt);
            g = hankel(be, dt);
            if (spans > 1) {
                V3 e = V3{-g.a, 0.0, 0.0};
                e = shift(filter(be, -g.b, e), e);
                e = shift(filter(be, -g.c, e), e);
#pragma unroll 4
                for (int k = 3; k < SR; ++k) e = shift(filter(be, 0.0, e), e);
                sd[br] = e;
            }
        }
        __syncthreads();
        if (mine && wave > 0) {                  // C^(32 (j - 1)) of the first span's
            d = sd[br];
            for (int i = 1; i < wave; ++i) d = carry(zero, d);
        }
    }
    if (!mine) return;
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
        const double z = filter(be, v[k], b);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((float)(w0 * b.c + w1 * b.b + w2 * b.a + w3 * z)), rx,
                                              vs + 4 * LB * k, 0, 0);
        b = shift(z, b);
    }
    if (r0 == 0) {
        x[(size_t)2 * LB + n] = (float)(w0 * b.c + w1 * b.b + w2 * b.a);
        x[(size_t)LB + n] = (float)(w0 * b.b + w1 * b.a);
        x[n] = (float)(w0 * b.a);
    }
}

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
    int constant = 0;             // every branch is admitted to the constant-coefficient solve
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
    int rc = SDBE_OK, refused = 0, *d_refused = nullptr, ncu = 0;
    const int nb = (max_spectra + SBLK - 1) / SBLK;
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
    d_refused = reinterpret_cast<int *>(p->tc);    // until the first call writes its tables
    if (hipMemcpy(p->fft_img, img.data(), FFT_TW_N * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->tw1k, tw.data(), 1024 * sizeof(double2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->win, h_window, (size_t)NT * LB * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d_refused, &refused, sizeof(int), hipMemcpyHostToDevice) != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    hipLaunchKernelGGL(k_pfb_spectral, dim3(LB / SOLVE_WG), dim3(SOLVE_WG), 0, 0, (const float *)p->win, nb, p->tab,
                       d_refused);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpy(&refused, d_refused, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess) {
        rc = SDBE_ERR_HIP;
        goto fail;
    }
    p->constant = refused == 0;
    if (p->constant) {
        p->nb = nb;
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
                hipLaunchKernelGGL(k_pfb_join<true>, br, wg, 0, s, tab, N, nb, (const double *)P, (const double *)Q, A, B, p->tc);
            else
                hipLaunchKernelGGL(k_pfb_join<false>, br, wg, 0, s, tab, N, nb, (const double *)P, (const double *)Q, A, B, p->tc);
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
