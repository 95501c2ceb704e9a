// Building blocks of the LDS-resident FFT kernels (fft.hip, fft256.hip): complex
// helpers, the in-register radix-2 DFT, the two-level transform over a lane group
// and the reference's prepare expression.
//
// The single-kernel paths are bound by vector instructions, so the transforms count them: a
// product for every twiddle between the levels and radix-4 passes took 332 per lane and 16
// values of an inverse 128-point transform; the folded butterflies below take 296, with 8
// twiddles read from LDS instead of 15 (a float inverse 312: kFoldInverse).  25600 slices of
// 64 px in float: 622 -> 612 us; 6400 in double: 501 -> 476 us; 6400 of 128 px in float: 861
// -> 842 us; 648 of 96 px in double (fftg.hip): 221 -> 205 us.  Offsets of slices like a
// scan's against 64 bits, in float: 20 to 150 px 0 to 22% nearer than before.
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace emida_amd {

// ------------------------------------------------------------------ complex helpers
template <class T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) {
    return {a.re + b.re, a.im + b.im};
}
template <class T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) {
    return {a.re - b.re, a.im - b.im};
}
template <class T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> w) {
    return {a.re * w.re - a.im * w.im, a.re * w.im + a.im * w.re};
}
template <class T>
__device__ __forceinline__ cplx<T> cmul_conj(cplx<T> a, cplx<T> w) {  // a * conj(w)
    return {a.re * w.re + a.im * w.im, a.im * w.re - a.re * w.im};
}
// The reference's product p * conj(r) (src/hadamard.cu:39-40), same expression.
template <class T>
__device__ __forceinline__ cplx<T> hadamard(cplx<T> p, cplx<T> r) {
    return {p.re * r.re + p.im * r.im, -p.re * r.im + p.im * r.re};
}

// cos and tan of 2 pi q / 32, q < 8; the tangent as the sine over the rounded cosine, so
// that their product is the sine to one rounding.
template <class T>
constexpr T cos32(int q) {
    return T(q == 0 ? 1 : q == 1 ? 0.9807852804032304 : q == 2 ? 0.9238795325112867 : q == 3 ? 0.8314696123025452
           : q == 4 ? 0.7071067811865476 : q == 5 ? 0.5555702330196022 : q == 6 ? 0.3826834323650898 : 0.19509032201612828);
}
template <class T>
constexpr T tan32(int q) {
    return q == 0 ? T(0) : T(cos32<double>(8 - q) / (double)cos32<T>(q));
}

__host__ __device__ constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }
__host__ __device__ constexpr int brev_c(int v, int bits) {
    int r = 0;
    for (int b = 0; b < bits; ++b) r |= ((v >> b) & 1) << (bits - 1 - b);
    return r;
}

// Radix-2 butterflies (a, b) -> (a + w b, a - w b), decimation in time: the twiddle before
// the butterfly folds into it.  w = exp(-+ i p) = cos p (1 -+ i tan p), 0 <= p < pi / 2 (INV:
// upper sign conjugated): u = b / cos p is two fused operations, a +- cos p u four, six in
// all where a product and two sums take eight.  The rounding of u scales with the product
// itself (u times cos p).  TURN: w times a quarter turn more.
template <class T, bool INV, bool TURN>
__device__ __forceinline__ void butterfly_tan(cplx<T>& a, cplx<T>& b, T c, T t) {
    const T ur = fma(INV ? -t : t, b.im, b.re), ui = fma(INV ? t : -t, b.re, b.im);
    // w b / c, or that times -i (INV: i)
    const T vr = TURN ? (INV ? -ui : ui) : ur, vi = TURN ? (INV ? ur : -ur) : ui;
    const cplx<T> s = a;
    a = cplx<T>{fma(c, vr, s.re), fma(c, vi, s.im)};
    b = cplx<T>{fma(-c, vr, s.re), fma(-c, vi, s.im)};
}
// w = 1, or a quarter turn.
template <class T, bool INV, bool TURN>
__device__ __forceinline__ void butterfly_one(cplx<T>& a, cplx<T>& b) {
    const cplx<T> s = a, v = TURN ? (INV ? cplx<T>{-b.im, b.re} : cplx<T>{b.im, -b.re}) : b;
    a = cadd(s, v);
    b = csub(s, v);
}

// 32 double points fill the registers: each half is computed where it stands, not moved
// towards its uses (spills otherwise).
template <class T, int N>
__device__ __forceinline__ void hold(cplx<T> (&x)[N]) {
    if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i].re), "+v"(x[i].im));
    }
}

// In-register DFT of N <= 32 points, natural order in and out (the digit reversal only
// renames registers).  HALF_ZERO: x[N/2..N-1] = 0, not read.
template <class T, int N, bool INV, bool HALF_ZERO = false>
__device__ __forceinline__ void dft_reg(cplx<T> (&x)[N]) {
    static_assert(N >= 2 && N <= 32 && (N & (N - 1)) == 0, "N must be a power of two <= 32");
    if constexpr (N == 32) {  // (in one piece its registers go to scratch)
        cplx<T> e[16], o[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            e[i] = x[HALF_ZERO ? 2 * i % 16 : 2 * i];
            o[i] = x[HALF_ZERO ? 2 * i % 16 + 1 : 2 * i + 1];
        }
        dft_reg<T, 16, INV, HALF_ZERO>(e);
        hold(e);
        dft_reg<T, 16, INV, HALF_ZERO>(o);
        hold(o);
        butterfly_one<T, INV, false>(e[0], o[0]);
        butterfly_one<T, INV, true>(e[8], o[8]);
#pragma unroll
        for (int j = 1; j < 8; ++j) {
            butterfly_tan<T, INV, false>(e[j], o[j], cos32<T>(j), tan32<T>(j));
            butterfly_tan<T, INV, true>(e[j + 8], o[j + 8], cos32<T>(j), tan32<T>(j));
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            x[i] = e[i];
            x[i + 16] = o[i];
        }
        hold(x);
        return;
    }
    cplx<T> y[N];
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = x[HALF_ZERO ? brev_c(i, ilog2(N)) % (N / 2) : brev_c(i, ilog2(N))];
#pragma unroll
    for (int n = HALF_ZERO ? 4 : 2; n <= N; n *= 2) {
#pragma unroll
        for (int b = 0; b < N; b += n) {
#pragma unroll
            for (int j = 0; j < n / 2; ++j) {
                cplx<T>&p = y[b + j], &q = y[b + j + n / 2];
                if (j == 0) butterfly_one<T, INV, false>(p, q);
                else if (4 * j == n) butterfly_one<T, INV, true>(p, q);
                else if (4 * j < n) butterfly_tan<T, INV, false>(p, q, cos32<T>(32 * j / n), tan32<T>(32 * j / n));
                else butterfly_tan<T, INV, true>(p, q, cos32<T>(32 * j / n - 8), tan32<T>(32 * j / n - 8));
            }
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = y[i];
}

// Intra-wave LDS hand-off between the lanes of one FFT group.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// DFT of N points x[m] W_M^(m f) (INV: conjugated), natural order: the twiddles between the
// two levels of an M-point transform folded into the second level's butterflies.  The pass
// that joins blocks of n points takes W_M^(f N / n + j M / n), j < n / 2: below a quarter
// turn for j < n / 4 and n >= 4 with f < M / N, so (cos, tan) from the table, a quarter turn
// more for the others; n = 2 reaches half a turn: w itself, a - w b as 2 a - (a + w b).
// tab (load_twist): (cos, tan) of 2 pi t / M, t < M / 4, then W_2R^r, r < R.
constexpr int twist_elems(int m, int r) { return m / 4 + r; }
// F: points of the whole DFT where this is the half of its even or odd inputs.
template <class T, int N, int M, int R, bool INV, int F = N>
__device__ __forceinline__ void dft_twist(cplx<T> (&x)[N], const cplx<T>* tab, int f) {
    if constexpr (N == 32) {
        cplx<T> e[16], o[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            e[i] = x[2 * i];
            o[i] = x[2 * i + 1];
        }
        dft_twist<T, 16, M, R, INV, F>(e, tab, f);
        hold(e);
        dft_twist<T, 16, M, R, INV, F>(o, tab, f);
        hold(o);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const cplx<T> ct = tab[f + j * (M / 32)];
            butterfly_tan<T, INV, false>(e[j], o[j], ct.re, ct.im);
            butterfly_tan<T, INV, true>(e[j + 8], o[j + 8], ct.re, ct.im);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            x[i] = e[i];
            x[i + 16] = o[i];
        }
        hold(x);
        return;
    }
    cplx<T> y[N];
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = x[brev_c(i, ilog2(N))];
    const cplx<T> w = tab[M / 4 + f * (F * R / M)];
#pragma unroll
    for (int b = 0; b < N; b += 2) {
        const cplx<T> a = y[b], q = y[b + 1];
        const T wi = INV ? -w.im : w.im;
        const T sr = fma(-wi, q.im, fma(w.re, q.re, a.re)), si = fma(wi, q.re, fma(w.re, q.im, a.im));
        y[b] = cplx<T>{sr, si};
        y[b + 1] = cplx<T>{fma(T(2), a.re, -sr), fma(T(2), a.im, -si)};
    }
#pragma unroll
    for (int n = 4; n <= N; n *= 2) {
#pragma unroll
        for (int j = 0; j < n / 4; ++j) {
            const cplx<T> ct = tab[f * (F / n) + j * (M / n)];
#pragma unroll
            for (int b = 0; b < N; b += n) {
                butterfly_tan<T, INV, false>(y[b + j], y[b + j + n / 2], ct.re, ct.im);
                butterfly_tan<T, INV, true>(y[b + j + n / 4], y[b + j + n / 4 + n / 2], ct.re, ct.im);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = y[i];
}

// Forward transform: lane n2 holds x[n1] = input[L*n1 + n2]; on return lane j holds
// X[(j + L*i) + R*k2] in x[i*L + k2].  scr: L*(R+1) elements of this group.
// HALF_ZERO: the inputs x[R/2..R-1] are zero padding.
template <class T, int R, int L, int M, bool HALF_ZERO>
__device__ __forceinline__ void fft_fwd(cplx<T> (&x)[R], int lane, cplx<T>* scr, const cplx<T>* tw) {
    constexpr int Q = R / L;
    dft_reg<T, R, false, HALF_ZERO>(x);
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) scr[lane * (R + 1) + k1] = x[k1];
    wave_sync();
    cplx<T> y[Q][L];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int m = 0; m < L; ++m) y[i][m] = scr[m * (R + 1) + lane + L * i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        dft_twist<T, L, M, R, false>(y[i], tw, lane + L * i);
#pragma unroll
        for (int k2 = 0; k2 < L; ++k2) x[i * L + k2] = y[i][k2];
    }
}

// Second level of an inverse transform.  Folded twiddles multiply an output by one cosine per
// pass, and the rounding of those few cosines moves the whole output: unlike the errors of a
// sum it differs from one shift to the next, which tilts the fitted peak (offsets of 64 px
// slices in float: 20% further from 64 bits, 33 px 40%).  With the products W_M^(lane k) before
// plain passes, outputs 0..L-1 meet no other twiddle and the errors of the R products average
// out: offsets 16% nearer than with radix 4 at 64 px, 22% at 250.  It costs 16 operations and 7
// twiddles (25600 slices of 64 px: 608 -> 612 us; 672 of 161 x 95: 281 -> 292 us).  Folded where
// that rounding is far below the fit's own (double), and in fft256.hip, whose neighbourhood comes from
// direct sums (128 px: offsets 1% nearer than with radix 4).
template <class T>
constexpr bool kFoldInverse = sizeof(T) == 8;
// tab elements of an inverse transform of M = R L points
template <class T>
constexpr int inv_twist_elems(int m, int r) { return twist_elems(m, r) + (kFoldInverse<T> ? 0 : m + m / r); }
template <class T, int R, int M, bool FOLD>
__device__ __forceinline__ void dft_last(cplx<T> (&x)[R], const cplx<T>* tw, int lane) {
    if constexpr (FOLD) {
        dft_twist<T, R, M, R, true>(x, tw, lane);
    } else {
        const cplx<T>* t = tw + twist_elems(M, R) + lane * (R + 1);
#pragma unroll
        for (int k = 1; k < R; ++k) x[k] = cmul_conj(x[k], t[k]);
        dft_reg<T, R, true>(x);
    }
}

// Inverse (unnormalised) transform from the frequency layout to natural order:
// on return lane n2 holds output[L*n1 + n2] in x[n1].
template <class T, int R, int L, int M, bool FOLD = kFoldInverse<T>>
__device__ __forceinline__ void fft_inv(cplx<T> (&x)[R], int lane, cplx<T>* scr, const cplx<T>* tw) {
    constexpr int Q = R / L;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        cplx<T> y[L];
#pragma unroll
        for (int k2 = 0; k2 < L; ++k2) y[k2] = x[i * L + k2];
        dft_reg<T, L, true>(y);
#pragma unroll
        for (int n2 = 0; n2 < L; ++n2) scr[n2 * (R + 1) + lane + L * i] = y[n2];
    }
    wave_sync();
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) x[k1] = scr[lane * (R + 1) + k1];
    wave_sync();
    dft_last<T, R, M, FOLD>(x, tw, lane);
}

// Prepared pixel (src/prepare_pics.cu:36-41), no contraction.
// Workgroup maximum / minimum for arrays used once per kernel: one barrier (the
// trailing one that would guard the array's reuse is not needed).  Every thread of
// the workgroup must call them (the wave steps read all 64 lanes).
template <class T, int NT>
__device__ __forceinline__ T block_max_once(T v, T* sv) {
    v = wave_reduce(v, -(T)__builtin_huge_val(), [](T x, T y) { return fmax(x, y); });
    if (threadIdx.x % kWave == 0) sv[threadIdx.x / kWave] = v;
    __syncthreads();
    v = sv[0];
#pragma unroll
    for (int k = 1; k < NT / kWave; ++k) v = fmax(v, sv[k]);
    return v;
}
template <int NT>
__device__ __forceinline__ uint32_t block_min_once_u32(uint32_t v, uint32_t* sv) {
    v = wave_reduce(v, 0xffffffffu, [](uint32_t x, uint32_t y) { return min(x, y); });
    if (threadIdx.x % kWave == 0) sv[threadIdx.x / kWave] = v;
    __syncthreads();
    v = sv[0];
#pragma unroll
    for (int k = 1; k < NT / kWave; ++k) v = min(v, sv[k]);
    return v;
}

template <class T, class IN>
__device__ __forceinline__ T prep_px(IN px, T mean, T wx, T wy) {
#pragma clang fp contract(off)
    T v = (T)px;
    v -= mean;
    v = v * wx * wy;
    return v;
}

template <class T>
__device__ __forceinline__ T mean_of(T sum, uint32_t area) {
#pragma clang fp contract(off)
    return sum / (T)area;
}

// Workgroup -> slice (pattern * nb + roi).  Workgroups are dispatched round robin
// over the 8 XCDs (b mod 8); XCD x takes a contiguous run of the ROI-major order
// (roi * npat + pattern), so the patterns of a ROI run back to back on one XCD and
// that ROI's reference spectrum stays in the XCD's L2.
__device__ __forceinline__ uint32_t xcd_slice(uint32_t b, uint32_t total, uint32_t nb) {
    const uint32_t o = xcd_remap(b, total);
    const uint32_t npat = total / nb;
    return (o % npat) * nb + o / npat;
}

template <class T, class IN, class SUM>
struct fft_args {
    const IN* pics;          // patterns (FROM_PATTERN)
    const SUM* sums;         // per-slice sums (FROM_PATTERN, IN != uint16)
    const T* hx;             // Hann windows (FROM_PATTERN)
    const T* hy;
    const size2* begins;     // ROI corners
    size2 src;               // pattern size
    uint32_t side;           // slice side s (at most half the transform size)
    uint32_t nb;             // ROIs per pattern
    uint32_t total;          // slices in this launch
    const T* prepared;       // prepared s x s slices (!FROM_PATTERN)
    const cplx<T>* spectra;  // reference spectra (PIPE)
    cplx<T>* spectra_out;    // reference spectra (!PIPE)
    int fit;
    const double* lsq;
    data_index<T>* maxes;
    T* neigh;
    double* offsets;
    double* coefs;
    T* corr_out;             // optional (2s)^2 circular buffers in the reference layout, row-major
    const cplx<T>* twt;      // twiddle tables (fft_twiddles)
};

// Copy of the M-entry table into LDS.
template <class T, int M>
__device__ __forceinline__ void load_twiddles(cplx<T>* tw, const cplx<T>* table, int tid, int nt) {
    for (int t = tid; t < M; t += nt) tw[t] = table[tw_offset(M) + t];
}
// The twiddles of dft_twist (twist_elems(M, R) elements) and, unless FOLD, W_M^(n k) as
// [n][k], n < M / R, k < R, rows of R + 1 (an odd stride: a group's lanes on distinct banks).
template <class T, int M, int R, bool FOLD = kFoldInverse<T>>
__device__ __forceinline__ void load_twist(cplx<T>* tw, const cplx<T>* table, int tid, int nt) {
    for (int t = tid; t < twist_elems(M, R); t += nt)
        tw[t] = table[t < M / 4 ? tan_offset(M) + t : tw_offset(M) + (t - M / 4) * (M / (2 * R))];
    if constexpr (!FOLD) {
        for (int t = tid; t < M + M / R; t += nt) {
            const int n = t / (R + 1), k = t % (R + 1);
            tw[twist_elems(M, R) + t] = table[tw_offset(M) + (k < R ? n * k % M : 0)];
        }
    }
}

}  // namespace emida_amd
