// FFT cross-correlation for every slice shape the single-kernel pipelines (fft.hip,
// fft256.hip) do not take: non-square slices, double slices of side 65..256 and float
// slices of side 129..256 (transforms of up to 512 x 512).  cuFFT plans any
// 2s.x x 2s.y transform for the reference (src/gpu_offset.hpp:121-123,171-183); here
// the transform is Mx x My, each the power of two >= 2s of its axis (or 192 or 384), with the same
// correlation values (zero padding beyond 2s changes no shift |d| < s), read through
// the reference's 2s.x x 2s.y layout as in fft.hip.
//
// Four kernels per launch chunk, with a work buffer of half spectra in HBM
// ([slice][y][kx], kx <= Mx/2, the layout of an R2C result):
//  1. rows: two real rows packed as one complex row (prepared from the pattern or
//     read from prepared slices), an Mx-point transform, split into the two half
//     spectra (the split's factor 1/2 omitted: results come out doubled);
//  2. columns: an My-point transform of each half-spectrum column, the product with the
//     conjugate reference spectrum (src/hadamard.cu:39-40) and the inverse transform, in
//     place - or, for the reference, the scaled spectrum stored ([roi][kx][ky],
//     column-major, read by lanes in order);
//  3. rows, inverse: two output rows packed as Ga + i Gb (Hermitian extension, DC and
//     Nyquist imaginary parts dropped, as a C2R does), one inverse transform yields both
//     real rows of the reference's (2s.x x 2s.y) circular correlation and their largest
//     value; the correlation itself is not written (the seams write it instead);
//  4. peaks: the arg-max over a slice's row pairs, the row pairs of the neighbourhood
//     again (cross_res_pos_policy_fft, src/kernels.cuh:36-53), fit and finalize.
// A transform runs on L lanes of one wave with R = M / L values each in registers and one
// transpose through LDS (fft_common.hpp).
//
// Bound: the half spectra in HBM.  8 patterns x 81 ROIs of 96 x 96 in double (192 x 192):
// 0.58 GB written and read, 197 us (rows 31, columns 75, inverse rows 56, peaks 11); radix-4 passes
// through LDS over 256 x 256, a staged column tile and the correlation written for a peak
// kernel took 495 us.  16 patterns x 42 ROIs of 161 x 95 in float (384 x 192): 252 us (sums
// 14, rows 43, columns 87, inverse rows 81, peaks 12), before 606 us.
//
// Scale: the pattern's spectrum comes out doubled (the omitted split factor); the
// stored reference spectrum is 2 s.x s.y / (Mx My) times the true one (the same
// stages double it, launch_fftg_ref multiplies by s.x s.y / (Mx My)), so the
// unnormalised inverse carries the reference's 4 s.x s.y scale; all factors are
// exact powers of two when M = 2s.
//
// The same kernels give the reference's own cross_corr_fft (R2C, product with a
// spectrum in the R2C layout, C2R; src/gpu_offset.hpp:303-316) on 2s x 2s buffers
// (standard layouts, factor 1/2 applied to undo the doubling, exact).
#include "fft_common.hpp"

namespace emida_amd {

namespace {

constexpr int kGNT = 256;  // threads of every kernel

// Transform lengths: powers of two, and 192 and (float) 384 as three transforms of a third of
// the length (every third input) and 3-point DFTs: they move 25% fewer bytes per axis than 256
// and 512 (161 x 95 in float, 576 slices: 225 us with 384 x 192, 250 with 512 x 256; 190 x 190,
// 400: 311 and 370; 96 x 96 in double, 648: 181 and 225).  384 in double spills (161 x 95: 504
// and 249 us); 48 and 96 gain less in bytes than the longer register transform costs (48 x 24
// in float: 229 and 172 when both were tried).
constexpr bool gthree(int m) { return m % 3 == 0; }
constexpr int gbase(int m) { return gthree(m) ? m / 3 : m; }  // length of the transforms in registers
constexpr int glanes(int m) { return gbase(m) >= 256 ? 16 : gbase(m) >= 64 ? 8 : gbase(m) >= 16 ? 4 : 2; }
constexpr int gsub(int m) { return gbase(m) / glanes(m); }  // values per lane of one of them
constexpr int gregs(int m) { return m / glanes(m); }        // values per lane
// Place of a lane's value r: time (input of the forward, output of the inverse transform) ...
__device__ __forceinline__ constexpr int gtime(int m, int r, int lane) {
    const int n = glanes(m) * (r % gsub(m)) + lane;
    return gthree(m) ? 3 * n + r / gsub(m) : n;
}
// ... and frequency.
__device__ __forceinline__ constexpr int gfreq(int m, int r, int lane) {
    const int q = r / gsub(m), i = r % gsub(m) / glanes(m), k2 = r % gsub(m) % glanes(m);
    return lane + glanes(m) * i + gsub(m) * k2 + gbase(m) * q;
}
// With at most M / 2 input values the second half of every register transform is zero.
constexpr bool gzero(int m, int r) { return r % gsub(m) >= gsub(m) / 2; }

// LDS: twiddles (complex): of the register transforms, then W_M^k and W_M^2k; per lane
// group, in T: the transpose scratch of the real or the imaginary parts, which also holds a
// whole real row.  Half of a complex scratch: twice the workgroups per CU (256-point
// transforms in double: 39 KB instead of 74).
template <class T>
constexpr int greg_tw(int m) { return inv_twist_elems<T>(gbase(m), gsub(m)); }
template <class T>
constexpr int gtw(int m) { return greg_tw<T>(m) + (gthree(m) ? 2 * gbase(m) : 0); }
constexpr int gslot(int m) { return gthree(m) ? m + 8 : glanes(m) * (gsub(m) + 1); }
template <class T>
constexpr size_t glds(int m) {
    return (2 * (size_t)gtw<T>(m) + (size_t)(kGNT / glanes(m)) * gslot(m)) * sizeof(T);
}
template <class T, int M, int NT = kGNT>
__device__ __forceinline__ void gload_twiddles(cplx<T>* tw, const cplx<T>* table, int tid) {
    constexpr int P = gbase(M);
    load_twist<T, P, gsub(M)>(tw, table, tid, NT);
    if constexpr (gthree(M)) {
        cplx<T>* t3 = tw + greg_tw<T>(M);
        for (int k = tid; k < P; k += NT) {
            t3[k] = table[tw_offset(M) + k];
            t3[P + k] = table[tw_offset(M) + 2 * k];
        }
    }
}

constexpr double kR3 = 0.8660254037844386;  // sin(pi / 3)

// fft_fwd and fft_inv of fft_common.hpp with the transpose in two passes, real parts then
// imaginary parts, through L (R + 1) values of T.
template <class T, int R, int L, bool HALF_ZERO>
__device__ __forceinline__ void gfft_fwd_reg(cplx<T> (&x)[R], int lane, T* scr, const cplx<T>* tw) {
    constexpr int Q = R / L;
    dft_reg<T, R, false, HALF_ZERO>(x);
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) scr[lane * (R + 1) + k1] = x[k1].re;
    wave_sync();
    cplx<T> y[Q][L];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int m = 0; m < L; ++m) y[i][m].re = scr[m * (R + 1) + lane + L * i];
    wave_sync();
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) scr[lane * (R + 1) + k1] = x[k1].im;
    wave_sync();
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int m = 0; m < L; ++m) y[i][m].im = scr[m * (R + 1) + lane + L * i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        dft_twist<T, L, R * L, R, false>(y[i], tw, lane + L * i);
#pragma unroll
        for (int k2 = 0; k2 < L; ++k2) x[i * L + k2] = y[i][k2];
    }
}

template <class T, int R, int L>
__device__ __forceinline__ void gfft_inv_reg(cplx<T> (&x)[R], int lane, T* scr, const cplx<T>* tw) {
    constexpr int Q = R / L;
#pragma unroll
    for (int i = 0; i < Q; ++i) dft_reg<T, L, true>(*reinterpret_cast<cplx<T>(*)[L]>(&x[i * L]));
    T re[R];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int n2 = 0; n2 < L; ++n2) scr[n2 * (R + 1) + lane + L * i] = x[i * L + n2].re;
    wave_sync();
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) re[k1] = scr[lane * (R + 1) + k1];
    wave_sync();
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int n2 = 0; n2 < L; ++n2) scr[n2 * (R + 1) + lane + L * i] = x[i * L + n2].im;
    wave_sync();
#pragma unroll
    for (int k1 = 0; k1 < R; ++k1) x[k1] = cplx<T>{re[k1], scr[lane * (R + 1) + k1]};
    wave_sync();
    dft_last<T, R, R * L, kFoldInverse<T>>(x, tw, lane);
}

// M-point transforms: registers in gtime order to gfreq order and back.  HALF_ZERO: the inputs
// with gzero are zero.
template <class T, int M, bool HALF_ZERO>
__device__ __forceinline__ void gfft_fwd(cplx<T> (&x)[gregs(M)], int lane, T* scr, const cplx<T>* tw) {
    using C = cplx<T>;
    constexpr int R = gsub(M), L = glanes(M), P = gbase(M);
    if constexpr (!gthree(M)) {
        gfft_fwd_reg<T, R, L, HALF_ZERO>(x, lane, scr, tw);
    } else {
        C(&x0)[R] = *reinterpret_cast<C(*)[R]>(&x[0]);
        C(&x1)[R] = *reinterpret_cast<C(*)[R]>(&x[R]);
        C(&x2)[R] = *reinterpret_cast<C(*)[R]>(&x[2 * R]);
        gfft_fwd_reg<T, R, L, HALF_ZERO>(x0, lane, scr, tw);
        gfft_fwd_reg<T, R, L, HALF_ZERO>(x1, lane, scr, tw);
        gfft_fwd_reg<T, R, L, HALF_ZERO>(x2, lane, scr, tw);
        const C* t3 = tw + greg_tw<T>(M);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = gfreq(P, r, lane);
            const C a = x[r], b = cmul(x[R + r], t3[k]), c = cmul(x[2 * R + r], t3[P + k]);
            const C s = cadd(b, c), d = csub(b, c), m{a.re - T(0.5) * s.re, a.im - T(0.5) * s.im};
            const C t{T(kR3) * d.im, T(-kR3) * d.re};  // -i sin(pi/3) (b - c)
            x[r] = cadd(a, s);
            x[R + r] = cadd(m, t);
            x[2 * R + r] = csub(m, t);
        }
    }
}

template <class T, int M>
__device__ __forceinline__ void gfft_inv(cplx<T> (&x)[gregs(M)], int lane, T* scr, const cplx<T>* tw) {
    using C = cplx<T>;
    constexpr int R = gsub(M), L = glanes(M), P = gbase(M);
    if constexpr (!gthree(M)) {
        gfft_inv_reg<T, R, L>(x, lane, scr, tw);
    } else {
        const C* t3 = tw + greg_tw<T>(M);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = gfreq(P, r, lane);
            const C a = x[r], s = cadd(x[R + r], x[2 * R + r]), d = csub(x[R + r], x[2 * R + r]);
            const C m{a.re - T(0.5) * s.re, a.im - T(0.5) * s.im}, t{T(-kR3) * d.im, T(kR3) * d.re};
            x[r] = cadd(a, s);
            x[R + r] = cmul_conj(cadd(m, t), t3[k]);
            x[2 * R + r] = cmul_conj(csub(m, t), t3[P + k]);
        }
        C(&x0)[R] = *reinterpret_cast<C(*)[R]>(&x[0]);
        C(&x1)[R] = *reinterpret_cast<C(*)[R]>(&x[R]);
        C(&x2)[R] = *reinterpret_cast<C(*)[R]>(&x[2 * R]);
        gfft_inv_reg<T, R, L>(x0, lane, scr, tw);
        gfft_inv_reg<T, R, L>(x1, lane, scr, tw);
        gfft_inv_reg<T, R, L>(x2, lane, scr, tw);
    }
}

}  // namespace

// Arguments of the four kernels (one launch chunk of slices first .. first + total - 1).
template <class T, class IN, class SUM>
struct fftg_args {
    const IN* pics;          // patterns (rows kernel, from pattern)
    const SUM* sums;         // per-slice sums (IN != uint16)
    const T* hx;             // Hann windows
    const T* hy;
    const size2* begins;     // ROI corners
    size2 src;               // pattern size
    const T* prepared;       // prepared slices (rows kernel, from prepared): [slice][rows][pitch]
    uint32_t pitch;          // prepared row pitch (elements)
    uint32_t in_rows, in_cols;  // rows / columns of input per slice (the rest is zero padding)
    uint32_t slice_elems;    // prepared elements per slice
    size2 side;              // slice size s
    uint32_t mx, my;         // transform sizes
    uint32_t nb;             // ROIs per pattern
    uint32_t first, total;   // slices of this chunk
    cplx<T>* work;           // [slice - first][my][mx/2 + 1]
    const cplx<T>* spectra;  // reference spectra (column kernel, product)
    cplx<T>* spectra_out;    // reference spectra (column kernel, spectrum out)
    T scale;                 // spectrum out: factor; product: factor on the product
    size2 out;               // output layout of the inverse rows kernel (2s.x x 2s.y)
    T* corr;                 // [slice - first][out.y][out.x] (the seams)
    uint32_t npat;           // patterns of a chunk of whole patterns, else 0
    const cplx<T>* twt;      // twiddle tables (fft_twiddles)
    int fit;                 // peak outputs (as launch_fft_pipe)
    const double* lsq;
    data_index<T>* maxes;
    T* neigh;
    double* offsets;
    double* coefs;
};

// Waves per SIMD the registers are budgeted for.  The pipeline's forward rows of 384 in float
// and columns of 128 in double need 186 and 172 registers by themselves and none of them in
// scratch at 168, which lets a third workgroup share a CU (the LDS holds three): 672 slices of
// 161 x 95 in float 277 -> 261 us, 2304 of 60 x 50 in double 212 -> 200.  The other kernels
// above 168 would spill 12 bytes to 800 a lane, among them the same lengths without zero
// padding (hz).
template <class T>
constexpr int gwaves(int m, int three, int size, bool hz) {
    return m == three && sizeof(T) == size && hz ? 3 : 2;
}

// ---------------------------------------------------------------- kernel 1: rows
// HZ: the second half of every row is zero padding (slices of at most Mx / 2 columns).
// Grid: (slices, splits); a slice's splits take its row pairs in turn (uint16: each sums
// the whole slice for the mean).
template <class T, class IN, class SUM, int MX, bool FROM_PATTERN, bool HZ>
__global__ __launch_bounds__(kGNT, gwaves<T>(MX, 384, 4, HZ)) void fftg_rows_kernel(fftg_args<T, IN, SUM> a) {
    using C = cplx<T>;
    constexpr int L = glanes(MX), R = gregs(MX), NG = kGNT / L, NCX = MX / 2 + 1;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C* tw = reinterpret_cast<C*>(lds_raw);
    __shared__ uint32_t red_u[kGNT / kWave];
    const int tid = threadIdx.x, g = tid / L, lane = tid % L;
    T* slot = reinterpret_cast<T*>(tw + gtw<T>(MX)) + gslot(MX) * g;
    const uint32_t sl = blockIdx.x, sn = a.first + sl;
    gload_twiddles<T, MX>(tw, a.twt, tid);

    const IN* pic = nullptr;
    const T* pre = nullptr;
    T mean = T(0);
    const int sx = (int)a.in_cols, sy = (int)a.in_rows;
    if constexpr (FROM_PATTERN) {
        const size2 b0 = a.begins[sn % a.nb];
        pic = a.pics + (size_t)(sn / a.nb) * a.src.area() + (size_t)b0.y * a.src.x + b0.x;
        if constexpr (std::is_same<IN, uint16_t>::value) {
            uint32_t su = 0;
            constexpr int U = 8;  // rows in flight per wave
            for (int x = tid % kWave; x < sx; x += kWave)
                for (int y0 = tid / kWave; y0 < sy; y0 += kGNT / kWave * U) {
                    uint32_t v[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int y = y0 + kGNT / kWave * u;
                        v[u] = pic[(size_t)min(y, sy - 1) * a.src.x + x];
                        v[u] = y < sy ? v[u] : 0u;
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) su += v[u];
                }
            su = wave_reduce(su, 0u, [](uint32_t x, uint32_t y) { return x + y; });
            if (tid % kWave == 0) red_u[tid / kWave] = su;
            __syncthreads();
            su = 0;
#pragma unroll
            for (int k = 0; k < kGNT / kWave; ++k) su += red_u[k];
            mean = mean_of<T>((T)su, sx * sy);
        } else {
            mean = mean_of<T>((T)a.sums[sn], sx * sy);
        }
    } else {
        pre = a.prepared + (size_t)sn * a.slice_elems;
    }
    __syncthreads();

    C* w = a.work + (size_t)sl * a.my * NCX;
    const int npairs = (sy + 1) / 2;
    for (int p = g + NG * (int)blockIdx.y; p < npairs; p += NG * (int)gridDim.y) {
        const bool second = 2 * p + 1 < sy;
        const int y0 = 2 * p, y1 = second ? 2 * p + 1 : 2 * p;
        C x[R];
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) x[n1] = C{T(0), T(0)};
        T wy0 = T(0), wy1 = T(0);
        if constexpr (FROM_PATTERN) {
            wy0 = a.hy[y0];
            wy1 = a.hy[y1];
        }
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            if (HZ && gzero(MX, n1)) continue;
            const int n = gtime(MX, n1, lane), nc = min(n, sx - 1);
            T v0, v1;
            if constexpr (FROM_PATTERN) {
                const T wx = a.hx[nc];
                v0 = prep_px<T, IN>(pic[(size_t)y0 * a.src.x + nc], mean, wx, wy0);
                v1 = prep_px<T, IN>(pic[(size_t)y1 * a.src.x + nc], mean, wx, wy1);
            } else {
                v0 = pre[(size_t)y0 * a.pitch + nc];
                v1 = pre[(size_t)y1 * a.pitch + nc];
            }
            if (n < sx) x[n1] = C{v0, second ? v1 : T(0)};
        }
        gfft_fwd<T, MX, HZ>(x, lane, slot, tw);
        // split: frequencies k and Mx - k through the slot, real parts, then imaginary parts
        constexpr int NK = MX / 2 / L + 1;  // frequencies lane + L i <= Mx / 2 of a lane
        T sre[NK], dre[NK];
        auto put = [&](auto&& part) {
#pragma unroll
            for (int r = 0; r < R; ++r) slot[gfreq(MX, r, lane)] = part(x[r]);
            wave_sync();
        };
        put([](const C& v) { return v.re; });
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int k = lane + L * i;
            const T z = slot[k], m = slot[k == 0 ? 0 : MX - k];
            sre[i] = z + m;
            dre[i] = m - z;
        }
        wave_sync();
        put([](const C& v) { return v.im; });
        C* r0 = w + (size_t)y0 * NCX;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int k = lane + L * i;
            const T z = slot[k], m = slot[k == 0 ? 0 : MX - k];
            if (k < NCX) {
                r0[k] = C{sre[i], z - m};
                if (second) r0[NCX + k] = C{z + m, dre[i]};
            }
        }
        wave_sync();  // the slot is the next row pair's scratch
    }
}

// ---------------------------------------------------------------- kernel 2: columns
enum { COLS_PIPE = 0, COLS_SPECTRUM = 1, COLS_STD_PIPE = 2, COLS_STD_SPECTRUM = 3 };
constexpr bool gcols_hz(int mode) { return mode == COLS_PIPE || mode == COLS_SPECTRUM; }

// One column per lane group, read and written in place: the NG groups of a workgroup take
// adjacent columns, so the lanes of a row read at least 64 consecutive bytes.  The columns
// of the patterns of one ROI run back to back on one XCD (one spectrum column in its L2).
template <class T, int MY, int MODE>
__global__ __launch_bounds__(kGNT, gwaves<T>(MY, 128, 8, gcols_hz(MODE))) void fftg_cols_kernel(fftg_args<T, T, T> a, uint32_t nblk) {
    using C = cplx<T>;
    constexpr bool HZ = gcols_hz(MODE);
    constexpr int L = glanes(MY), R = gregs(MY), NG = kGNT / L;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C* tw = reinterpret_cast<C*>(lds_raw);
    const int tid = threadIdx.x, g = tid / L, lane = tid % L;
    T* slot = reinterpret_cast<T*>(tw + gtw<T>(MY)) + gslot(MY) * g;
    const int ncx = (int)a.mx / 2 + 1;
    const uint32_t gx = div_up((uint32_t)ncx, (uint32_t)NG), b = xcd_remap(blockIdx.x, nblk);
    uint32_t sl, col;
    if (a.npat) {
        const uint32_t roi = b / (gx * a.npat), in = b - roi * gx * a.npat;
        col = in / a.npat;
        sl = (in - col * a.npat) * a.nb + roi;
    } else {
        sl = b / gx;
        col = b - sl * gx;
    }
    const uint32_t roi = (a.first + sl) % a.nb;
    const int kx = (int)col * NG + g;
    gload_twiddles<T, MY>(tw, a.twt, tid);
    C* w = a.work + (size_t)sl * a.my * ncx + min(kx, ncx - 1);
    const int rows = HZ ? (int)a.side.y : (int)a.my;
    C x[R];
#pragma unroll
    for (int n1 = 0; n1 < R; ++n1) x[n1] = C{T(0), T(0)};
#pragma unroll
    for (int n1 = 0; n1 < R; ++n1) {
        if (HZ && gzero(MY, n1)) continue;
        const int y = gtime(MY, n1, lane);
        const C v = w[(size_t)min(y, rows - 1) * ncx];
        x[n1] = y < rows ? v : C{T(0), T(0)};
    }
    __syncthreads();  // twiddles
    if (kx >= ncx) return;
    // the reference spectrum: in flight during the forward transform where registers allow
    auto spec_at = [&](int r) {
        const int k = gfreq(MY, r, lane);
        if constexpr (MODE == COLS_PIPE) return a.spectra[((size_t)roi * ncx + kx) * MY + k];
        else return a.spectra[((size_t)roi * MY + k) * ncx + kx];
    };
    constexpr bool EARLY = R * sizeof(C) <= 256;
    C spec[EARLY ? R : 1];
    if constexpr (EARLY && (MODE == COLS_PIPE || MODE == COLS_STD_PIPE)) {
#pragma unroll
        for (int r = 0; r < R; ++r) spec[r] = spec_at(r);
    }
    gfft_fwd<T, MY, HZ>(x, lane, slot, tw);
    if constexpr (MODE == COLS_SPECTRUM || MODE == COLS_STD_SPECTRUM) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = gfreq(MY, r, lane);
            const C v = C{x[r].re * a.scale, x[r].im * a.scale};
            if constexpr (MODE == COLS_SPECTRUM) a.spectra_out[((size_t)roi * ncx + kx) * MY + k] = v;
            else a.spectra_out[((size_t)roi * MY + k) * ncx + kx] = v;
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (EARLY) x[r] = hadamard(x[r], spec[r]);
            else x[r] = hadamard(x[r], spec_at(r));
            if constexpr (MODE == COLS_STD_PIPE) x[r] = C{x[r].re * a.scale, x[r].im * a.scale};
        }
        gfft_inv<T, MY>(x, lane, slot, tw);
        // rows of the output the inverse rows kernel reads (the reference layout)
        const int sy = (int)a.side.y, pady = MY - 2 * sy;
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            const int y = gtime(MY, n1, lane);
            if (MODE == COLS_STD_PIPE || y <= sy || y > sy + pady) w[(size_t)y * ncx] = x[n1];
        }
    }
}

// ---------------------------------------------------------------- kernel 3: rows, inverse
// Output rows 2q and 2q + 1 of the reference layout of one slice, for one lane group: on
// return a lane holds their packed half spectra at frequencies gfreq.
template <class T, int MX>
__device__ __forceinline__ void load_row_pair(cplx<T> (&x)[gregs(MX)], const cplx<T>* w, int q, int sy, int pady,
                                              int lane) {
    using C = cplx<T>;
    constexpr int R = gregs(MX), NCX = MX / 2 + 1, S = MX / 2;
    // reference-layout row r <= s is circular row r, r > s is r + M - 2s
    const int ra = 2 * q, rb = 2 * q + 1;
    const C* ga_row = w + (size_t)(ra <= sy ? ra : ra + pady) * NCX;
    const C* gb_row = w + (size_t)(rb <= sy ? rb : rb + pady) * NCX;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = gfreq(MX, r, lane);
        const bool mirror = k > S;
        const int col = mirror ? MX - k : k;
        C ga = ga_row[col], gb = gb_row[col];
        if (mirror) {
            ga.im = -ga.im;
            gb.im = -gb.im;
        }
        if (k == 0 || k == S) {
            ga.im = T(0);
            gb.im = T(0);
        }
        x[r] = C{ga.re - gb.im, ga.im + gb.re};
    }
}

// One row pair per lane group.  PEAK: the pair's largest value and its lowest index go to the
// imaginary parts of columns 0 and Mx / 2 of the pair's first row, which a C2R drops; else the
// rows of the correlation buffer.
//
// Grid: (slices, blocks of NG row pairs).  With a slice's row pairs in rounds of one workgroup,
// its arg-max and its fit behind them, 648 slices were 1.3 rounds of the chip, most lanes idle
// during every fit, and the loop's registers spilled at 384.  Inverse rows / with peaks, before
// and now, us: 648 slices of 96 x 96 in double 73 / 56 + 11; 672 of 161 x 95 in float 108 /
// 81 + 12; a pass over 36 of 250 x 250 in float 151 / 78; over 16 of 128 x 128 in double 49 / 30.
template <class T, int MX, bool PEAK>
__global__ __launch_bounds__(kGNT, 2) void fftg_rows_inv_kernel(fftg_args<T, T, T> a) {
    using C = cplx<T>;
    constexpr int L = glanes(MX), R = gregs(MX), NG = kGNT / L, NCX = MX / 2 + 1;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C* tw = reinterpret_cast<C*>(lds_raw);
    const int tid = threadIdx.x, g = tid / L, lane = tid % L;
    T* slot = reinterpret_cast<T*>(tw + gtw<T>(MX)) + gslot(MX) * g;
    const uint32_t sl = blockIdx.x;
    C* w = a.work + (size_t)sl * a.my * NCX;
    // reference-layout index k <= s is circular position k, k > s is k + M - 2s
    const int sx = (int)a.out.x / 2, sy = (int)a.out.y / 2;
    const int padx = MX - (int)a.out.x, pady = (int)a.my - (int)a.out.y;
    const int npairs = (int)a.out.y / 2, q = (int)blockIdx.y * NG + g;
    C x[R];
    load_row_pair<T, MX>(x, w, min(q, npairs - 1), sy, pady, lane);
    gload_twiddles<T, MX, kGNT>(tw, a.twt, tid);
    __syncthreads();
    if (q >= npairs) return;
    gfft_inv<T, MX>(x, lane, slot, tw);
    const uint32_t ia = 2 * (uint32_t)q * a.out.x, ib = ia + a.out.x;
    if constexpr (PEAK) {
        // the lane's largest value and its first column, row a before row b (larger indices, so
        // strictly larger keeps the lowest)
        T va = -(T)__builtin_huge_val(), vb;
        int ca = MX, cb = MX;
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            const int c = gtime(MX, n1, lane);
            const T v = x[n1].re;
            if ((c <= sx || c > sx + padx) && (v > va || (gthree(MX) && v == va && c < ca && ca < MX))) va = v, ca = c;
        }
        vb = va;
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            const int c = gtime(MX, n1, lane);
            const T v = x[n1].im;
            if ((c <= sx || c > sx + padx) && (v > vb || (gthree(MX) && v == vb && c < cb && cb < MX))) vb = v, cb = c;
        }
        uint32_t bi = 0xffffffffu;
        if (ca < MX) bi = ia + (uint32_t)(ca <= sx ? ca : ca - padx);
        if (cb < MX) bi = ib + (uint32_t)(cb <= sx ? cb : cb - padx);
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) {
            const T v = __shfl_xor(vb, off);
            const uint32_t i = __shfl_xor(bi, off);
            if (v > vb || (v == vb && i < bi)) vb = v, bi = i;
        }
        if (lane == 0) {
            C* row = w + (size_t)(2 * q <= sy ? 2 * q : 2 * q + pady) * NCX;
            row[0].im = vb;
            *reinterpret_cast<uint32_t*>(&row[NCX - 1].im) = bi;
        }
    } else {
        T* out = a.corr + (size_t)sl * a.out.area();
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            const int c = gtime(MX, n1, lane);
            if (c <= sx || c > sx + padx) {
                const int rx = c <= sx ? c : c - padx;
                out[ia + rx] = x[n1].re;
                out[ib + rx] = x[n1].im;
            }
        }
    }
}

// ---------------------------------------------------------------- kernel 4: peaks
// One small workgroup per slice: arg-max over the row pairs (lowest index on ties), the row
// pairs of the neighbourhood again, one per lane group, fit and finalize as peak_kernel.
constexpr int gpeak_nt(int m) { return glanes(m) * 16 < kWave ? kWave : glanes(m) * 16; }
template <class T>
constexpr size_t gpeak_lds(int m) {
    return (2 * (size_t)gtw<T>(m) + (size_t)(gpeak_nt(m) / glanes(m)) * gslot(m)) * sizeof(T);
}
template <class T, int MX>
__global__ __launch_bounds__(gpeak_nt(MX)) void fftg_peak_kernel(fftg_args<T, T, T> a) {
    using C = cplx<T>;
    constexpr int NT = gpeak_nt(MX), L = glanes(MX), R = gregs(MX), NCX = MX / 2 + 1;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C* tw = reinterpret_cast<C*>(lds_raw);
    const int tid = threadIdx.x, g = tid / L, lane = tid % L;
    T* slot = reinterpret_cast<T*>(tw + gtw<T>(MX)) + gslot(MX) * g;
    const uint32_t sl = blockIdx.x, sn = a.first + sl;
    gload_twiddles<T, MX, NT>(tw, a.twt, tid);
    const C* w = a.work + (size_t)sl * a.my * NCX;
    const int sx = (int)a.out.x / 2, sy = (int)a.out.y / 2;
    const int padx = MX - (int)a.out.x, pady = (int)a.my - (int)a.out.y;
    T best = -(T)__builtin_huge_val();
    uint32_t bi = 0xffffffffu;
    for (int q = tid; q < (int)a.out.y / 2; q += NT) {
        const C* row = w + (size_t)(2 * q <= sy ? 2 * q : 2 * q + pady) * NCX;
        const T v = row[0].im;
        const uint32_t i = *reinterpret_cast<const uint32_t*>(&row[NCX - 1].im);
        if (v > best || (v == best && i < bi)) best = v, bi = i;
    }
    __shared__ T sv[NT / kWave];
    __shared__ uint32_t si[NT / kWave];
    __shared__ T nbv[81];
    __shared__ double cf[6];
    block_argmax<T, NT>(best, bi, sv, si);
    const size2 cross{a.out.x - 1, a.out.y - 1};
    const size2 mp = shift_pos(POLICY_FFT, bi, cross);
    const int fit = a.fit, rad = (fit - 1) / 2, kk = fit * fit;
    // neighbourhood row j: its row pair again, the row kept in slot j
    static_assert(NT / L >= 9, "one lane group per neighbourhood row");
    __syncthreads();  // twiddles
    if (g < fit) {
        const size2 c = clamp_pos((int)mp.x, (int)mp.y - rad + g, cross);
        const int ry = (int)((c.y + (a.out.y / 2 + 1)) % a.out.y);
        C x[R];
        load_row_pair<T, MX>(x, w, ry >> 1, sy, pady, lane);
        gfft_inv<T, MX>(x, lane, slot, tw);
#pragma unroll
        for (int n1 = 0; n1 < R; ++n1) {
            const T even = x[n1].re, odd = x[n1].im;
            slot[gtime(MX, n1, lane)] = ry & 1 ? odd : even;
        }
    }
    __syncthreads();
    for (int t = tid; t < kk; t += NT) {
        const int i = t % fit, j = t / fit;
        const size2 c = clamp_pos((int)mp.x - rad + i, (int)mp.y - rad + j, cross);
        const int rx = (int)((c.x + (a.out.x / 2 + 1)) % a.out.x);
        const T v = (reinterpret_cast<const T*>(tw + gtw<T>(MX)) + gslot(MX) * j)[rx <= sx ? rx : rx + padx];
        nbv[t] = v;
        if (a.neigh) a.neigh[(size_t)sn * kk + t] = v;
    }
    __syncthreads();
    if (tid < 6) cf[tid] = fit_coef<T>(a.lsq + tid * kk, nbv, kk);
    __syncthreads();
    if (tid == 0) {
        if (a.maxes) {
            a.maxes[sn].data = best;
            a.maxes[sn].index = bi;
        }
        double px, py, ox, oy;
        fit_peak(cf, px, py);
        finalize_offset(bi, cross, POLICY_FFT, fit, px, py, ox, oy);
        if (a.offsets) {
            a.offsets[2 * (size_t)sn] = ox;
            a.offsets[2 * (size_t)sn + 1] = oy;
        }
        if (a.coefs)
            for (int c = 0; c < 6; ++c) a.coefs[6 * (size_t)sn + c] = cf[c];
    }
}

// ---------------------------------------------------------------- launchers
namespace {

// THIRDS: also the lengths 192 and 384 (the reference's own transforms are powers of two).
template <class T, int N, bool THIRDS, class F>
void dispatch_n(uint32_t n, F&& f) {
    if constexpr (N <= 512) {
        if (n == (uint32_t)N) return f(std::integral_constant<int, N>{});
        if constexpr (THIRDS && (N == 128 || (N == 256 && sizeof(T) == 4)))
            if (n == (uint32_t)(N / 2 * 3)) return f(std::integral_constant<int, N / 2 * 3>{});
        return dispatch_n<T, N * 2, THIRDS>(n, std::forward<F>(f));
    } else {
        throw unsupported_error("FFT policy: transform side " + std::to_string(n) + " is beyond 512");
    }
}

template <class K>
void set_lds(K kern, size_t bytes) {
    EMIDA_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

template <class T, class IN, class SUM, bool FP, bool HZ>
void run_rows(const fftg_args<T, IN, SUM>& a, hipStream_t st) {
    dispatch_n<T, 4, HZ>(a.mx, [&](auto mc) {
        constexpr int MX = decltype(mc)::value, NG = kGNT / glanes(MX);
        auto k = fftg_rows_kernel<T, IN, SUM, MX, FP, HZ>;
        static const bool once = (set_lds(k, glds<T>(MX)), true);
        (void)once;
        // enough workgroups for every CU to hold a few, at most one row pair per lane group
        const uint32_t most = div_up((a.in_rows + 1) / 2, (uint32_t)NG);
        const uint32_t splits = std::max(1u, std::min(most, 1024u / std::max(1u, a.total)));
        k<<<dim3(a.total, splits), kGNT, glds<T>(MX), st>>>(a);
        EMIDA_LAUNCHED("fftg_rows_kernel");
    });
}

template <class T, int MODE>
void run_cols(fftg_args<T, T, T> a, hipStream_t st) {
    a.npat = a.first % a.nb == 0 && a.total % a.nb == 0 ? a.total / a.nb : 0;
    dispatch_n<T, 4, gcols_hz(MODE)>(a.my, [&](auto mc) {
        constexpr int MY = decltype(mc)::value;
        auto k = fftg_cols_kernel<T, MY, MODE>;
        static const bool once = (set_lds(k, glds<T>(MY)), true);
        (void)once;
        const uint32_t blocks = div_up(a.mx / 2 + 1, (uint32_t)(kGNT / glanes(MY))) * a.total;
        k<<<blocks, kGNT, glds<T>(MY), st>>>(a, blocks);
        EMIDA_LAUNCHED("fftg_cols_kernel");
    });
}

template <class T, bool PEAK>
void run_rows_inv(const fftg_args<T, T, T>& a, hipStream_t st) {
    dispatch_n<T, 4, true>(a.mx, [&](auto mc) {
        constexpr int MX = decltype(mc)::value;
        auto k = fftg_rows_inv_kernel<T, MX, PEAK>;
        static const bool once = (set_lds(k, glds<T>(MX)), true);
        (void)once;
        k<<<dim3(a.total, div_up(a.out.y / 2, (uint32_t)(kGNT / glanes(MX)))), kGNT, glds<T>(MX), st>>>(a);
        EMIDA_LAUNCHED("fftg_rows_inv_kernel");
        if constexpr (PEAK) {
            auto kp = fftg_peak_kernel<T, MX>;
            static const bool oncep = (set_lds(kp, gpeak_lds<T>(MX)), true);
            (void)oncep;
            kp<<<a.total, gpeak_nt(MX), gpeak_lds<T>(MX), st>>>(a);
            EMIDA_LAUNCHED("fftg_peak_kernel");
        }
    });
}

template <class T, class IN, class SUM>
fftg_args<T, T, T> as_t(const fftg_args<T, IN, SUM>& a) {
    fftg_args<T, T, T> b{};
    b.side = a.side;
    b.mx = a.mx;
    b.my = a.my;
    b.nb = a.nb;
    b.first = a.first;
    b.total = a.total;
    b.work = a.work;
    b.spectra = a.spectra;
    b.spectra_out = a.spectra_out;
    b.scale = a.scale;
    b.out = a.out;
    b.corr = a.corr;
    b.twt = a.twt;
    b.fit = a.fit;
    b.lsq = a.lsq;
    b.maxes = a.maxes;
    b.neigh = a.neigh;
    b.offsets = a.offsets;
    b.coefs = a.coefs;
    return b;
}

constexpr size_t kFftgWorkCap = (size_t)1 << 30;  // work buffer of one launch chunk

}  // namespace

uint32_t fftg_padded(bool is_double, uint32_t side) {
    const uint32_t m = fft_padded(side);
    return (m == 256 || (m == 512 && !is_double)) && 2 * side <= m / 4 * 3 ? m / 4 * 3 : m;
}

bool fftg_needed(bool is_double, size2 side) {
    if (side.x != side.y) return true;
    const uint32_t m = fft_padded(side.x);
    return m > 256 || (m > 128 && is_double);
}

size_t fftg_spectrum_bytes(bool is_double, size2 side) {
    return (size_t)(fftg_padded(is_double, side.x) / 2 + 1) * fftg_padded(is_double, side.y) * (is_double ? 16 : 8);
}

size_t fftg_slice_work_bytes(bool is_double, size2 side) { return fftg_spectrum_bytes(is_double, side); }

size_t fftg_chunk(bool is_double, size2 side, uint32_t total) {
    const size_t c = std::max<size_t>(1, kFftgWorkCap / fftg_slice_work_bytes(is_double, side));
    return std::min<size_t>(c, total);
}

size_t fftg_work_bytes(bool is_double, size2 side, uint32_t total) {
    return fftg_chunk(is_double, side, total) * fftg_slice_work_bytes(is_double, side);
}

// Reference spectra ([roi][kx][ky], 2 s.x s.y / (Mx My) times the true spectrum) from
// the reference pattern; work holds fftg_work_bytes(.., nb) bytes.
template <class T, class IN, class S>
void launch_fftg_ref(const IN* pics, const S* sums, const T* hx, const T* hy, const size2* begins, size2 src,
                     size2 side, uint32_t nb, cplx<T>* spectra, void* work, hipStream_t st) {
    if (nb == 0) return;
    fftg_args<T, IN, S> a{};
    a.twt = fft_twiddles<T>();
    a.pics = pics;
    a.sums = sums;
    a.hx = hx;
    a.hy = hy;
    a.begins = begins;
    a.src = src;
    a.in_rows = side.y;
    a.in_cols = side.x;
    a.side = side;
    a.mx = fftg_padded(sizeof(T) == 8, side.x);
    a.my = fftg_padded(sizeof(T) == 8, side.y);
    a.nb = nb;
    a.first = 0;
    a.total = nb;
    a.work = (cplx<T>*)work;
    a.spectra_out = spectra;
    // the row and column stages double it; s.x s.y / (Mx My) is exact for power-of-two lengths,
    // rounded once for 192 and 384
    a.scale = (T)((double)side.x * side.y / ((double)a.mx * a.my));
    const size_t chunk = fftg_chunk(sizeof(T) == 8, side, nb);
    for (uint32_t f = 0; f < nb; f += (uint32_t)chunk) {
        a.first = f;
        a.total = (uint32_t)std::min<size_t>(chunk, nb - f);
        run_rows<T, IN, S, true, true>(a, st);
        run_cols<T, COLS_SPECTRUM>(as_t(a), st);
    }
}

// Pipeline of `total` slices, from the patterns to the offsets.
template <class T, class IN, class S>
void launch_fftg_pipe(const IN* pics, const S* sums, const T* hx, const T* hy, const size2* begins, size2 src,
                      size2 side, uint32_t nb, uint32_t total, const cplx<T>* spectra, int fit, data_index<T>* maxes,
                      T* neigh, double* offsets, double* coefs, void* work, hipStream_t st) {
    if (total == 0) return;
    fftg_args<T, IN, S> a{};
    a.twt = fft_twiddles<T>();
    a.pics = pics;
    a.sums = sums;
    a.hx = hx;
    a.hy = hy;
    a.begins = begins;
    a.src = src;
    a.in_rows = side.y;
    a.in_cols = side.x;
    a.side = side;
    a.mx = fftg_padded(sizeof(T) == 8, side.x);
    a.my = fftg_padded(sizeof(T) == 8, side.y);
    a.nb = nb;
    a.work = (cplx<T>*)work;
    a.spectra = spectra;
    a.out = size2{2 * side.x, 2 * side.y};
    a.fit = fit;
    a.lsq = lstsq_device_table() + lstsq_offset(fit);
    a.maxes = maxes;
    a.neigh = neigh;
    a.offsets = offsets;
    a.coefs = coefs;
    const size_t chunk = fftg_chunk(sizeof(T) == 8, side, total);
    for (uint32_t f = 0; f < total; f += (uint32_t)chunk) {
        a.first = f;
        a.total = (uint32_t)std::min<size_t>(chunk, total - f);
        run_rows<T, IN, S, true, true>(a, st);
        run_cols<T, COLS_PIPE>(as_t(a), st);
        run_rows_inv<T, true>(as_t(a), st);
    }
}

// Prepared s.x x s.y slices -> (2s.x) x (2s.y) circular correlation buffers
// (cross_corr_fft seam); spectra: nb spectra; work: chunk slices of half spectra.
template <class T>
void launch_fftg_corr_prepared(const T* pics, const T* ref, T* res, size2 side, uint32_t nb, uint32_t batch,
                               cplx<T>* spectra, void* work, size_t chunk, hipStream_t st) {
    fftg_args<T, T, T> a{};
    a.twt = fft_twiddles<T>();
    a.prepared = ref;
    a.pitch = side.x;
    a.slice_elems = side.area();
    a.in_rows = side.y;
    a.in_cols = side.x;
    a.side = side;
    a.mx = fftg_padded(sizeof(T) == 8, side.x);
    a.my = fftg_padded(sizeof(T) == 8, side.y);
    a.nb = nb;
    a.work = (cplx<T>*)work;
    a.spectra_out = spectra;
    a.scale = (T)((double)side.x * side.y / ((double)a.mx * a.my));
    a.out = size2{2 * side.x, 2 * side.y};
    for (uint32_t f = 0; f < nb; f += (uint32_t)chunk) {  // reference spectra, chunk by chunk
        a.first = f;
        a.total = (uint32_t)std::min<size_t>(chunk, nb - f);
        a.work = (cplx<T>*)work;
        run_rows<T, T, T, false, true>(a, st);
        fftg_args<T, T, T> b = a;
        b.work = (cplx<T>*)work;
        run_cols<T, COLS_SPECTRUM>(b, st);
    }
    // the spectrum kernel indexes ROIs from the slice index: shift it per chunk
    const uint32_t total = nb * batch;
    for (uint32_t f = 0; f < total; f += (uint32_t)chunk) {
        fftg_args<T, T, T> b = a;
        b.prepared = pics;
        b.first = f;
        b.total = (uint32_t)std::min<size_t>(chunk, total - f);
        b.spectra = spectra;
        b.spectra_out = nullptr;
        b.corr = res + (size_t)f * b.out.area();
        run_rows<T, T, T, false, true>(b, st);
        run_cols<T, COLS_PIPE>(b, st);
        run_rows_inv<T, false>(b, st);
    }
}

// The reference's own cross_corr_fft on its buffers (src/gpu_offset.hpp:303-316):
// R2C of every 2s.x x 2s.y real buffer of `pic`, product with the conjugate of the
// ROI's spectrum in `spectra` (R2C layout [ky][kx], kx <= s.x), unnormalised C2R into
// `res` (2s.x x 2s.y).  Both transform sides must be powers of two.
template <class T>
void launch_fftg_std_corr(const T* pic, const cplx<T>* spectra, T* res, size2 side, uint32_t nb, uint32_t total,
                          void* work, size_t chunk, hipStream_t st) {
    fftg_args<T, T, T> a{};
    a.twt = fft_twiddles<T>();
    a.prepared = pic;
    a.pitch = 2 * side.x;
    a.slice_elems = 4 * side.area();
    a.in_rows = 2 * side.y;
    a.in_cols = 2 * side.x;
    a.side = size2{side.x, side.y};
    a.mx = 2 * side.x;
    a.my = 2 * side.y;
    if (fft_padded(side.x) != a.mx || fft_padded(side.y) != a.my)
        throw unsupported_error("cross_corr_fft: 2s must be a power of two on both axes");
    a.nb = nb;
    a.spectra = spectra;
    a.scale = (T)0.5;  // undoes the doubling of the row and column stages (exact)
    a.out = size2{2 * side.x, 2 * side.y};
    a.work = (cplx<T>*)work;
    for (uint32_t f = 0; f < total; f += (uint32_t)chunk) {
        fftg_args<T, T, T> b = a;
        b.first = f;
        b.total = (uint32_t)std::min<size_t>(chunk, total - f);
        b.corr = res + (size_t)f * b.out.area();
        run_rows<T, T, T, false, false>(b, st);
        run_cols<T, COLS_STD_PIPE>(b, st);
        run_rows_inv<T, false>(b, st);
    }
}

// R2C of 2s.x x 2s.y real buffers (rows of `pitch` elements, 2s.y rows) into the R2C
// layout ([ky][kx], kx <= s.x) of `spectra`, unnormalised (cuFFT's R2C).
template <class T>
void launch_fftg_std_r2c(const T* pic, uint32_t pitch, cplx<T>* spectra, size2 side, uint32_t n, void* work,
                         size_t chunk, hipStream_t st) {
    fftg_args<T, T, T> a{};
    a.twt = fft_twiddles<T>();
    a.prepared = pic;
    a.pitch = pitch;
    a.slice_elems = pitch * 2 * side.y;
    a.in_rows = 2 * side.y;
    a.in_cols = 2 * side.x;
    a.side = side;
    a.mx = 2 * side.x;
    a.my = 2 * side.y;
    if (fft_padded(side.x) != a.mx || fft_padded(side.y) != a.my)
        throw unsupported_error("cross_corr_fft: 2s must be a power of two on both axes");
    a.nb = n;
    a.scale = (T)0.5;
    a.work = (cplx<T>*)work;
    a.spectra_out = spectra;
    for (uint32_t f = 0; f < n; f += (uint32_t)chunk) {
        fftg_args<T, T, T> b = a;
        b.first = f;
        b.total = (uint32_t)std::min<size_t>(chunk, n - f);
        run_rows<T, T, T, false, false>(b, st);
        run_cols<T, COLS_STD_SPECTRUM>(b, st);
    }
}

#define INST_FFTG(T, IN, S)                                                                                     \
    template void launch_fftg_ref<T, IN, S>(const IN*, const S*, const T*, const T*, const size2*, size2, size2, \
                                            uint32_t, cplx<T>*, void*, hipStream_t);                            \
    template void launch_fftg_pipe<T, IN, S>(const IN*, const S*, const T*, const T*, const size2*, size2, size2,\
                                             uint32_t, uint32_t, const cplx<T>*, int, data_index<T>*, T*, double*, \
                                             double*, void*, hipStream_t);
INST_FFTG(float, uint16_t, uint32_t)
INST_FFTG(double, uint16_t, uint32_t)
INST_FFTG(float, float, float)
INST_FFTG(double, double, double)
INST_FFTG(float, double, double)
INST_FFTG(double, float, float)

template void launch_fftg_corr_prepared<float>(const float*, const float*, float*, size2, uint32_t, uint32_t,
                                               cplx<float>*, void*, size_t, hipStream_t);
template void launch_fftg_corr_prepared<double>(const double*, const double*, double*, size2, uint32_t, uint32_t,
                                                cplx<double>*, void*, size_t, hipStream_t);
template void launch_fftg_std_corr<float>(const float*, const cplx<float>*, float*, size2, uint32_t, uint32_t, void*,
                                          size_t, hipStream_t);
template void launch_fftg_std_corr<double>(const double*, const cplx<double>*, double*, size2, uint32_t, uint32_t,
                                           void*, size_t, hipStream_t);
template void launch_fftg_std_r2c<float>(const float*, uint32_t, cplx<float>*, size2, uint32_t, void*, size_t,
                                         hipStream_t);
template void launch_fftg_std_r2c<double>(const double*, uint32_t, cplx<double>*, size2, uint32_t, void*, size_t,
                                          hipStream_t);

}  // namespace emida_amd
