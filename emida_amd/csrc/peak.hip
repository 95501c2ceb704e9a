// Arg-max, neighbourhood gather, least-squares subpixel peak and finalize.
//
// Reference: src/maxarg.cu:119-187 (arg-max per slice), src/extract_neighbors.cu:13-49
// (F x F gather with position policy and clamp), src/subpixel_max.hpp:14-97 and
// src/subpixel_max.cpp:5-58 (coefficients = (A^T A)^-1 A^T * neighbourhood, peak of
// the quadratic), src/gpu_offset.hpp:280-301 (offset formula).  The reference fits
// on the CPU; here one workgroup per slice does all four steps.  The fit runs in
// double without contraction in the reference's order, so it matches the CPU
// result bit for bit.
#include <mutex>
#include <type_traits>
#include <vector>

#include "kernels.hpp"

namespace emida_amd {

// --------------------------------------------------------------- least-squares tables
// (A^T A)^-1 A^T for f(x,y) = a + bx + cy + dx^2 + exy + fy^2 on an s x s grid,
// by exact rational Gauss-Jordan elimination; every entry is rounded once.
namespace {
struct rational {
    __int128 n, d;
};
__int128 gcd_i128(__int128 a, __int128 b) {
    if (a < 0) a = -a;
    if (b < 0) b = -b;
    while (b != 0) {
        __int128 t = a % b;
        a = b;
        b = t;
    }
    return a;
}
rational make_r(__int128 n, __int128 d) {
    if (d < 0) {
        n = -n;
        d = -d;
    }
    __int128 g = gcd_i128(n, d);
    if (g == 0) g = 1;
    return {n / g, d / g};
}
}  // namespace

void lstsq_host(int s, double* out) {
    const int m = s * s;
    std::vector<std::vector<rational>> g(6, std::vector<rational>(6 + m));
    auto basis = [s](int k, int i) -> long long {
        const long long x = k % s, y = k / s;
        const long long v[6] = {1, x, y, x * x, x * y, y * y};
        return v[i];
    };
    for (int i = 0; i < 6; ++i) {
        for (int j = 0; j < 6; ++j) {
            long long acc = 0;
            for (int k = 0; k < m; ++k) acc += basis(k, i) * basis(k, j);
            g[i][j] = make_r(acc, 1);
        }
        for (int k = 0; k < m; ++k) g[i][6 + k] = make_r(basis(k, i), 1);
    }
    for (int c = 0; c < 6; ++c) {
        int piv = c;
        while (g[piv][c].n == 0) ++piv;
        std::swap(g[piv], g[c]);
        const rational p = g[c][c];
        for (auto& e : g[c]) e = make_r(e.n * p.d, e.d * p.n);
        for (int r = 0; r < 6; ++r) {
            if (r == c || g[r][c].n == 0) continue;
            const rational f = g[r][c];
            for (int k = 0; k < 6 + m; ++k) {
                const rational t = make_r(f.n * g[c][k].n, f.d * g[c][k].d);
                g[r][k] = make_r(g[r][k].n * t.d - t.n * g[r][k].d, g[r][k].d * t.d);
            }
        }
    }
    for (int i = 0; i < 6; ++i)
        for (int k = 0; k < m; ++k) out[i * m + k] = (double)(long long)g[i][6 + k].n / (double)(long long)g[i][6 + k].d;
}

int lstsq_offset(int fit) {
    switch (fit) {
        case 3: return 0;
        case 5: return 6 * 9;
        case 7: return 6 * (9 + 25);
        case 9: return 6 * (9 + 25 + 49);
        default: throw arg_error("fitsize must be 3, 5, 7 or 9");
    }
}

// The tables live in a static device array (each GPU holds its own copy): filled once
// per device with a copy, never allocated, so entry points that must not allocate can
// use them; host code uses the address hipGetSymbolAddress gives, never the name.
static __device__ double g_lstsq[6 * (9 + 25 + 49 + 81)];

const double* lstsq_device_table() {
    static std::mutex mu;
    static std::vector<double*> per_device;
    int dev = 0;
    EMIDA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    if ((int)per_device.size() <= dev) per_device.resize(dev + 1, nullptr);
    if (!per_device[dev]) {
        std::vector<double> host(6 * (9 + 25 + 49 + 81));
        for (int s = 3; s <= 9; s += 2) lstsq_host(s, host.data() + lstsq_offset(s));
        EMIDA_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_lstsq), host.data(), host.size() * sizeof(double)));
        void* d = nullptr;
        EMIDA_HIP(hipGetSymbolAddress(&d, HIP_SYMBOL(g_lstsq)));
        if (!d) throw hip_error("hipGetSymbolAddress returned no address for the least-squares table");
        per_device[dev] = (double*)d;
    }
    return per_device[dev];
}

// --------------------------------------------------------------- device pieces
template <class T>
__device__ inline T lowest() {
    return -__builtin_huge_val();
}
template <>
__device__ inline float lowest<float>() {
    return -__builtin_huge_valf();
}

// --------------------------------------------------------------- fused peak kernel
template <class T, int NT>
__global__ __launch_bounds__(NT) void peak_kernel(const T* __restrict__ corr, size_t corr_len, uint32_t area,
                                                  size2 cross, int policy, int fit, const double* __restrict__ lsq,
                                                  data_index<T>* __restrict__ maxes, T* __restrict__ neigh,
                                                  double* __restrict__ offsets, double* __restrict__ coefs,
                                                  uint32_t total, const uint32_t* __restrict__ row_max) {
    __shared__ T sv[NT / kWave];
    __shared__ uint32_t si[NT / kWave];
    __shared__ T nbv[81];
    __shared__ double cf[6];
    const uint32_t sn = blockIdx.x;
    if (sn >= total) return;
    const T* d = corr + (size_t)sn * area;
    T best = lowest<T>();
    uint32_t bi = 0xffffffffu;
    if (row_max) {
        // the maximum from the row maxima; its lowest index lies in the first row whose
        // maximum equals it, so only that row is read
        const uint32_t* rm = row_max + (size_t)sn * cross.y;
        uint32_t mc = 0;
        for (uint32_t r = threadIdx.x; r < cross.y; r += NT) mc = max(mc, rm[r]);
        mc = ~block_min_u32<NT>(~mc, si);
        const T m = mc ? (T)screen_max_value(mc) : lowest<T>();
        if (m > lowest<T>()) {
            uint32_t row = 0xffffffffu, x = 0xffffffffu;
            for (uint32_t r = threadIdx.x; r < cross.y; r += NT)
                if (rm[r] == mc) row = min(row, r);
            row = block_min_u32<NT>(row, si);
            for (uint32_t i = threadIdx.x; i < cross.x; i += NT)
                if (d[(size_t)row * cross.x + i] == m) x = min(x, i);
            x = block_min_u32<NT>(x, si);
            if (x != 0xffffffffu) {
                best = m;
                bi = row * cross.x + x;
            }
        }
    }
    if (bi == 0xffffffffu) {
        for (uint32_t i = threadIdx.x; i < area; i += NT) {
            const T v = d[i];
            if (v > best) {
                best = v;
                bi = i;
            }
        }
        block_argmax<T, NT>(best, bi, sv, si);
    }
    const int k = fit * fit;
    const size2 mp = shift_pos(policy, bi, cross);
    const int r = (fit - 1) / 2;
    for (int t = threadIdx.x; t < k; t += NT) {
        const int i = t % fit, j = t / fit;
        const size2 c = clamp_pos((int)mp.x - r + i, (int)mp.y - r + j, cross);
        const size_t idx = pos_index(policy, sn, c, cross);
        const T v = idx < corr_len ? corr[idx] : (T)0;
        nbv[t] = v;
        if (neigh) neigh[(size_t)sn * k + t] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) cf[threadIdx.x] = fit_coef<T>(lsq + threadIdx.x * k, nbv, k);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (maxes) {
            maxes[sn].data = best;
            maxes[sn].index = bi;
        }
        double px, py, ox, oy;
        fit_peak(cf, px, py);
        finalize_offset(bi, cross, policy, fit, px, py, ox, oy);
        if (offsets) {
            offsets[2 * (size_t)sn] = ox;
            offsets[2 * (size_t)sn + 1] = oy;
        }
        if (coefs)
            for (int c = 0; c < 6; ++c) coefs[6 * (size_t)sn + c] = cf[c];
    }
}

template <class T, int NT>
__global__ __launch_bounds__(NT) void maxarg_kernel(const T* __restrict__ data, uint32_t area,
                                                    data_index<T>* __restrict__ out, uint32_t total) {
    __shared__ T sv[NT / kWave];
    __shared__ uint32_t si[NT / kWave];
    const uint32_t sn = blockIdx.x;
    if (sn >= total) return;
    const T* d = data + (size_t)sn * area;
    T best = lowest<T>();
    uint32_t bi = 0xffffffffu;
    for (uint32_t i = threadIdx.x; i < area; i += NT) {
        const T v = d[i];
        if (v > best) {
            best = v;
            bi = i;
        }
    }
    block_argmax<T, NT>(best, bi, sv, si);
    if (threadIdx.x == 0) {
        out[sn].data = best;
        out[sn].index = bi;
    }
}

template <class T>
__global__ void extract_kernel(const T* __restrict__ data, size_t data_len, const data_index<T>* __restrict__ max_i,
                               T* __restrict__ neigh, int s, size2 size, int policy, uint32_t total) {
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = s * s;
    const size_t sn = g / k;
    if (sn >= total) return;
    const int t = (int)(g % k), i = t % s, j = t / s, r = (s - 1) / 2;
    const size2 mp = shift_pos(policy, max_i[sn].index, size);
    const size2 c = clamp_pos((int)mp.x - r + i, (int)mp.y - r + j, size);
    const size_t idx = pos_index(policy, (uint32_t)sn, c, size);
    neigh[g] = idx < data_len ? data[idx] : (T)0;
}

template <class T>
__global__ void subpixel_kernel(const T* __restrict__ neigh, int s, uint32_t n, const double* __restrict__ lsq,
                                const data_index<T>* __restrict__ maxes, size2 cross, int policy,
                                double* __restrict__ offsets, double* __restrict__ coefs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = s * s;
    double c[6];
    for (int row = 0; row < 6; ++row) c[row] = fit_coef<T>(lsq + row * k, neigh + (size_t)i * k, k);
    double px, py;
    fit_peak(c, px, py);
    if (maxes) finalize_offset(maxes[i].index, cross, policy, s, px, py, px, py);
    if (offsets) {
        offsets[2 * (size_t)i] = px;
        offsets[2 * (size_t)i + 1] = py;
    }
    if (coefs)
        for (int row = 0; row < 6; ++row) coefs[6 * (size_t)i + row] = c[row];
}

// --------------------------------------------------------------- exact refinement
// Precision form: the matrix-core screen (float) locates the peak; the values the
// result depends on are then evaluated the way the brute kernels evaluate them (one
// accumulator, y outer, x inner, fma; src/cross_corr.cu:36-61) from the T-precision
// prepared slices, so they equal the brute policy's correlation values bit for bit.
//   candidates: every shift whose screen value is within tau of the screen maximum,
//     tau = tol_rel ||p|| ||r|| + tol_abs (||p|| + ||r||) bounding |screen - T value|
//     twice over (caller's bound), so the brute policy's arg-max is among them;
//   arg-max over the candidates' exact values, lowest index on ties;
//   the F x F neighbourhood (identity position policy and clamp, spilling into the next
//     slice as the brute path does) evaluated exactly; fit and finalize as peak_kernel.
// A slice with more than kRefineCap candidates (a flat, noise-dominated screen) or
// without a finite screen maximum is swept whole: every shift of the window is
// evaluated exactly, box by box, so its arg-max is the brute policy's as well.
constexpr int kRefineCap = 512;
// Candidates too wide for one box take boxes of 16 x 16, up to two for every round it would
// take to evaluate them one chain per lane (in float, whose products wait longer on one another,
// none for the first round), else the chains.  Boxes are counted first: evaluating six a round
// and then the chains all the same cost unrelated 128 x 128 patterns (160 slices, more than six
// boxes) 1.43 ms in float and 1.39 in double, where the chains take 0.57 and 0.70; a limit of
// four boxes 0.92 and 0.83.  Many candidates side by side want the boxes: 784 slices of 64 x 64
// in float, flat tops, 163 us, by chains 317.
template <class T>
constexpr int spread_boxes(int rounds) {
    return 2 * rounds - (sizeof(T) == 8 ? 0 : 2);
}
constexpr int kRowList = 256;  // screens of at most this many rows use the row maxima

template <class T>
__device__ inline T exact_corr(const T* __restrict__ p, const T* __restrict__ r, size2 s, int sx, int sy) {
    const int x_end = min((int)s.x - sx, (int)s.x), y_end = min((int)s.y - sy, (int)s.y);
    const int x0 = max(-sx, 0);
    T sum = 0;
    for (int y = max(-sy, 0); y < y_end; ++y) {
        const T* pr = p + (size_t)(y + sy) * s.x + sx;
        const T* qr = r + (size_t)y * s.x;
        int x = x0;
        // the operands of 8 products are loaded before their 8 dependent fmas, so one
        // memory latency is paid per 8 terms; the summation order is unchanged
        for (; x + 8 <= x_end; x += 8) {
            T u[8], v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                u[i] = pr[x + i];
                v[i] = qr[x + i];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) sum = fma(u[i], v[i], sum);
        }
        for (; x < x_end; ++x) sum = fma(pr[x], qr[x], sum);
    }
    return sum;
}

// Exact value of buffer element `g` of the launch (slice g / area, shift of g % area).
template <class T>
__device__ inline T exact_at(size_t g, size_t corr_len, const T* p, const T* r, size2 s, size2 cross, uint32_t nb) {
    if (g >= corr_len) return T(0);
    const uint32_t area = cross.area();
    const uint32_t sn = (uint32_t)(g / area), pos = (uint32_t)(g % area);
    const int sx = (int)(pos % cross.x) - (int)(cross.x - 1) / 2;
    const int sy = (int)(pos / cross.x) - (int)(cross.y - 1) / 2;
    const size_t a = (size_t)s.x * s.y;
    return exact_corr<T>(p + (size_t)sn * a, r + (size_t)(sn % nb) * a, s, sx, sy);
}

// Orders a wave's LDS accesses.
__device__ __forceinline__ void box_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exact values of a box of up to kBoxRows x kBoxW shifts of one slice, by one wave on the
// matrix cores, in the brute order: v_mfma_f64_4x4x4 and v_mfma_f32_16x16x4 round like a chain
// of fused multiply-adds over ascending k that starts at the accumulator, so one accumulator
// per shift fed with the pattern columns in order, reference row after reference row, gives
// exact_corr's bits.  The rows of A are the 16 y-shifts, the columns of B the x-shifts
// (the Toeplitz matrix of the reference row); terms outside a shift's overlap multiply an
// exact zero (finite values).
//
// A reference row moves the 16 pattern rows by one.  They stay in registers (lane l holds
// columns l / 16 + 4 t of the row Y with Y mod 16 = l % 16); each step loads the one new row
// into the lanes of the one that left, and the accumulators, which belong to y-shifts, move
// to the next row of D instead.  Only the reference row passes through LDS (one row per
// buffer, zeros around it).  That leaves a wave its own LDS of 11 KB and 12 waves on a CU;
// pattern rows staged in LDS (one shift per lane, vector FMAs, waves waiting on LDS 77% of
// the time) took 5.5 ms for 12,800 slices of 128 x 128 in double where this takes 1.95 ms.
constexpr int kBoxRows = 16;
constexpr int kBoxW = 32;
constexpr int kRowBuf = 192;  // elements of a reference row buffer

template <class T>
struct box_frag;
template <>
struct box_frag<double> {
    using acc = double;
    static constexpr int NJ = 4, REGS = 1;
    static __device__ __forceinline__ void mac(acc& c, double a, double b) {
        c = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ double get(const acc& c, int) { return c; }
    // lane l holds D[4 ((l % 16) / 4) + l / 16][l % 4]
    static __device__ __forceinline__ int row(int lane, int) { return 4 * (lane % 16 / 4) + lane / 16; }
    static __device__ __forceinline__ int col(int lane) { return lane % 4; }
    // every row of D becomes the next one's (15 becomes 0's)
    static __device__ __forceinline__ void turn(acc& c, int lane) {
        const int m = (row(lane, 0) + 15) & 15;
        c = __shfl(c, 16 * (m & 3) + 4 * (m >> 2) + lane % 4);
    }
};
typedef float box_f4 __attribute__((ext_vector_type(4)));
template <>
struct box_frag<float> {
    using acc = box_f4;
    static constexpr int NJ = 16, REGS = 4;
    static __device__ __forceinline__ void mac(acc& c, float a, float b) {
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float get(const acc& c, int r) { return c[r]; }
    // lane l, register r holds D[4 (l / 16) + r][l % 16]
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane / 16) + r; }
    static __device__ __forceinline__ int col(int lane) { return lane % 16; }
    static __device__ __forceinline__ void turn(acc& c, int lane) {
        const float up = __shfl(c[3], (lane + 48) & 63);
        c = box_f4{up, c[0], c[1], c[2]};
    }
};

// Shifts [sx0, sx0 + NJ NF) x [sy0, sy0 + 16) over the reference rows [y0, y1); KS column
// steps of 4 cover the slice (S a multiple of 8, at most 4 KS).  out: [16][kBoxW].
template <class T, int KS, int NF>
__device__ __forceinline__ void box_sums(const T* __restrict__ p, const T* __restrict__ r, int S, int SY, int sx0,
                                         int sy0, int y0, int y1, T* rbuf, T* out) {
    using F = box_frag<T>;
    constexpr int NJ = F::NJ, SH = NJ / 4, SPAN = NJ * NF - 1, PER = kRowBuf / kWave;
    constexpr int GS = KS % 8 ? 4 : 8;  // steps per group, whose operands load together
    static_assert(4 * KS + SPAN <= kRowBuf, "reference row buffer");
    const int lane = threadIdx.x % kWave, i = lane % 16, k = lane / 16, j = F::col(lane);
    // groups of GS steps that hold terms of the box
    const int g0 = max(0, sx0) / (4 * GS), g1 = (min(S, S + sx0 + SPAN) + 4 * GS - 1) / (4 * GS);
    typename F::acc acc[NF];
#pragma unroll
    for (int n = 0; n < NF; ++n) acc[n] = typename F::acc{};
    T a[KS];
    {
        const int Yb = y0 + sy0, Y = Yb + ((i - Yb) & 15);
        const bool in = Y >= 0 && Y < SY;
        const T* src = p + (size_t)(in ? Y : 0) * S + k;
#pragma unroll
        for (int t = 0; t < KS; ++t) a[t] = in && 4 * t < S ? src[4 * t] : T(0);
    }
    // element e of the row buffer: reference column e - (SPAN + sx0)
    T next[PER];
    auto fetch = [&](int y) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int c = lane + kWave * q - (SPAN + sx0);
            const bool in = c >= 0 && c < S;
            const T v = r[(size_t)y * S + (in ? c : 0)];
            next[q] = in ? v : T(0);
        }
    };
    auto put = [&](int y) {
#pragma unroll
        for (int q = 0; q < PER; ++q) rbuf[(y & 1) * kRowBuf + lane + kWave * q] = next[q];
        box_sync();
    };
    if (y0 < y1) {
        fetch(y0);
        put(y0);
    }
    for (int y = y0; y < y1; ++y) {
        fetch(min(y + 1, y1 - 1));
        const T* rb = rbuf + (y & 1) * kRowBuf + k - j + SPAN;
        const int Yn = y + sy0 + 16;  // the row that takes the place of y + sy0
        const bool take = ((Yn - i) & 15) == 0, in = Yn >= 0 && Yn < SY;
        const T* src = p + (size_t)(in ? Yn : 0) * S + k;
#pragma unroll
        for (int g = 0; g < KS / GS; ++g) {
            if (g < g0 || g >= g1) continue;
            constexpr int LEAD = SH * (NF - 1);
            T b[GS + LEAD];
#pragma unroll
            for (int u = 0; u < GS + LEAD; ++u) b[u] = rb[4 * (GS * g + u - LEAD)];
#pragma unroll
            for (int tt = 0; tt < GS; ++tt)
#pragma unroll
                for (int n = 0; n < NF; ++n) F::mac(acc[n], a[GS * g + tt], b[tt + LEAD - SH * n]);
            if (take) {
#pragma unroll
                for (int tt = 0; tt < GS; ++tt) {
                    const int t = GS * g + tt;
                    a[t] = in && 4 * t < S ? src[4 * t] : T(0);
                }
            }
        }
        put(y + 1);
#pragma unroll
        for (int n = 0; n < NF; ++n) F::turn(acc[n], lane);
    }
#pragma unroll
    for (int n = 0; n < NF; ++n)
#pragma unroll
        for (int q = 0; q < F::REGS; ++q)
            out[((F::row(lane, q) - y1 - sy0) & 15) * kBoxW + NJ * n + j] = F::get(acc[n], q);
    box_sync();
}

// Exact values of positions [x0, x0 + bw) x [y0, y0 + bh) of the cross buffer (shift =
// position - (cross - 1) / 2) into out[row * kBoxW + column]; bw <= kBoxW, bh <= kBoxRows.
// All NT threads of the workgroup call it; with four waves each takes a quarter of the
// columns (rbuf: two row buffers per wave).
template <class T, int NT, int KS>
__device__ __forceinline__ void eval_box(const T* __restrict__ p, const T* __restrict__ r, size2 s, size2 cross,
                                         int x0, int y0, int bw, int bh, T* rbuf, T* out) {
    if (bw <= 0 || bh <= 0) return;
    constexpr int NJ = box_frag<T>::NJ, NW = NT / kWave;
    const int S = (int)s.x, SY = (int)s.y, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int sx0 = x0 - (int)(cross.x - 1) / 2, sy0 = y0 - (int)(cross.y - 1) / 2;
    const int ya = max(0, -(sy0 + bh - 1)), yb = max(ya, min(SY, SY - sy0));  // rows with terms of the box
    if constexpr (NW > 1) __syncthreads();  // out may still be read
    auto run = [&](auto nf) {
        constexpr int NF = decltype(nf)::value;
        const int x = NJ * NF * wv;
        if (x < bw)
            box_sums<T, KS, NF>(p, r, S, SY, sx0 + x, sy0, ya, yb, rbuf + 2 * kRowBuf * wv, out + x);
    };
    // the fewest fragments that hold the box's columns
    if constexpr (NJ * NW == 4) {
        if (bw <= 8) run(std::integral_constant<int, 2>{});
        else if (bw <= 12) run(std::integral_constant<int, 3>{});
        else if (bw <= 16) run(std::integral_constant<int, 4>{});
        else run(std::integral_constant<int, 8>{});
    } else if constexpr (NJ * NW == 16) {
        if (bw <= 16) run(std::integral_constant<int, 1>{});
        else run(std::integral_constant<int, 2>{});
    } else {
        run(std::integral_constant<int, 1>{});
    }
    if constexpr (NW > 1) __syncthreads();
}

// NT = 64: one wave per slice; 256: four.  KS column steps of 4 cover the slice width.
template <class T, int NT, int KS>
__global__ __launch_bounds__(NT, 3) void refine_kernel(const float* __restrict__ screen, size_t corr_len,
                                                    const T* __restrict__ p, const T* __restrict__ r, size2 s,
                                                    size2 cross, uint32_t nb, double tol_rel, double tol_abs,
                                                    int fit, const double* __restrict__ lsq,
                                                    data_index<T>* __restrict__ maxes, T* __restrict__ neigh,
                                                    double* __restrict__ offsets, double* __restrict__ coefs,
                                                    uint32_t total, const uint32_t* __restrict__ smax,
                                                    screen_lists lists) {
    __shared__ float svf[NT / kWave];
    __shared__ uint32_t si[NT / kWave];
    __shared__ double sd[NT / kWave];
    __shared__ T sv[NT / kWave];
    __shared__ uint32_t cand[kRefineCap];
    __shared__ uint32_t ncand, nrow, overflow;
    __shared__ uint16_t rlist[kRowList];  // rows of the screen that can hold candidates
    __shared__ uint8_t rcnt[kRowList];    // and how many they hold
    __shared__ T nbv[81];
    __shared__ double cf[6];
    __shared__ T rbuf[NT / kWave * 2 * kRowBuf];  // reference rows of eval_box
    __shared__ T boxv[kBoxRows * kBoxW];          // the box values it leaves
    if (blockIdx.x >= total) return;
    // the patterns of one ROI run back to back on one XCD (one reference slice in its L2)
    const uint32_t L = xcd_remap(blockIdx.x, total), npat = total / nb;
    const uint32_t sn = (L % npat) * nb + L / npat;
    const int tid = threadIdx.x;
    const uint32_t area = cross.area();
    const size_t a = (size_t)s.x * s.y;
    const float* sc = screen ? screen + (size_t)sn * area : nullptr;  // none with candidate lists
    const T* ps = p + (size_t)sn * a;
    const T* rs = r + (size_t)(sn % nb) * a;

    // screen maximum (NaN ignored) and its lowest index; 8 loads in flight per thread.
    // Given the maximum from the matrix-core kernel, the index is found by the
    // candidate pass below instead (one read of the screen instead of two).
    constexpr int U = 8;
    float m = -__builtin_huge_valf();
    uint32_t mi = 0xffffffffu;
    uint32_t mcode = 0;  // largest row-maximum code (0: no value)
    if (smax) {
        for (uint32_t r = tid; r < cross.y; r += NT) mcode = max(mcode, smax[(size_t)sn * cross.y + r]);
        mcode = ~block_min_u32<NT>(~mcode, si);
        if (mcode) m = screen_max_value(mcode);
    } else {
        for (uint32_t i0 = tid; i0 < area; i0 += NT * U) {
            float v[U];
#pragma unroll
            for (int k = 0; k < U; ++k) v[k] = i0 + k * NT < area ? sc[i0 + k * NT] : -__builtin_huge_valf();
#pragma unroll
            for (int k = 0; k < U; ++k)
                if (v[k] > m) {
                    m = v[k];
                    mi = i0 + k * NT;
                }
        }
        block_argmax<float, NT>(m, mi, svf, si);
    }

    // ||p||, ||r|| in double (given with the candidate lists)
    double tau;
    if (lists.cnt) {
        tau = refine_tau(lists, sn, sn % nb);
    } else {
    double pp = 0, rr = 0;
    for (size_t i0 = tid; i0 < a; i0 += NT * U) {
        double u[U], w[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            u[k] = i0 + k * NT < a ? (double)ps[i0 + k * NT] : 0.0;
            w[k] = i0 + k * NT < a ? (double)rs[i0 + k * NT] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            pp += u[k] * u[k];
            rr += w[k] * w[k];
        }
    }
    for (int off = kWave / 2; off > 0; off >>= 1) {
        pp += __shfl_xor(pp, off);
        rr += __shfl_xor(rr, off);
    }
    if (tid % kWave == 0) sd[tid / kWave] = pp;
    __syncthreads();
    pp = 0;
    for (int k = 0; k < NT / kWave; ++k) pp += sd[k];
    __syncthreads();
    if (tid % kWave == 0) sd[tid / kWave] = rr;
    __syncthreads();
    rr = 0;
    for (int k = 0; k < NT / kWave; ++k) rr += sd[k];
    const double np = sqrt(pp), nr = sqrt(rr);
    tau = tol_rel * np * nr + tol_abs * (np + nr);
    }

    // Slices that fit the vector L1 are touched while the candidates are found: the box reads
    // them a row ahead, which hides an L1 hit but not a read from HBM (16 x 128 in float, 784
    // slices: refinement 78 us, 54 touched; beyond these sizes it gains nothing or evicts).
    constexpr int LINE = 128 / (int)sizeof(T), LINES = 4 * kWave / NT;
    constexpr size_t kTouch = NT == kWave ? 8192 : 16384;  // bytes of a slice
    const bool touch = a * sizeof(T) <= kTouch;
    T warm[2 * LINES];
#pragma unroll
    for (int k = 0; k < LINES; ++k) {
        const size_t i = touch ? min((size_t)(tid + NT * k) * LINE, a - 1) : 0;
        warm[2 * k] = ps[i];
        warm[2 * k + 1] = rs[i];
    }

    // candidates.  Given the row maxima, only rows whose maximum reaches the threshold
    // (or equals the slice maximum) can hold one, and only those rows are read.
    if (tid == 0) ncand = nrow = overflow = 0;
    __syncthreads();
    const double thr = (double)m - tau;
    uint32_t mil = 0xffffffffu;  // lowest index holding m (given maximum)
    auto take = [&](uint32_t idx, float v) {
        if (idx < area && (double)v >= thr) {
            const uint32_t c = atomicAdd(&ncand, 1u);
            if (c < kRefineCap) cand[c] = idx;
        }
        if (smax && idx < area && v == m && idx < mil) mil = idx;
    };
    if (lists.cnt) {
        // the rows that can hold a candidate, then the positions they published, several loads
        // in flight; a row with more than kListCap of them, or more rows than the list holds,
        // make the slice sweep, which needs none
        for (uint32_t r = tid; r < cross.y; r += NT) {
            const uint32_t code = smax[(size_t)sn * cross.y + r], c = lists.cnt[(size_t)sn * cross.y + r];
            if (code && ((double)screen_max_value(code) >= thr || code == mcode)) {
                const uint32_t k = atomicAdd(&nrow, 1u);
                if (k < (uint32_t)kRowList) {
                    rlist[k] = r;
                    rcnt[k] = (uint8_t)min(c, (uint32_t)kListCap);
                }
                if (k >= (uint32_t)kRowList || c > (uint32_t)kListCap) overflow = 1;
            }
        }
        __syncthreads();
        const uint32_t n = overflow ? 0u : nrow * (uint32_t)kListCap;
        const cand_entry* ent = lists.ent + (size_t)sn * cross.y * kListCap;
        constexpr int V = 4;
        for (uint32_t e0 = tid; e0 < n; e0 += NT * V) {
            cand_entry en[V];
            uint32_t row[V];
            bool on[V];
#pragma unroll
            for (int q = 0; q < V; ++q) {
                const uint32_t e = min(e0 + NT * q, n - 1), k = e % kListCap;
                row[q] = rlist[e / kListCap];
                on[q] = e == e0 + NT * q && k < rcnt[e / kListCap];
                en[q] = ent[on[q] ? row[q] * kListCap + k : 0];
            }
#pragma unroll
            for (int q = 0; q < V; ++q)
                if (on[q]) take(row[q] * cross.x + en[q].x, en[q].v);
        }
    } else if (smax && cross.y <= (uint32_t)kRowList) {
        for (uint32_t r = tid; r < cross.y; r += NT) {
            const uint32_t code = smax[(size_t)sn * cross.y + r];
            if (code && ((double)screen_max_value(code) >= thr || code == mcode)) rlist[atomicAdd(&nrow, 1u)] = r;
        }
        __syncthreads();
        const uint32_t n = nrow * cross.x;
        for (uint32_t i0 = tid; i0 < n; i0 += NT * U) {
            uint32_t idx[U];
            float v[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const uint32_t e = i0 + k * NT;
                idx[k] = e < n ? (uint32_t)rlist[e / cross.x] * cross.x + e % cross.x : area;
                v[k] = e < n ? sc[idx[k]] : -__builtin_huge_valf();
            }
#pragma unroll
            for (int k = 0; k < U; ++k) take(idx[k], v[k]);
        }
    } else {
        for (uint32_t i0 = tid; i0 < area; i0 += NT * U) {
            float v[U];
#pragma unroll
            for (int k = 0; k < U; ++k) v[k] = i0 + k * NT < area ? sc[i0 + k * NT] : -__builtin_huge_valf();
#pragma unroll
            for (int k = 0; k < U; ++k) take(i0 + k * NT, v[k]);
        }
    }
    if (smax) mi = block_min_u32<NT>(mil, si);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2 * LINES; ++k) asm volatile("" ::"v"(warm[k]));  // (keeps the loads)
    const bool sweep = ncand > (uint32_t)kRefineCap || mi == 0xffffffffu || overflow;
    const uint32_t nc = sweep ? 0u : ncand;
    // exact values; arg-max with the lowest index on ties.  Candidates whose bounding
    // box fits one box evaluation take the staged path, others one chain each.
    // (in registers: with four LDS updates per candidate, 225 ties of a flat 8 x 8 slice took 28 of
    // the kernel's 41 us)
    uint32_t ux0 = 0xffffffffu, uy0 = ux0, ux1 = ux0, uy1 = ux0;
    for (uint32_t c = tid; c < nc; c += NT) {
        const uint32_t cx = cand[c] % cross.x, cy = cand[c] / cross.x;
        ux0 = min(ux0, cx), uy0 = min(uy0, cy), ux1 = min(ux1, ~cx), uy1 = min(uy1, ~cy);
    }
    const int bb[4] = {(int)block_min_u32<NT>(ux0, si), (int)block_min_u32<NT>(uy0, si),
                       (int)~block_min_u32<NT>(ux1, si), (int)~block_min_u32<NT>(uy1, si)};
    const int k = fit * fit, rad = (fit - 1) / 2;
    // One box when the candidates' box grown by the fit radius fits: it holds every candidate
    // and the in-window neighbourhood of any of them.  Else one box of the candidates; else
    // (spread candidates) boxes of 16 x 16 around the first one left where few hold them all,
    // one chain per lane where not; a swept slice takes the whole window in boxes.
    const int cbw = bb[2] - bb[0] + 1, cbh = bb[3] - bb[1] + 1;
    const int ex0 = max(0, bb[0] - rad), ey0 = max(0, bb[1] - rad);
    const int ebw = min((int)cross.x - 1, bb[2] + rad) - ex0 + 1, ebh = min((int)cross.y - 1, bb[3] + rad) - ey0 + 1;
    const bool merged = !sweep && ebh <= kBoxRows && ebw <= kBoxW;
    const bool boxed = merged || (!sweep && cbh <= kBoxRows && cbw <= kBoxW);
    T best = lowest<T>();
    uint32_t bi = 0xffffffffu;
    auto offer = [&](T v, uint32_t i) {
        if (v > best || (v == best && i < bi)) {
            best = v;
            bi = i;
        }
    };
    size2 mp{0, 0};
    int bx0 = 0, by0 = 0, bw = 0, bh = 0;
    constexpr uint32_t kTaken = 1u << 31;  // mark of a candidate whose box has been taken
    auto next_box = [&] {                  // of the lowest one left
        uint32_t first = kTaken;
        for (uint32_t c = tid; c < nc; c += NT) first = min(first, cand[c]);
        first = block_min_u32<NT>(first, si);
        bx0 = max(0, (int)(first % cross.x) - 8);
        by0 = (int)(first / cross.x);
        bw = min(16, (int)cross.x - bx0);
        bh = min(16, (int)cross.y - by0);
        return first < kTaken;
    };
    auto in_box = [&](uint32_t i, int& x, int& y) {
        x = (int)(i % cross.x) - bx0;
        y = (int)(i / cross.x) - by0;
        return x >= 0 && y >= 0 && x < bw && y < bh;
    };
    bool chains = !sweep && !boxed;
    if (chains) {
        int n = 0, x, y;
        const int most = spread_boxes<T>((int)div_up(nc, (uint32_t)NT));
        while ((chains = next_box()) && ++n <= most) {
            for (uint32_t c = tid; c < nc; c += NT)
                if (cand[c] < kTaken && in_box(cand[c], x, y)) cand[c] |= kTaken;
        }
        for (uint32_t c = tid; c < nc; c += NT) cand[c] &= ~kTaken;
    }
    enum { CANDIDATES, SWEEP, PEAK };
    for (int mode = sweep ? SWEEP : CANDIDATES;;) {
        if (mode == CANDIDATES) {
            if (boxed) {
                bx0 = merged ? ex0 : bb[0];
                by0 = merged ? ey0 : bb[1];
                bw = merged ? ebw : cbw;
                bh = merged ? ebh : cbh;
            } else if (!chains) {
                next_box();
            }
        } else if (mode == SWEEP) {
            bw = min(kBoxW, (int)cross.x - bx0);
            bh = min(kBoxRows, (int)cross.y - by0);
        } else {
            bx0 = max(0, (int)mp.x - rad);
            by0 = max(0, (int)mp.y - rad);
            bw = min((int)cross.x - 1, (int)mp.x + rad) - bx0 + 1;
            bh = min((int)cross.y - 1, (int)mp.y + rad) - by0 + 1;
        }
        if (mode == CANDIDATES && chains) {
            for (uint32_t c = tid; c < nc; c += NT)
                offer(exact_at<T>((size_t)sn * area + cand[c], corr_len, p, r, s, cross, nb), cand[c]);
        } else {
            eval_box<T, NT, KS>(ps, rs, s, cross, bx0, by0, bw, bh, rbuf, boxv);
        }
        if (mode == PEAK) break;
        if (mode == CANDIDATES) {
            if (!chains) {
                int left = 0, x, y;
                for (uint32_t c = tid; c < nc; c += NT) {
                    const uint32_t i = cand[c];
                    if (i >= kTaken) continue;
                    if (in_box(i, x, y)) {
                        offer(boxv[y * kBoxW + x], i);
                        cand[c] = kTaken;
                    } else {
                        ++left;
                    }
                }
                if (__syncthreads_or(left)) continue;
            }
        } else {
            for (int e = tid; e < bw * bh; e += NT) {
                const int x = e % bw, y = e / bw;
                offer(boxv[y * kBoxW + x], (uint32_t)(by0 + y) * cross.x + (uint32_t)(bx0 + x));
            }
            bx0 += kBoxW;
            if (bx0 >= (int)cross.x) {
                bx0 = 0;
                by0 += kBoxRows;
            }
            if (by0 < (int)cross.y) continue;
        }
        block_argmax<T, NT>(best, bi, sv, si);
        mp = shift_pos(POLICY_BRUTE, bi, cross);
        if (merged) break;
        mode = PEAK;
    }

    // neighbourhood, exact: the in-window part from the last box, positions the clamp puts
    // one past the window (spilling into the next row or slice) one chain each
    for (int t = tid; t < k; t += NT) {
        const int i = t % fit, j = t / fit;
        const size2 c = clamp_pos((int)mp.x - rad + i, (int)mp.y - rad + j, cross);
        const int x = (int)c.x - bx0, y = (int)c.y - by0;
        const T v = c.x < cross.x && c.y < cross.y && x >= 0 && y >= 0 && x < bw && y < bh
                        ? boxv[y * kBoxW + x]
                        : exact_at<T>(pos_index(POLICY_BRUTE, sn, c, cross), corr_len, p, r, s, cross, nb);
        nbv[t] = v;
        if (neigh) neigh[(size_t)sn * k + t] = v;
    }
    __syncthreads();
    if (tid < 6) cf[tid] = fit_coef<T>(lsq + tid * k, nbv, k);
    __syncthreads();
    if (tid == 0) {
        if (maxes) {
            maxes[sn].data = best;
            maxes[sn].index = bi;
        }
        double px, py, ox, oy;
        fit_peak(cf, px, py);
        finalize_offset(bi, cross, POLICY_BRUTE, fit, px, py, ox, oy);
        if (offsets) {
            offsets[2 * (size_t)sn] = ox;
            offsets[2 * (size_t)sn + 1] = oy;
        }
        if (coefs)
            for (int c = 0; c < 6; ++c) coefs[6 * (size_t)sn + c] = cf[c];
    }
}

// --------------------------------------------------------------- launchers
constexpr int kPeakNT = 256;

template <class T>
void launch_peak(const T* corr, size_t corr_len, uint32_t area, size2 cross, int policy, int fit,
                 data_index<T>* maxes, T* neigh, double* offsets, double* coefs, uint32_t total, hipStream_t st,
                 const uint32_t* row_max) {
    const double* lsq = lstsq_device_table() + lstsq_offset(fit);
    if (total == 0) return;
    peak_kernel<T, kPeakNT><<<total, kPeakNT, 0, st>>>(corr, corr_len, area, cross, policy, fit, lsq, maxes, neigh,
                                                      offsets, coefs, total, row_max);
    EMIDA_LAUNCHED("peak_kernel");
}

template <class T>
void launch_maxarg(const T* data, uint32_t area, data_index<T>* out, uint32_t total, hipStream_t st) {
    if (total == 0) return;
    maxarg_kernel<T, kPeakNT><<<total, kPeakNT, 0, st>>>(data, area, out, total);
    EMIDA_LAUNCHED("maxarg_kernel");
}

template <class T>
void launch_extract(const T* data, size_t data_len, const data_index<T>* max_i, T* neigh, int s, size2 size,
                    int policy, uint32_t total, hipStream_t st) {
    const size_t n = (size_t)total * s * s;
    if (n == 0) return;
    extract_kernel<T><<<(unsigned)div_up(n, (size_t)256), 256, 0, st>>>(data, data_len, max_i, neigh, s, size,
                                                                       policy, total);
    EMIDA_LAUNCHED("extract_kernel");
}

template <class T>
void launch_subpixel(const T* neigh, int s, uint32_t n, const data_index<T>* maxes, size2 cross, int policy,
                     double* offsets, double* coefs, hipStream_t st) {
    const double* lsq = lstsq_device_table() + lstsq_offset(s);
    if (n == 0) return;
    subpixel_kernel<T><<<div_up(n, 64u), 64, 0, st>>>(neigh, s, n, lsq, maxes, cross, policy, offsets, coefs);
    EMIDA_LAUNCHED("subpixel_kernel");
}

constexpr uint32_t kRefineOneWave = 768;

template <class T>
void launch_refine(const float* screen, size_t corr_len, const T* p, const T* r, size2 s, size2 cross, uint32_t nb,
                   double tol_rel, double tol_abs, int fit, data_index<T>* maxes, T* neigh, double* offsets,
                   double* coefs, uint32_t total, hipStream_t st, const uint32_t* screen_max,
                   const screen_lists* lists) {
    if (total == 0) return;
    if (s.x > 2 * (uint32_t)kWave) throw arg_error("exact refinement needs slices at most 128 wide");
    if (lists && (!screen_max || !lists->cnt || !lists->ent || !lists->pn2 || !lists->rn2))
        throw arg_error("exact refinement: candidate lists need the row maxima, counts, entries and norms");
    if (!lists && !screen) throw arg_error("exact refinement: no screen");
    screen_lists none{};
    const double* lsq = lstsq_device_table() + lstsq_offset(fit);
    if (nb == 0 || total % nb) throw arg_error("exact refinement: slices must be whole sets of ROIs");
    if (s.x % 8) throw arg_error("exact refinement needs a slice width that is a multiple of 8");
    // One wave per slice; four, which split a box's columns and the chains of spread candidates,
    // where that leaves most SIMDs without a wave (a pass in double at 128 x 128 and 100, 400,
    // 1,000, 1,600, 6,400 slices: one wave 2.09, 2.12, 2.25, 2.40, 5.95 ms, four 2.04, 2.10,
    // 2.36, 2.69, 7.10 ms).
    auto launch = [&](auto ks) {
        auto go = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            refine_kernel<T, NT, decltype(ks)::value><<<total, NT, 0, st>>>(
                screen, corr_len, p, r, s, cross, nb, tol_rel, tol_abs, fit, lsq, maxes, neigh, offsets, coefs, total,
                screen_max, lists ? *lists : none);
        };
        if (total >= kRefineOneWave) go(std::integral_constant<int, kWave>{});
        else go(std::integral_constant<int, 4 * kWave>{});
    };
    if (s.x <= 16) launch(std::integral_constant<int, 4>{});
    else if (s.x <= 32) launch(std::integral_constant<int, 8>{});
    // (40 x 24 in double, 4,000 swept slices: 549 us with 16 steps, 436 with 12)
    else if (s.x <= 48) launch(std::integral_constant<int, 12>{});
    else if (s.x <= 64) launch(std::integral_constant<int, 16>{});
    else launch(std::integral_constant<int, 32>{});
    EMIDA_LAUNCHED("refine_kernel");
}
template void launch_refine<float>(const float*, size_t, const float*, const float*, size2, size2, uint32_t, double,
                                   double, int, data_index<float>*, float*, double*, double*, uint32_t,
                                   hipStream_t, const uint32_t*, const screen_lists*);
template void launch_refine<double>(const float*, size_t, const double*, const double*, size2, size2, uint32_t,
                                    double, double, int, data_index<double>*, double*, double*, double*, uint32_t,
                                    hipStream_t, const uint32_t*, const screen_lists*);

#define INST_PEAK(T)                                                                                          \
    template void launch_peak<T>(const T*, size_t, uint32_t, size2, int, int, data_index<T>*, T*, double*,     \
                                 double*, uint32_t, hipStream_t, const uint32_t*);                            \
    template void launch_maxarg<T>(const T*, uint32_t, data_index<T>*, uint32_t, hipStream_t);                \
    template void launch_extract<T>(const T*, size_t, const data_index<T>*, T*, int, size2, int, uint32_t,    \
                                    hipStream_t);                                                             \
    template void launch_subpixel<T>(const T*, int, uint32_t, const data_index<T>*, size2, int, double*,      \
                                     double*, hipStream_t);
INST_PEAK(float)
INST_PEAK(double)

}  // namespace emida_amd
