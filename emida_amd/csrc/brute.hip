// Definition-based ("brute") 2-D cross-correlation.
//
// Reference: src/cross_corr.cu:11-74.  For every shift (sx, sy) of the result
// (res index = shift + (res_size - 1) / 2) the sum over the overlap of
// pic[y + sy][x + sx] * ref[y][x] is accumulated in one register, y outer and x
// inner, as fused multiply-adds (the reference's nvcc build contracts
// `sum += a * b`), so double and float results are bit-identical to that order.
//
// Float and double run on the matrix cores (cross_corr_mm_kernel); slices of a few pixels and
// those of which eight reference rows and the pattern rows of a workgroup's shifts do not fit
// its LDS (square ones from 200 wide with a narrow window to 570 with a wide one in double, 460
// to 1,190 in float) take the thread-per-shift kernel: one workgroup per (slice, 4-row band of
// shifts, 64-column band of shifts), staged in LDS when both slices fit in 64 KiB.  int32 has
// no matrix instruction with its wrapping sums and keeps the vector kernels: a register-blocked
// one ("tiled") for slices up to 128 pixels wide, windows up to 256 wide and launches of at
// least 256 workgroups, one with eight x-shifts per thread sliding a register window over
// zero-padded rows ("x8") for other slices that fit in LDS, and the thread-per-shift one.
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"

namespace emida_amd {

template <class T>
__device__ inline T mac(T a, T b, T acc) {
    return fma(a, b, acc);
}
template <>
__device__ inline int32_t mac<int32_t>(int32_t a, int32_t b, int32_t acc) {
    return (int32_t)((uint32_t)acc + (uint32_t)a * (uint32_t)b);
}

constexpr int kBruteTX = 64, kBruteTY = 4;
constexpr size_t kBruteLds = 64 * 1024;

template <class T, bool LDS>
__global__ __launch_bounds__(kBruteTX* kBruteTY) void cross_corr_kernel(const T* __restrict__ pics,
                                                                        const T* __restrict__ ref,
                                                                        T* __restrict__ res, size2 size,
                                                                        size2 res_size, uint32_t ref_slices) {
    extern __shared__ unsigned char smem_raw[];
    const uint32_t sn = blockIdx.z;
    const T* p = pics + (size_t)sn * size.area();
    const T* q = ref + (size_t)(sn % ref_slices) * size.area();
    if constexpr (LDS) {
        T* sp = reinterpret_cast<T*>(smem_raw);
        T* sq = sp + size.area();
        for (uint32_t i = threadIdx.y * kBruteTX + threadIdx.x; i < size.area(); i += kBruteTX * kBruteTY) {
            sp[i] = p[i];
            sq[i] = q[i];
        }
        __syncthreads();
        p = sp;
        q = sq;
    }
    const uint32_t rx = blockIdx.x * kBruteTX + threadIdx.x;
    const uint32_t ry = blockIdx.y * kBruteTY + threadIdx.y;
    if (rx >= res_size.x || ry >= res_size.y) return;
    const int sx = (int)rx - (int)((res_size.x - 1) / 2);
    const int sy = (int)ry - (int)((res_size.y - 1) / 2);
    const int x_end = min((int)size.x - sx, (int)size.x);
    const int y_end = min((int)size.y - sy, (int)size.y);
    const int x0 = max(-sx, 0);
    T sum = 0;
    for (int y = max(-sy, 0); y < y_end; ++y) {
        const T* pr = p + (size_t)(y + sy) * size.x + sx;
        const T* qr = q + (size_t)y * size.x;
        for (int x = x0; x < x_end; ++x) sum = mac<T>(pr[x], qr[x], sum);
    }
    res[(size_t)sn * res_size.area() + (size_t)ry * res_size.x + rx] = sum;
}

// The same sums, NX consecutive x-shifts per thread, for slices staged in LDS: an
// NX-value window slides along the pattern row (one new pattern value and one
// reference value per column feed NX fmas).  Each thread walks the union of its
// shifts' overlaps, rounded up to whole blocks of NX columns, so the window moves in
// registers by compile-time index within a block; the pattern rows are stored with
// NX - 1 zeros before and 2 NX - 2 after them and the reference rows with NX zeros
// after them, so a term outside a shift's own overlap multiplies an exact zero and
// leaves its sum unchanged (finite values), and every sum still sees its own terms
// y outer, x inner.  Indices: the window reads pattern column x + sx0 + t, t < NX,
// for x in [xu0, xu0 + NX * blocks) with xu0 + NX * blocks <= xu1 + NX - 1, which
// stays in [-(NX - 1), S + 2 NX - 2); reference columns stay below S + NX - 1.
constexpr int kXN = 8;  // x-shifts per thread (4: 0.146 ms, 16: 0.167 ms at 32 x 32 slices, 63 x 63 windows; 8: 0.130 ms)
constexpr int kXNTX = 64 / kXN, kXNTY = 256 / kXNTX;
constexpr int kXNPadL = kXN - 1, kXNPadR = 2 * kXN - 2;

template <class T>
__host__ __device__ inline size_t xn_lds_elems(size2 size) {
    return (size_t)size.y * (size.x + kXNPadL + kXNPadR) + (size_t)size.y * (size.x + kXN);
}

template <class T>
__global__ __launch_bounds__(kXNTX* kXNTY) void cross_corr_x8_kernel(const T* __restrict__ pics,
                                                                    const T* __restrict__ ref,
                                                                    T* __restrict__ res, size2 size,
                                                                    size2 res_size, uint32_t ref_slices) {
    constexpr int NX = kXN;
    extern __shared__ unsigned char smem_raw[];
    const uint32_t sn = blockIdx.z;
    const int S = (int)size.x, SY = (int)size.y, W = S + kXNPadL + kXNPadR, SQ = S + NX;
    T* sp = reinterpret_cast<T*>(smem_raw);  // SY rows of W: zeros, pattern row, zeros
    T* sq = sp + (size_t)SY * W;             // SY rows of SQ: reference row, zeros
    const T* p = pics + (size_t)sn * size.area();
    const T* q = ref + (size_t)(sn % ref_slices) * size.area();
    const int tid = threadIdx.y * kXNTX + threadIdx.x;
    for (int i = tid; i < SY * W; i += kXNTX * kXNTY) {
        const int y = i / W, c = i % W - kXNPadL;
        sp[i] = (c >= 0 && c < S) ? p[(size_t)y * S + c] : T(0);
    }
    for (int i = tid; i < SY * SQ; i += kXNTX * kXNTY) {
        const int y = i / SQ, c = i % SQ;
        sq[i] = c < S ? q[(size_t)y * S + c] : T(0);
    }
    __syncthreads();
    const uint32_t rx0 = (blockIdx.x * kXNTX + threadIdx.x) * NX;
    const uint32_t ry = blockIdx.y * kXNTY + threadIdx.y;
    if (rx0 >= res_size.x || ry >= res_size.y) return;
    const int nsh = min(NX, (int)(res_size.x - rx0));  // shifts of this thread in the window
    const int sx0 = (int)rx0 - (int)((res_size.x - 1) / 2);
    const int sy = (int)ry - (int)((res_size.y - 1) / 2);
    const int xu0 = max(0, -(sx0 + nsh - 1)), xu1 = min(S, S - sx0);  // union of the overlaps
    T acc[NX];
#pragma unroll
    for (int t = 0; t < NX; ++t) acc[t] = T(0);
    if (xu0 < xu1) {
        const int blocks = (xu1 - xu0 + NX - 1) / NX;
        for (int y = max(-sy, 0); y < min(SY, SY - sy); ++y) {
            const T* pr = sp + (size_t)(y + sy) * W + kXNPadL + sx0 + xu0;  // pr[j + t]: column xu0 + j + sx0 + t
            const T* qr = sq + (size_t)y * SQ + xu0;
            T w[2 * NX - 1];
#pragma unroll
            for (int t = 0; t < NX - 1; ++t) w[t] = pr[t];
            for (int b = 0; b < blocks; ++b, pr += NX, qr += NX) {
                T qv[NX];
#pragma unroll
                for (int u = 0; u < NX; ++u) {
                    w[NX - 1 + u] = pr[NX - 1 + u];
                    qv[u] = qr[u];
                }
#pragma unroll
                for (int u = 0; u < NX; ++u)
#pragma unroll
                    for (int t = 0; t < NX; ++t) acc[t] = mac<T>(w[u + t], qv[u], acc[t]);
#pragma unroll
                for (int t = 0; t < NX - 1; ++t) w[t] = w[NX + t];
            }
        }
    }
    T* o = res + (size_t)sn * res_size.area() + (size_t)ry * res_size.x + rx0;
#pragma unroll
    for (int t = 0; t < NX; ++t)
        if (t < nsh) o[t] = acc[t];
}

// ------------------------------------------------------------------ tiled kernel
// The same sums, register-blocked.  A workgroup takes 16 patterns of one ROI, a band
// of x-shifts (64 per wave) and a band of y-shifts (4 per wave); it walks the
// reference rows y and, per row, the pattern columns k in blocks of 8.  A thread
// holds 2 patterns x 8 consecutive x-shifts x 4 y-shifts of accumulators; per column
// k it reads 2 x 4 pattern values from LDS and slides an 8-wide window over the
// reference row, so each pattern value feeds 8 and each reference value 8 x 4
// multiply-adds.  The reference row is zero-padded in LDS and pattern rows are
// zero-padded to a multiple of 8, so the loop runs over the union of the thread's
// overlaps: a term outside a shift's overlap adds a product with an exact zero and
// leaves its sum unchanged (for finite values), and every sum still sees its own
// terms y outer, x inner, in the reference's order.
constexpr int kTiledP = 16;   // patterns per workgroup
constexpr int kTiledMI = 2;   // patterns per thread
constexpr int kTiledNI = 8;   // x-shifts per thread
constexpr int kTiledTT = 4;   // y-shifts per thread
constexpr int kTiledSXW = 64; // x-shifts per wave
constexpr size_t kTiledRingMax = 64 * 1024;

struct tiled_shape {
    int wx, wy;       // waves along x-shifts and y-shifts
    int rows;         // pattern rows per step (y-shifts per workgroup) = 4 wy
    int spad;         // slice width rounded up to 8
    int off;          // reference row offset in the padded LDS row
    int rlen;         // padded reference row length
    size_t lds;       // bytes: ring + reference row
};

template <class T>
inline bool tiled_plan(size2 size, size2 res, tiled_shape& t) {
    t.spad = (int)div_up(size.x, 8u) * 8;
    if (t.spad > 128 || res.x > 4u * kTiledSXW) return false;
    t.wx = (int)div_up(res.x, (uint32_t)kTiledSXW);
    t.wy = t.wx == 1 ? 4 : (t.wx == 2 ? 2 : 1);
    while (t.wy > 1 && (size_t)kTiledP * kTiledTT * t.wy * t.spad * sizeof(T) > kTiledRingMax) t.wy /= 2;
    t.rows = kTiledTT * t.wy;
    // a thread's window reads R[y][k - sx] for k in [k8 - 8, khi) and its x-shifts
    // sx in [-rx, 64 wx - rx); with off = 64 wx - rx + 16 every index k - sx + off lies
    // in [16, spad + rx + off)
    const int rx = (int)(res.x - 1) / 2;
    t.off = kTiledSXW * t.wx - rx + 16;
    t.rlen = t.spad + rx + t.off;
    t.lds = (size_t)kTiledP * t.rows * t.spad * sizeof(T) + (size_t)t.rlen * sizeof(T);
    return true;
}

template <class T>
struct pair_of {
    T v[2];
};

// Pattern ring: [rows][spad][16], column k of a row holding the 16 patterns' values in
// pattern order.  Staged with the pattern index fastest (consecutive threads write
// consecutive words); a lane reads its pattern pair of column k8 + j at a per-row base
// plus the compile-time offset 128 j bytes, so the inner loop needs no address
// arithmetic per read (the 8 pairs a wave reads are 128 contiguous bytes).
template <class T>
__global__ __launch_bounds__(256, 2) void cross_corr_tiled_kernel(const T* __restrict__ pics,
                                                                   const T* __restrict__ ref, T* __restrict__ res,
                                                                   size2 size, size2 res_size, uint32_t nb,
                                                                   uint32_t npat, tiled_shape sh, uint32_t n_wg) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* ring = reinterpret_cast<T*>(smem_raw);
    T* rrow = ring + (size_t)kTiledP * sh.rows * sh.spad;
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid % 64, wave = tid / 64;
    const int S = (int)size.x, SY = (int)size.y, SP = sh.spad, ROWS = sh.rows;
    const uint32_t n_syt = div_up(res_size.y, (uint32_t)ROWS);
    const uint32_t L = xcd_remap(blockIdx.x, n_wg);
    const uint32_t syt = L % n_syt, slab = L / n_syt;
    const uint32_t roi = slab % nb, p0 = (slab / nb) * kTiledP;
    const int rx = (int)(res_size.x - 1) / 2, ry = (int)(res_size.y - 1) / 2;
    const int sy0 = (int)syt * ROWS - ry;
    const size_t slice_elems = (size_t)size.x * size.y;
    const T* refs = ref + (size_t)roi * slice_elems;

    const int wx = (wave % sh.wx + (int)syt) % sh.wx, wy = wave / sh.wx;
    const int pg = lane % 8, sg = lane / 8;
    const int sxw0 = -rx + wx * kTiledSXW;          // first x-shift of the wave
    const int sxb = sxw0 + sg * kTiledNI;           // first x-shift of the thread
    const int syt0 = sy0 + wy * kTiledTT;           // first y-shift of the thread

    T acc[kTiledMI][kTiledNI][kTiledTT];
#pragma unroll
    for (int i = 0; i < kTiledMI; ++i)
#pragma unroll
        for (int n = 0; n < kTiledNI; ++n)
#pragma unroll
            for (int t = 0; t < kTiledTT; ++t) acc[i][n][t] = T(0);

    for (size_t e = tid; e * sizeof(T) < sh.lds; e += nt) ring[e] = T(0);
    __syncthreads();

    // pattern row Y into its ring slot; rows past the slice (read by the last
    // steps' y-shifts) are zeros, so the accumulation needs no per-row condition
    // (rows before it only ever map to slots still holding the initial zeros)
    auto stage_prow = [&](int Y) {
        if (Y < 0) return;
        T* dst = ring + (size_t)(Y % ROWS) * SP * kTiledP;
        if (Y >= SY) {
            for (int e = tid; e < kTiledP * SP; e += nt) dst[e] = T(0);
            return;
        }
        for (int e = tid; e < kTiledP * S; e += nt) {
            const int p = e % kTiledP, k = e / kTiledP;
            const uint32_t pp = p0 + p;
            const T v = pp < npat ? pics[((size_t)pp * nb + roi) * slice_elems + (size_t)Y * S + k] : T(0);
            dst[k * kTiledP + p] = v;
        }
    };
    auto stage_rrow = [&](int y) {
        for (int e = tid; e < S; e += nt) rrow[sh.off + e] = refs[(size_t)y * S + e];
    };

    // k range of the wave: union of the overlaps of its x-shifts, in blocks of 8
    const int klo = max(0, sxw0) & ~7;
    const int khi = min(SP, (min(S, S + sxw0 + kTiledSXW - 1) + 7) & ~7);

    const int y_lo = max(0, -(sy0 + ROWS - 1)), y_hi = min(SY, SY - sy0);
    for (int Y = y_lo + sy0; Y < y_lo + sy0 + ROWS - 1; ++Y) stage_prow(Y);
    for (int y = y_lo; y < y_hi; ++y) {
        stage_prow(y + sy0 + ROWS - 1);
        stage_rrow(y);
        __syncthreads();
        if (klo < khi) {
            // window values: of the block being accumulated, cur[j] = R[y][k8 + j - sxb],
            // and of the one before, prev[j] = R[y][k8 - 8 + j - sxb]; two register blocks
            // alternate in the two roles (no copies), two column blocks per iteration
            T wa[8], wb[8];
            const T* rp = rrow + sh.off - sxb;
#pragma unroll
            for (int j = 0; j < 8; ++j) wa[j] = rp[klo - 8 + j];
            // this lane's pattern pair in column klo of the rows of its 4 y-shifts
            const pair_of<T>* pr[kTiledTT];
#pragma unroll
            for (int t = 0; t < kTiledTT; ++t) {
                const int Y = y + syt0 + t;
                const int slot = (Y % ROWS + ROWS) % ROWS;
                pr[t] = reinterpret_cast<const pair_of<T>*>(ring + ((size_t)slot * SP + klo) * kTiledP) + pg;
            }
            // columns k8 .. k8 + 7: load the block into cur, accumulate
            auto block = [&](int k8, const T (&prev)[8], T (&cur)[8]) {
#pragma unroll
                for (int j = 0; j < 8; ++j) cur[j] = rp[k8 + j];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    pair_of<T> a[kTiledTT];
#pragma unroll
                    for (int t = 0; t < kTiledTT; ++t) a[t] = pr[t][j * (kTiledP / 2)];
#pragma unroll
                    for (int t = 0; t < kTiledTT; ++t) {
#pragma unroll
                        for (int n = 0; n < kTiledNI; ++n) {
                            const T b = (j - n >= 0) ? cur[(j - n) & 7] : prev[(8 + j - n) & 7];
#pragma unroll
                            for (int i = 0; i < kTiledMI; ++i) acc[i][n][t] = mac<T>(a[t].v[i], b, acc[i][n][t]);
                        }
                    }
                }
#pragma unroll
                for (int t = 0; t < kTiledTT; ++t) pr[t] += 8 * (kTiledP / 2);
            };
            int k8 = klo;
            for (; k8 + 8 < khi; k8 += 16) {
                block(k8, wa, wb);
                block(k8 + 8, wb, wa);
            }
            if (k8 < khi) block(k8, wa, wb);
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < kTiledTT; ++t) {
        const int sy = syt0 + t;
        if (sy + ry >= (int)res_size.y) continue;
#pragma unroll
        for (int i = 0; i < kTiledMI; ++i) {
            const uint32_t p = p0 + 2 * pg + i;
            if (p >= npat) continue;
            T* out = res + (((size_t)p * nb + roi) * res_size.y + (sy + ry)) * res_size.x;
#pragma unroll
            for (int n = 0; n < kTiledNI; ++n) {
                const int sx = sxb + n;
                if (sx + rx < (int)res_size.x) out[sx + rx] = acc[i][n][t];
            }
        }
    }
}

// ------------------------------------------------------------------ matrix-core kernel
// The same sums for float and double on the matrix cores, bit for bit: on gfx950
// v_mfma_f64_4x4x4 and v_mfma_f32_16x16x4 round like a chain of fused multiply-adds over
// k = 0..3 that starts at the accumulator (subnormals kept), so one accumulator per shift
// fed with ascending pattern columns of ascending rows sees its terms y outer, x inner.
//
// For one slice and reference row y, C[sy][sx] += sum_c P[y + sy][c] * R[y][c - sx]: the
// rows of A are 16 consecutive y-shifts (pattern rows), the columns of B are x-shifts (a
// Toeplitz matrix of the reference row), k runs over 4 pattern columns.  No batch of
// patterns is needed, so a single pattern fills the matrix cores as a batch does.
//
// A wave holds tiles of 16 y-shifts x NJ TB x-shifts, TB fragments of NJ x-shifts each
// (double: NJ = 4, the four 4 x 4 blocks of the instruction being 4 groups of y-shifts;
// float: NJ = 16).  Fragment n at column step t reads G(t - n NJ / 4), with
// G(u)[k][j] = R[base + 4 u + k - j]: a step loads one A fragment and one G and keeps the
// earlier G's in registers.  Steps in which a fragment's Toeplitz block is zero are left
// out.  Double: where the window is wide, tiles lie on one side of shift 0, so the zero
// steps are a triangle at the start of a tile (sx >= 0) or at its end (sx < 0), written out
// as straight-line blocks of 8 steps.  Float: a condition per fragment and 4 steps.
// Rows outside the slice read a zero row and columns past it read zero padding: those
// terms add a product with an exact zero.  Such a term is not neutral for infinities and
// NaN, so a workgroup that stages one sums its shifts term by term instead.
//
// Bound: the matrix pipe (72 TFLOP/s measured for v_mfma_f64_4x4x4 alone).  FP64, 100 ROIs
// of 128 x 128, 16 patterns, 255 x 255 window: 15.4 ms (register-blocked vector kernel
// 27.8 ms; 65 TFLOP/s executed, of which 55 useful); FP64, 25 ROIs of 32 x 32, 16 patterns: 46 us (8-shift vector
// kernel 98 us; 800 workgroups on 256 CUs, 12 us of it staging and results);
// float, 63 ROIs of 75 x 61, 12 patterns, 41 x 33 window: 210 us (935 us; the
// window is computed as 48 x 48).
typedef float mm_f4 __attribute__((ext_vector_type(4)));

template <class T>
struct mm_frag;
template <>
struct mm_frag<double> {
    using acc = double;
    static constexpr int NJ = 4, REGS = 1;
    static __device__ __forceinline__ void mac(acc& c, double a, double b) {
        c = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ double get(const acc& c, int) { return c; }
    // lane l holds D[4 ((l % 16) / 4) + l / 16][l % 4]
    static __device__ __forceinline__ int row(int lane, int) { return 4 * (lane % 16 / 4) + lane / 16; }
    static __device__ __forceinline__ int col(int lane) { return lane % 4; }
};
template <>
struct mm_frag<float> {
    using acc = mm_f4;
    static constexpr int NJ = 16, REGS = 4;
    static __device__ __forceinline__ void mac(acc& c, float a, float b) {
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float get(const acc& c, int r) { return c[r]; }
    // lane l, register r holds D[4 (l / 16) + r][l % 16]
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane / 16) + r; }
    static __device__ __forceinline__ int col(int lane) { return lane % 16; }
};

constexpr int kMmTY = 16;  // y-shifts of a tile

struct mm_shape {
    int tb;              // fragments per tile
    int x0;              // first x-shift of tile 0
    int ntx, nty;        // tiles of a slice
    int wx, wy;          // waves along x-shift tiles and y-shift tiles (wx * wy = 4, or one)
    int ntw;             // x-shift tiles per wave (1 or 2)
    int nxb, nyb;        // workgroups of one slice along x and y
    int cy;              // reference rows per staged chunk
    int prows;           // pattern rows per staged chunk
    int pitch, rpitch;   // LDS row lengths of pattern and reference rows
    int padl;            // zeros before the first reference row
    size_t lds;
};

template <class T>
inline bool mm_plan(size2 size, size2 res, uint64_t total, mm_shape& m) {
    constexpr int NJ = mm_frag<T>::NJ;
    const int rx = (int)(res.x - 1) / 2, w = (int)res.x, S = (int)size.x;
    if (size.x > 4096 || size.y > 65536) return false;
    m.nty = div_up((int)res.y, kMmTY);
    // Tile width: a wide tile reads fewer fragments per product, a narrow one rounds the
    // window and the slice width up less; a narrower one has to save an eighth (a 41 x 33
    // window of 75 x 61 slices in float: 48 wide 217 us, 32 wide 286 us, 16 wide 290 us).
    m.tb = 0;
    int best = 0;
    for (int tb : {32 / NJ, 48 / NJ, 16 / NJ}) {
        if (NJ == 4 && tb == 12) continue;
        const int tx = NJ * tb, unit = NJ == 4 ? tx : 16;
        const int cost = div_up(w, tx) * tx * div_up(S, unit) * unit;
        if (m.tb == 0 || 8ll * cost < 7ll * best) {
            best = cost;
            m.tb = tb;
        }
    }
    const int tx = NJ * m.tb;
    m.ntx = div_up(w, tx);
    m.x0 = -rx;
    const int nneg = div_up(rx, tx);
    const bool split = nneg + div_up(w - rx, tx) == m.ntx;  // tiles on one side of shift 0 cost nothing
    if (split) m.x0 = -tx * nneg;
    // two x-shift tiles per wave (a long and a short one) where that leaves every SIMD four
    // waves; small launches spread over twice the waves instead
    m.ntw = m.ntx > 1 && total * m.nty * div_up(m.ntx, 2) >= 4096 ? 2 : 1;
    const int per = div_up(m.ntx, m.ntw);
    m.wx = per >= 4 ? 4 : (per >= 2 ? 2 : 1);
    m.wy = 4 / m.wx;
    // Small slices take one wave to a workgroup where one or two tiles are all they have (beside
    // it the other three would only stage, which pays for larger slices and tall ones) or where
    // there are two and more for every CU.  Pass over 800 slices, us, four waves / one: 24 x 8 in
    // float 24.1 / 19.9, 8 x 8 16.2 / 14.0, 16 x 16 27.3 / 24.0, 24 x 8 in double 29.7 / 25.6; 25
    // of 16 x 16 in double 15.8 / 18.3, 100 of 24 x 24 with a 9 x 9 window 17.8 / 19.4.
    if (size.area() <= 256 && size.y <= 16 && ((m.nty == 1 && m.ntx <= 2) || total >= 512)) {
        m.ntw = std::min(m.ntx, 2);
        m.wx = m.wy = 1;
    }
    m.nxb = div_up(m.ntx, m.wx * m.ntw);
    m.nyb = div_up(m.nty, m.wy);
    // Pattern rows 2 mod 4 doubles (4 mod 8 floats) apart: the rows of an A fragment fall on
    // distinct banks.  Both kinds of row are followed by the zeros the fragments read past the
    // slice (a pattern row: a tile's columns; a reference row: those and, for a tile across
    // shift 0, its width; float fragments read up to 31 past either end).
    m.pitch = div_up(S, 8) * 8 + (NJ == 4 ? tx + 6 : 20);
    const int padr = NJ == 4 ? (split ? tx : 2 * tx) + 4 : 36;
    m.padl = NJ == 4 ? (split ? 4 : tx + 4) : 36;
    m.rpitch = S + padr;
    const int span = kMmTY * m.wy - 1;
    auto bytes = [&](int cy) {
        m.prows = std::min((int)size.y, cy + span);
        return ((size_t)(m.prows + 1) * m.pitch + (size_t)cy * m.rpitch + m.padl) * sizeof(T);
    };
    // the most rows per chunk that let three workgroups share a CU's 160 KB, else two, else one
    for (size_t budget : {(size_t)53248, (size_t)79872, (size_t)155648}) {
        int cy = (int)size.y;
        while (cy > 0 && bytes(cy) > budget) --cy;
        if (cy >= std::min(8, (int)size.y)) {
            m.cy = cy;
            m.lds = bytes(cy);
            return true;
        }
    }
    return false;
}

template <class T>
__device__ __forceinline__ bool mm_not_finite(T v) {
    if constexpr (sizeof(T) == 8)
        return (__builtin_bit_cast(uint64_t, v) >> 52 & 0x7ff) == 0x7ff;
    else
        return (__builtin_bit_cast(uint32_t, v) >> 23 & 0xff) == 0xff;
}

enum { MM_FULL, MM_HEAD, MM_TAIL };

// Rows [y0, y1) of the chunk for one tile.  pa_of(y): this lane's A element of pattern column
// 0; pr_of(y): its G element of reference column 0 (k - j from the row's start).
template <int TB, class PA, class PR>
__device__ __forceinline__ void mm_tile(double (&acc)[TB], int y0, int y1, PA&& pa_of, PR&& pr_of, int s0, int S) {
    using F = mm_frag<double>;
    constexpr int TX = F::NJ * TB;
    static_assert(F::NJ == 4, "a step moves one fragment");
    double g[TB];  // G(t - n) in g[(t - n) mod TB]; a block of TB steps covers TX columns
    auto block = [&](const double* pa, const double* pr, auto mode_c) {
        constexpr int MODE = decltype(mode_c)::value;
        double a[TB];
#pragma unroll
        for (int t = 0; t < TB; ++t) a[t] = pa[4 * t];
        double h[TB];
#pragma unroll
        for (int t = 0; t < (MODE == MM_TAIL ? 1 : TB); ++t) h[t] = pr[4 * t];
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            if (MODE != MM_TAIL || t == 0) g[t] = h[t];
#pragma unroll
            for (int n = 0; n < TB; ++n) {
                if (MODE == MM_HEAD && t < n) continue;
                if (MODE == MM_TAIL && t > n) continue;
                F::mac(acc[n], a[t], g[(t - n + TB) % TB]);
            }
        }
    };
    using full = std::integral_constant<int, MM_FULL>;
    if (s0 >= 0) {  // columns from s0: the first block is the triangle n <= t
        const int blocks = (S - s0 + TX - 1) / TX;
        if (blocks <= 0) return;
        for (int y = y0; y < y1; ++y) {
            const double* pa = pa_of(y) + s0;
            const double* pr = pr_of(y);
            block(pa, pr, std::integral_constant<int, MM_HEAD>{});
            for (int b = 1; b < blocks; ++b) block(pa + b * TX, pr + b * TX, full{});
        }
    } else {
        // columns from 0; left of shift 0 the last block is the triangle n >= t (of a slice
        // padded to a whole number of blocks)
        const bool neg = s0 + TX <= 0;
        const int blocks = neg ? (max(0, S + s0) + TX - 1) / TX : (S + TX - 1) / TX;
        if (neg && S + s0 + TX - 1 <= 0) return;
        for (int y = y0; y < y1; ++y) {
            const double* pa = pa_of(y);
            const double* pr = pr_of(y) - s0;
#pragma unroll
            for (int n = 1; n < TB; ++n) g[TB - n] = pr[-4 * n];
            for (int b = 0; b < blocks; ++b) block(pa + b * TX, pr + b * TX, full{});
            if (neg) block(pa + blocks * TX, pr + blocks * TX, std::integral_constant<int, MM_TAIL>{});
        }
    }
}

// The same in float, in groups of 4 steps (16 columns, the width of a fragment): fragment n
// at group c reads the G's of group c - n, which move up one fragment per group.
template <int TB, class PA, class PR>
__device__ __forceinline__ void mm_tile(mm_f4 (&acc)[TB], int y0, int y1, PA&& pa_of, PR&& pr_of, int s0, int S) {
    using F = mm_frag<float>;
    const int xb = max(0, s0), base = max(0, -s0);
    auto lo = [&](int n) { return (max(0, s0 + 16 * n) - xb) >> 4; };
    auto hi = [&](int n) { return (min(S, S + s0 + 16 * n + 15) - xb + 15) >> 4; };
    const int groups = hi(TB - 1);
    int all_lo = 0, all_hi = groups;  // groups in which every fragment has terms
#pragma unroll
    for (int n = 0; n < TB; ++n) {
        all_lo = max(all_lo, lo(n));
        all_hi = min(all_hi, hi(n));
    }
    for (int y = y0; y < y1; ++y) {
        const float* pa = pa_of(y) + xb;
        const float* pr = pr_of(y) + base;
        float g[TB][4];
        auto load = [&](const float* q, bool in, float (&v)[4]) {  // zeros where they lie wholly outside the row
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = in ? q[4 * i] : 0.0f;
        };
#pragma unroll
        for (int n = 1; n < TB; ++n) load(pr - 16 * n, base - 16 * n > -16 && base - 16 * n - 15 < S, g[n - 1]);
        auto up = [&] {
#pragma unroll
            for (int n = TB - 1; n > 0; --n)
#pragma unroll
                for (int i = 0; i < 4; ++i) g[n][i] = g[n - 1][i];
        };
        auto some = [&](int c) {
            float a[4];
            up();
            load(pa + 16 * c, true, a);
            load(pr + 16 * c, base + 16 * c - 15 < S, g[0]);
#pragma unroll
            for (int n = 0; n < TB; ++n) {
                if (c < lo(n) || c >= hi(n)) continue;
#pragma unroll
                for (int i = 0; i < 4; ++i) F::mac(acc[n], a[i], g[n][i]);
            }
        };
        int c = 0;
        for (; c < min(all_lo, groups); ++c) some(c);
        if (c < all_hi) {
            // the next group's fragments load while this one's products run
            float a[4], an[4], gn[4];
            load(pa + 16 * c, true, a);
            load(pr + 16 * c, true, gn);
            for (; c < all_hi; ++c) {
                up();
#pragma unroll
                for (int i = 0; i < 4; ++i) g[0][i] = gn[i];
                const int d = min(c + 1, all_hi - 1);
                load(pa + 16 * d, true, an);
                load(pr + 16 * d, true, gn);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int n = 0; n < TB; ++n) F::mac(acc[n], a[i], g[n][i]);
#pragma unroll
                for (int i = 0; i < 4; ++i) a[i] = an[i];
            }
        }
        for (; c < groups; ++c) some(c);
    }
}

template <class T, int TB, int NW>
__global__ __launch_bounds__(64 * NW, 3) void cross_corr_mm_kernel(const T* __restrict__ pics, const T* __restrict__ ref,
                                                               T* __restrict__ res, size2 size, size2 res_size,
                                                               uint32_t nb, uint32_t npat, mm_shape m,
                                                               uint32_t n_wg, uint32_t slab0) {
    using F = mm_frag<T>;
    constexpr int NJ = F::NJ, TX = NJ * TB, NT = kWave * NW;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* prow = reinterpret_cast<T*>(smem_raw);  // prows pattern rows, then one zero row
    T* zrow = prow + (size_t)m.prows * m.pitch;
    T* rrow = zrow + m.pitch;                  // cy reference rows between zeros
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int S = (int)size.x, SY = (int)size.y;
    const int rx = (int)(res_size.x - 1) / 2, ry = (int)(res_size.y - 1) / 2;
    // the workgroups of one slice, then the patterns of one ROI, run back to back on one XCD
    const uint32_t L = xcd_remap(blockIdx.x, n_wg);
    const uint32_t per = (uint32_t)(m.nxb * m.nyb), in_launch = L / per, in = L - in_launch * per;
    const uint32_t slab = slab0 + in_launch;
    const uint32_t roi = slab / npat, sn = (slab - roi * npat) * nb + roi;
    // workgroups that start together on one CU (32 CUs apart in this order) and waves on one
    // SIMD take different y-shift bands: the central ones are several times longer
    const uint32_t turn = slab + (slab >> 4);
    const uint32_t in_t = (in + turn) % per;
    const int yb = (int)(in_t / (uint32_t)m.nxb), xb = (int)in_t - yb * m.nxb;
    const T* p = pics + (size_t)sn * size.area();
    const T* q = ref + (size_t)roi * size.area();

    const int wv = (wave + (int)(turn / per)) & (NW - 1);
    const int wxi = wv % m.wx, wyi = wv / m.wx;
    const int sy0g = yb * kMmTY * m.wy - ry;       // first y-shift of the workgroup
    const int sy0 = sy0g + kMmTY * wyi;            // and of the wave
    int s0[2];                                     // first x-shift of the wave's tiles
    bool on[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int ti = xb * m.wx * m.ntw + wxi + w * m.wx;
        on[w] = w < m.ntw && ti < m.ntx && yb * m.wy + wyi < m.nty;
        s0[w] = m.x0 + TX * ti;
    }
    const int arow = lane % 16, k = lane / 16, j = F::col(lane);

    for (int e = tid; (size_t)e * sizeof(T) < m.lds; e += NT) prow[e] = T(0);
    // staging: element e = tid + NT i lies in row e / S, column e % S
    const int row0 = tid / S, col0 = tid % S, drow = NT / S, dcol = NT % S;

    typename F::acc acc[2][TB];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int n = 0; n < TB; ++n) acc[w][n] = typename F::acc{};
    bool bad = false;

    const int y_lo = max(0, -(sy0g + kMmTY * m.wy - 1)), y_hi = min(SY, SY - sy0g);
    for (int yc = y_lo; yc < y_hi; yc += m.cy) {
        const int ye = min(y_hi, yc + m.cy);
        const int Ya = max(0, yc + sy0g), Yb = min(SY, ye - 1 + sy0g + kMmTY * m.wy);
        __syncthreads();
        constexpr int V = 8;  // loads in flight per thread
        auto stage = [&](const T* src, int rows, T* dst, int pitch) {
            const int n = rows * S;
            int col = col0, at = row0 * pitch + col0;  // of element e: e % S and its LDS place
            for (int e0 = tid; e0 < n; e0 += NT * V) {
                T v[V];
#pragma unroll
                for (int i = 0; i < V; ++i) v[i] = src[min(e0 + i * NT, n - 1)];
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    bad |= mm_not_finite(v[i]);
                    if (e0 + i * NT < n) dst[at] = v[i];
                    const bool wrap = col + dcol >= S;
                    col += dcol - (wrap ? S : 0);
                    at += drow * pitch + dcol + (wrap ? pitch - S : 0);
                }
            }
        };
        stage(p + (size_t)Ya * S, Yb - Ya, prow, m.pitch);
        stage(q + (size_t)yc * S, ye - yc, rrow + m.padl, m.rpitch);
        __syncthreads();
        auto pa_of = [&](int y) {
            const int Y = y + sy0 + arow;
            return ((unsigned)Y < (unsigned)SY ? prow + (Y - Ya) * m.pitch : zrow) + k;
        };
        auto pr_of = [&](int y) { return rrow + (y - yc) * m.rpitch + m.padl + k - j; };
#pragma unroll
        for (int w = 0; w < 2; ++w)
            if (on[w])
                mm_tile<TB>(acc[w], max(yc, -(sy0 + kMmTY - 1)), min(ye, SY - sy0), pa_of, pr_of, s0[w], S);
    }

    T* out = res + (size_t)sn * res_size.area();
    if (__syncthreads_or(bad)) {
        const int nx = TX * m.wx * m.ntw, x0 = m.x0 + nx * xb;
        for (int e = tid; e < nx * kMmTY * m.wy; e += NT) {
            const int sx = x0 + e % nx, sy = sy0g + e / nx;
            if (sx < -rx || sx + rx >= (int)res_size.x || sy + ry >= (int)res_size.y) continue;
            T sum = 0;
            for (int y = max(-sy, 0); y < min(SY, SY - sy); ++y)
                for (int x = max(-sx, 0); x < min(S, S - sx); ++x)
                    sum = mac<T>(p[(size_t)(y + sy) * S + x + sx], q[(size_t)y * S + x], sum);
            out[(size_t)(sy + ry) * res_size.x + sx + rx] = sum;
        }
        return;
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        if (!on[w]) continue;
#pragma unroll
        for (int n = 0; n < TB; ++n) {
            const int sx = s0[w] + NJ * n + j;
            if (sx < -rx || sx + rx >= (int)res_size.x) continue;
#pragma unroll
            for (int r = 0; r < F::REGS; ++r) {
                const int sy = sy0 + F::row(lane, r);
                if (sy + ry < (int)res_size.y) out[(size_t)(sy + ry) * res_size.x + sx + rx] = F::get(acc[w][n], r);
            }
        }
    }
}

// Workgroups of the register-blocked kernel for this launch, or 0 where it does not run
// (shape outside the tiled limits, or fewer workgroups than CUs, where the finer grids of
// the other vector kernels are faster).
template <class T>
uint64_t tiled_workgroups(size2 size, size2 res_size, uint32_t ref_slices, uint32_t batch, tiled_shape& sh) {
    if (!tiled_plan<T>(size, res_size, sh)) return 0;
    const uint64_t n_wg =
        (uint64_t)ref_slices * div_up(batch, (uint32_t)kTiledP) * div_up(res_size.y, (uint32_t)sh.rows);
    return (n_wg >= 256 && n_wg <= (1u << 24)) ? n_wg : 0;
}


// Slices up to this many pixels run one thread per shift: the chains are shorter than what the
// matrix-core kernel does around them (pass over 800 slices in double, us: 4 x 4 16.2 and 12.1,
// 6 x 6 17.0 and 14.2; 8 x 8 in float 16.2 and 17.8).
constexpr uint32_t kTinyArea = 48;

const char* cross_corr_kernel_name(bool is_double, size2 size, size2 res_size, uint32_t ref_slices, uint32_t batch) {
    mm_shape m;
    const uint64_t total = (uint64_t)ref_slices * batch;
    const bool mm = is_double ? mm_plan<double>(size, res_size, total, m) : mm_plan<float>(size, res_size, total, m);
    return mm && !(total <= 65535u && size.area() <= kTinyArea) ? "cross_corr_mm_kernel" : "cross_corr_kernel";
}

template <class T>
void launch_cross_corr(const T* pics, const T* ref, T* res, size2 size, size2 res_size, uint32_t ref_slices,
                       uint32_t batch, hipStream_t st) {
    if (res_size.x > 2 * size.x + 1 || res_size.y > 2 * size.y + 1)
        throw arg_error("cross_corr: res_size must be at most 2*size+1 per axis");
    const uint32_t total = ref_slices * batch;
    if (total == 0 || res_size.area() == 0) return;
    tiled_shape sh;
    const uint64_t n_tiled = tiled_workgroups<T>(size, res_size, ref_slices, batch, sh);
    // more slices than a grid's z extent only where the register-blocked rule holds
    if (!n_tiled && total > 65535u) throw arg_error("cross_corr: more than 65535 slices in one launch");
    if constexpr (std::is_floating_point<T>::value) {
        mm_shape m;
        if (!(total <= 65535u && size.area() <= kTinyArea) && mm_plan<T>(size, res_size, total, m)) {
            auto launch_nw = [&](auto tb, auto nw) {
                auto kern = cross_corr_mm_kernel<T, decltype(tb)::value, decltype(nw)::value>;
                static const hipError_t attr =
                    hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 155648);
                EMIDA_HIP(attr);
                // a grid's extent is below 2^32 threads: whole slices per launch, one launch nearly always
                const uint32_t per = (uint32_t)(m.nxb * m.nyb), most = ((1u << 24) - 1) / per;
                for (uint32_t slab = 0; slab < total; slab += std::min(most, total - slab)) {
                    const uint32_t n_wg = std::min(most, total - slab) * per;
                    kern<<<n_wg, kWave * nw, m.lds, st>>>(pics, ref, res, size, res_size, ref_slices, batch, m, n_wg,
                                                          slab);
                    EMIDA_LAUNCHED("cross_corr_mm_kernel");
                }
            };
            auto launch = [&](auto tb) {
                if (m.wx * m.wy == 1) launch_nw(tb, std::integral_constant<int, 1>{});
                else launch_nw(tb, std::integral_constant<int, 4>{});
            };
            constexpr int NJ = mm_frag<T>::NJ;
            if (m.tb == 32 / NJ) launch(std::integral_constant<int, 32 / NJ>{});
            else if (m.tb == 16 / NJ) launch(std::integral_constant<int, 16 / NJ>{});
            else if constexpr (NJ == 16) launch(std::integral_constant<int, 3>{});
            return;
        }
    }
    if constexpr (!std::is_floating_point<T>::value) {
        if (const uint64_t n_wg = n_tiled) {
            auto kern = cross_corr_tiled_kernel<T>;
            static const hipError_t attr =
                hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
            EMIDA_HIP(attr);
            kern<<<(uint32_t)n_wg, 64 * sh.wx * sh.wy, sh.lds, st>>>(pics, ref, res, size, res_size, ref_slices,
                                                                       batch, sh, (uint32_t)n_wg);
            EMIDA_LAUNCHED("cross_corr_tiled_kernel");
            return;
        }
        if (xn_lds_elems<T>(size) * sizeof(T) <= kBruteLds) {
            dim3 block(kXNTX, kXNTY);
            dim3 grid(div_up(res_size.x, (uint32_t)(kXNTX * kXN)), div_up(res_size.y, (uint32_t)kXNTY), total);
            cross_corr_x8_kernel<T><<<grid, block, xn_lds_elems<T>(size) * sizeof(T), st>>>(pics, ref, res, size,
                                                                                            res_size, ref_slices);
            EMIDA_LAUNCHED("cross_corr_x8_kernel");
            return;
        }
    }
    dim3 block(kBruteTX, kBruteTY);
    dim3 grid(div_up(res_size.x, (uint32_t)kBruteTX), div_up(res_size.y, (uint32_t)kBruteTY), total);
    const size_t lds = 2 * (size_t)size.area() * sizeof(T);
    if (lds <= kBruteLds) {
        cross_corr_kernel<T, true><<<grid, block, lds, st>>>(pics, ref, res, size, res_size, ref_slices);
    } else {
        cross_corr_kernel<T, false><<<grid, block, 0, st>>>(pics, ref, res, size, res_size, ref_slices);
    }
    EMIDA_LAUNCHED("cross_corr_kernel");
}

template void launch_cross_corr<float>(const float*, const float*, float*, size2, size2, uint32_t, uint32_t,
                                       hipStream_t);
template void launch_cross_corr<double>(const double*, const double*, double*, size2, size2, uint32_t, uint32_t,
                                        hipStream_t);
template void launch_cross_corr<int32_t>(const int32_t*, const int32_t*, int32_t*, size2, size2, uint32_t,
                                         uint32_t, hipStream_t);

}  // namespace emida_amd
