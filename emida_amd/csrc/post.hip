// Deformation post-step: per pattern, the projective map (homography) between the
// ROI middles and their displaced positions, fitted algebraically, and its strain and
// rotation.  One wave per pattern, four from 449 ROIs on.
//
// Reference (Python post-processing of the offsets):
//  - python/process_offsets.py:31-97 (and python/test.py:137-198): relative to the
//    pattern centre (cx, cy) and detector distance z, old = mid - c, new = old + offset;
//    rows  [-ox z, -oy z, -z^2, 0, 0, 0, ox nx, oy nx, z nx]
//          [0, 0, 0, -ox z, -oy z, -z^2, ox ny, oy ny, z ny]
//    per ROI; the 3 x 3 map is the right singular vector of the smallest singular value
//    (up to scale); the script prints it divided by its [2][2] element;
//  - jove/analyze.py:37-95: ROIs are used where the fitted quadratic peak is a
//    maximum with determinant a c - b^2 > 1e-6 (a = -coef[3], b = -coef[4] / 2,
//    c = -coef[5]); quality = median of that determinant over all ROIs; a pattern needs
//    more than 10 such ROIs; the map is scaled to determinant 1 (divided by the cube
//    root of its determinant); polar decomposition F = R U with strain log(U) and
//    rotation log(R) from Rodrigues' formula.
// jove/analyze.py:28 fills the second row's oy column with ox ny; this follows
// process_offsets.py (oy ny), the form the algebra requires.
//
// Here the normal matrix G = A^T A (9 x 9) is accumulated in double as the weighted sums of
// v v^T, v = (ox, oy, z), it consists of (weights 1, nx, ny, nx^2 + ny^2: 24 values), and its
// eigenvector of the smallest eigenvalue found by inverse iteration on a block Cholesky
// factorisation (Golub and Van Loan, Matrix Computations, 4th ed., 4.2 and 8.2); where that
// does not converge to rounding within 24 steps, or G is not positive definite beyond its
// last pivot (degenerate ROI layouts, NaN), by cyclic Jacobi rotations.  For the
// well-conditioned systems of ROI grids (largest / second-smallest singular value of A about
// 3) either equals the SVD's singular vector to ~1e-15.  The polar decomposition uses the
// eigen-decomposition of F^T F (3 x 3 Jacobi).  The quality determinant is evaluated
// without contraction, as numpy does, and the median is found by selection, so quality and
// the ROI selection equal numpy's bit for bit.
#include <cmath>

#include "offset.hpp"

namespace emida_amd {
namespace {

constexpr int kPostNT = 256;
constexpr uint32_t kPostMaxRois = 8192;

// Cyclic Jacobi eigen-decomposition of the symmetric N x N matrix a (row-major, in
// place: eigenvalues end on the diagonal); v receives the eigenvectors as columns.
template <int N>
__device__ void jacobi_eigen(double* a, double* v) {
    for (int i = 0; i < N * N; ++i) v[i] = (i / N == i % N) ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0, diag = 0;
        for (int i = 0; i < N; ++i) {
            diag += a[i * N + i] * a[i * N + i];
            for (int j = i + 1; j < N; ++j) off += a[i * N + j] * a[i * N + j];
        }
        if (!(off > 1e-30 * diag)) break;  // converged (also stops on NaN)
        for (int p = 0; p < N - 1; ++p)
            for (int q = p + 1; q < N; ++q) {
                const double apq = a[p * N + q];
                if (apq == 0.0) continue;
                const double theta = (a[q * N + q] - a[p * N + p]) / (2.0 * apq);
                const double t = fabs(theta) > 1e150 ? 0.5 / theta
                                                     : (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
                for (int k = 0; k < N; ++k) {  // columns p, q
                    const double kp = a[k * N + p], kq = a[k * N + q];
                    a[k * N + p] = c * kp - s * kq;
                    a[k * N + q] = s * kp + c * kq;
                }
                for (int k = 0; k < N; ++k) {  // rows p, q
                    const double pk = a[p * N + k], qk = a[q * N + k];
                    a[p * N + k] = c * pk - s * qk;
                    a[q * N + k] = s * pk + c * qk;
                }
                for (int k = 0; k < N; ++k) {
                    const double kp = v[k * N + p], kq = v[k * N + q];
                    v[k * N + p] = c * kp - s * kq;
                    v[k * N + q] = s * kp + c * kq;
                }
            }
    }
}

// 1 / sqrt(v) and 1 / v to about an ulp for v in [1e-290, 1e290] (NaN or infinity outside
// it): the hardware's estimate and Newton steps, a third of the chain of the exactly rounded
// square root and division.
__device__ __forceinline__ double fast_rsqrt(double v) {
    double r = __builtin_amdgcn_rsq(v);
#pragma unroll
    for (int i = 0; i < 2; ++i) r = fma(r, 0.5 * fma(-v * r, r, 1.0), r);
    return r;
}
__device__ __forceinline__ double fast_rcp(double v) {
    double r = __builtin_amdgcn_rcp(v);
#pragma unroll
    for (int i = 0; i < 2; ++i) r = fma(r, fma(-v, r, 1.0), r);
    return r;
}

// The same for a symmetric 3 x 3 matrix held in registers (every index a constant); the
// eigenvectors become the columns of v.
__device__ __forceinline__ void jacobi_eigen3(double (&a)[3][3], double (&v)[3][3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) v[i][j] = i == j ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 60; ++sweep) {
        const double off = a[0][1] * a[0][1] + a[0][2] * a[0][2] + a[1][2] * a[1][2];
        const double diag = a[0][0] * a[0][0] + a[1][1] * a[1][1] + a[2][2] * a[2][2];
        if (!(off > 1e-30 * diag)) break;  // converged (also stops on NaN)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = p + 1; q < 3; ++q) {
                const double apq = a[p][q];
                if (apq == 0.0) continue;
                // t = tan of the rotation: sgn(d) h / (|d| + sqrt(d^2 + h^2))
                const double d = a[q][q] - a[p][p], h = 2.0 * apq, rr = d * d + h * h;
                double t;
                if (rr > 1e-280 && rr < 1e280) {
                    t = copysign(h, d == 0.0 ? h : h * d) * fast_rcp(fabs(d) + rr * fast_rsqrt(rr));
                } else {
                    const double theta = d / h;
                    t = fabs(theta) > 1e150 ? 0.5 / theta
                                            : (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                }
                const double c = fast_rsqrt(t * t + 1.0), s = t * c;
#pragma unroll
                for (int k = 0; k < 3; ++k) {  // columns p, q
                    const double kp = a[k][p], kq = a[k][q];
                    a[k][p] = c * kp - s * kq;
                    a[k][q] = s * kp + c * kq;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {  // rows p, q
                    const double pk = a[p][k], qk = a[q][k];
                    a[p][k] = c * pk - s * qk;
                    a[q][k] = s * pk + c * qk;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double kp = v[k][p], kq = v[k][q];
                    v[k][p] = c * kp - s * kq;
                    v[k][q] = s * kp + c * kq;
                }
            }
    }
}

// Lower Cholesky factor of a symmetric 3 x 3 matrix, in place (strictly lower part), with
// the reciprocals of its diagonal; false when a pivot is not above floor_k.
__device__ __forceinline__ bool cholesky3(double (&m)[3][3], double (&inv)[3], double floor0, double floor1,
                                          double floor2) {
    bool ok = m[0][0] > floor0;
    inv[0] = fast_rsqrt(m[0][0]);
    m[1][0] *= inv[0];
    m[2][0] *= inv[0];
    const double d1 = m[1][1] - m[1][0] * m[1][0];
    ok &= d1 > floor1;
    inv[1] = fast_rsqrt(d1);
    m[2][1] = (m[2][1] - m[2][0] * m[1][0]) * inv[1];
    double d2 = m[2][2] - m[2][0] * m[2][0] - m[2][1] * m[2][1];
    // the last pivot of the whole factorisation is rounding noise for exact data: kept
    // positive, which leaves the null direction dominant in the solves
    if (floor2 < 0) d2 = fmax(d2, -floor2);
    else ok &= d2 > floor2;
    inv[2] = fast_rsqrt(d2);
    return ok;
}
// L^-1 b and L^-T b.
__device__ __forceinline__ void solve_l(const double (&m)[3][3], const double (&inv)[3], double (&b)[3]) {
    b[0] *= inv[0];
    b[1] = (b[1] - m[1][0] * b[0]) * inv[1];
    b[2] = (b[2] - m[2][0] * b[0] - m[2][1] * b[1]) * inv[2];
}
__device__ __forceinline__ void solve_lt(const double (&m)[3][3], const double (&inv)[3], double (&b)[3]) {
    b[2] *= inv[2];
    b[1] = (b[1] - m[2][1] * b[2]) * inv[1];
    b[0] = (b[0] - m[1][0] * b[1] - m[2][0] * b[2]) * inv[0];
}

// The sums of w v v^T the normal matrix consists of: w in {1, nx, ny, nx^2 + ny^2}, the
// entries as monomials {ox^2, ox oy, oy^2, ox, oy, 1} (the powers of z are put in here).
__device__ __forceinline__ void weighted_block(const double* g, double z, double f, double (&m)[3][3]) {
    m[0][0] = f * g[0];
    m[0][1] = m[1][0] = f * g[1];
    m[1][1] = f * g[2];
    m[0][2] = m[2][0] = f * z * g[3];
    m[1][2] = m[2][1] = f * z * g[4];
    m[2][2] = f * z * z * g[5];
}

// Unit eigenvector x of the smallest eigenvalue of
//   G = [S1 0 S2; 0 S1 S3; S2 S3 S4], S1 = z^2 W_1, S2 = -z W_nx, S3 = -z W_ny, S4 = W_q,
// by inverse iteration; false when it did not settle.
__device__ __forceinline__ bool null_vector(const double (&g)[4][6], double z, double (&x)[9]) {
    double l[3][3], li[3], c[3][3], ci[3], w1[3][3], w2[3][3];
    weighted_block(g[0], z, z * z, l);
    weighted_block(g[1], z, -z, w1);
    weighted_block(g[2], z, -z, w2);
    weighted_block(g[3], z, 1.0, c);
    const double scale = l[0][0] + l[1][1] + l[2][2] + c[0][0] + c[1][1] + c[2][2];
    const double c22 = c[2][2];  // the last diagonal element, before its block's Schur complement
    bool ok = cholesky3(l, li, 1e-12 * scale, 1e-12 * scale, 1e-12 * scale);
#pragma unroll
    for (int j = 0; j < 3; ++j) {  // W1 = L^-1 S2, W2 = L^-1 S3, column by column
        double b1[3] = {w1[0][j], w1[1][j], w1[2][j]}, b2[3] = {w2[0][j], w2[1][j], w2[2][j]};
        solve_l(l, li, b1);
        solve_l(l, li, b2);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            w1[i][j] = b1[i];
            w2[i][j] = b2[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) c[i][j] -= w1[k][i] * w1[k][j] + w2[k][i] * w2[k][j];
    // The last pivot's floor is of its own diagonal element's size, not of the whole trace's:
    // ROIs close to the centre make S1 1e6 times S4, and a floor of 1e-17 of the trace stood
    // there above the rounding noise, 5e-9 off in x where Jacobi rotations come within 6e-13
    // (50 ROIs within 0.1 % of a pattern, z its size).  With this floor the same layouts come
    // within 5e-13.  Raising the other pivots' floor as well, to 1e-8 or 1e-6 (Jacobi for more
    // layouts), gains nothing: over 3,334 fits from well to barely determined the mean error
    // is 0.55 times that of Jacobi alone so, 0.65 and 0.73 times there.
    ok &= cholesky3(c, ci, 1e-12 * scale, 1e-12 * scale, -1e-17 * c22);
    if (!ok) return false;
#pragma unroll
    for (int i = 0; i < 9; ++i) x[i] = i % 4 == 0 ? 0.57735026918962573 : 0.0;  // the identity map
    for (int it = 0; it < 24; ++it) {
        double b1[3] = {x[0], x[1], x[2]}, b2[3] = {x[3], x[4], x[5]}, b3[3] = {x[6], x[7], x[8]};
        solve_l(l, li, b1);
        solve_l(l, li, b2);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) b3[i] -= w1[k][i] * b1[k] + w2[k][i] * b2[k];
        solve_l(c, ci, b3);
        solve_lt(c, ci, b3);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b1[i] -= w1[i][k] * b3[k];
                b2[i] -= w2[i][k] * b3[k];
            }
        solve_lt(l, li, b1);
        solve_lt(l, li, b2);
        const double y[9] = {b1[0], b1[1], b1[2], b2[0], b2[1], b2[2], b3[0], b3[1], b3[2]};
        double ss = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) ss += y[i] * y[i];
        const double r = fast_rsqrt(ss);
        double far = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const double v = y[i] * r;
            far = fmax(far, fabs(v - x[i]));
            x[i] = v;
        }
        if (!(ss > 1e-290 && ss < 1e290)) return false;
        if (far < 1e-15) return true;
    }
    return false;
}

struct post_args {
    const double* mids;    // [n_rois][2] or [n_patterns][n_rois][2]
    uint32_t mids_stride;  // doubles between patterns' mids (0: shared)
    uint32_t n;            // ROIs per pattern
    const double* offsets; // [n_patterns][n][2]
    const double* coefs;   // [n_patterns][n][6] or null
    uint32_t npat;
    double cx, cy, z;
    double det_min;
    uint32_t min_rois;
    int32_t* mask;
    double* quality;
    double* H;
    double* F;
    double* eps;
    double* omega;
};

// NW waves per pattern (1: four patterns per workgroup; 4: one), K ROIs per lane; n <= 64 NW K.
// They are held in registers up to 2,048 ROIs (but for 28 to 36 bytes a lane with one wave);
// the 32 per lane beyond go to scratch (944 bytes a lane): a pattern of 2,049 ROIs takes 110 us
// where one of 2,048 takes 24, 1,000 patterns of 8,192 450 us (the kernel described below 43 ms).
// Every lane runs the solve on the same values.
//
// Bound: the reads of the offsets and coefficients, and the chain of dependent operations of
// the solve, which the waves of a SIMD hide for each other.  5,000 patterns x 400 ROIs
// (128 MB): 66 us; one thread of a workgroup running the 9 x 9 Jacobi rotations out of
// LDS, and a rank count over all pairs for the median, took 2,540 us.  Four patterns per wave
// with their solves in four lanes: 95 us where this form took 78 us (fewer waves to hide the
// chain).
template <int NW, int K>
__global__ __launch_bounds__(kPostNT, NW == 1 ? 4 : 2) void deform_fit_kernel(post_args a) {
    typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // pairs at any double
    constexpr int GROUPS = kPostNT / kWave / NW;
    __shared__ double jg[GROUPS][81], jv[GROUPS][81];
    __shared__ double xd[NW == 1 ? 1 : 2 * NW * 26];  // exchange between the waves of a pattern
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), wv = wave % NW, slot = wave / NW;
    const uint32_t p = blockIdx.x * GROUPS + slot;
    if (p >= a.npat) return;  // NW = 4: the whole workgroup
    const uint32_t n = a.n;
    const double* mids = a.mids + (size_t)p * a.mids_stride;
    const double* offs = a.offsets + (size_t)p * n * 2;
    const double z = a.z;

    // Values of all the pattern's waves: a wave's partial results go to xd, everyone combines
    // them in the same order.  Two halves of xd alternate, so one barrier per exchange will do.
    int turn = 0;
    auto exchange = [&](const double* mine, int count, auto&& use) {
        if constexpr (NW > 1) {
            double* buf = xd + (turn ^= 1) * (NW * 26);
            if (lane == 0)
                for (int i = 0; i < count; ++i) buf[wv * 26 + i] = mine[i];
            __syncthreads();
            for (int w = 0; w < NW; ++w) use(buf + w * 26);
        } else {
            use(mine);
        }
    };

    // ---- loads: one ROI per lane and step, all in flight together
    double d[K], cq[K], ox[K], oy[K], nx[K], ny[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i = min((uint32_t)(k * NW + wv) * kWave + lane, n - 1);
        const d2u m = *(const d2u*)(mids + 2 * (size_t)i), o = *(const d2u*)(offs + 2 * (size_t)i);
        ox[k] = m.x;
        oy[k] = m.y;
        nx[k] = o.x;
        ny[k] = o.y;
        if (a.coefs) {
            const double* q = a.coefs + ((size_t)p * n + i) * 6;
            const d2u q45 = *(const d2u*)(q + 4);
            d[k] = q45.x;
            cq[k] = q45.y;
        }
    }
    // ---- quality determinants, ROI selection count, NaN flag
    uint64_t in[K];  // lanes of step k that hold a ROI (wave-uniform masks)
    uint64_t used[K];
    double cnt = 0, nan = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i0 = (uint32_t)(k * NW + wv) * kWave;
        const bool here = i0 + lane < n;
        in[k] = __ballot(here);
        used[k] = in[k];
        if (a.coefs) {
#pragma clang fp contract(off)
            const double qa = -a.coefs[((size_t)p * n + min(i0 + lane, n - 1)) * 6 + 3], qb = -d[k] / 2, qc = -cq[k];
            const double det = qa * qc - qb * qb;
            d[k] = det;
            used[k] = __ballot(here && det > a.det_min);
            nan += __popcll(__ballot(here && det != det));
        }
        cnt += __popcll(used[k]);
    }
    {
        const double mine[2] = {cnt, nan};
        cnt = nan = 0;
        exchange(mine, 2, [&](const double* v) {
            cnt += v[0];
            nan += v[1];
        });
    }

    // ---- median of the determinants (numpy: middle element, or the mean of the two), by
    // quickselect: each step counts the values below and at a pivot taken from those left
    if (a.quality) {
        double quality = NAN;
        if (a.coefs && nan == 0) {
            const uint32_t k1 = (n - 1) / 2, k2 = n / 2;
            uint64_t left[K];
#pragma unroll
            for (int k = 0; k < K; ++k) left[k] = in[k];
            uint32_t below = 0;  // values known to lie below those left
            double v1 = 0, v2 = 0;
            for (uint32_t step = 0; step < n; ++step) {
                // this wave's candidate: the first value left of a lane that turns from step to step
                double mine = 0;
                bool has = false;
#pragma unroll
                for (int k = K - 1; k >= 0; --k) {
                    const bool l = left[k] >> lane & 1;
                    mine = l ? d[k] : mine;
                    has |= l;
                }
                const uint64_t who = __ballot(has);
                const int r = (step * 23 + 31) & 63;  // the first candidate at or after lane r, cyclically
                const uint64_t rot = r ? (who >> r | who << (64 - r)) : who;
                const int src = who ? (__builtin_ctzll(rot) + r) & 63 : 0;
                const uint64_t bits = __builtin_bit_cast(uint64_t, mine);
                double pv = __builtin_bit_cast(
                    double, (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), src) << 32 |
                                (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, src));
                if constexpr (NW > 1) {
                    const double cand[2] = {pv, who ? 1.0 : 0.0};
                    int w = 0;
                    const int from = (int)(step % NW);
                    double best = 0, rank = 2 * NW;
                    exchange(cand, 2, [&](const double* v) {
                        const double order = (w - from + NW) % NW;
                        if (v[1] != 0 && order < rank) {
                            rank = order;
                            best = v[0];
                        }
                        ++w;
                    });
                    pv = best;
                }
                double less = 0, eq = 0;
                uint64_t lt[K], gt[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    lt[k] = __ballot(d[k] < pv) & left[k];
                    gt[k] = __ballot(d[k] > pv) & left[k];
                    less += __popcll(lt[k]);
                    eq += __popcll(left[k] & ~(lt[k] | gt[k]));
                }
                if constexpr (NW > 1) {
                    const double counts[2] = {less, eq};
                    less = eq = 0;
                    exchange(counts, 2, [&](const double* v) {
                        less += v[0];
                        eq += v[1];
                    });
                }
                if (k1 < below + (uint32_t)less) {
#pragma unroll
                    for (int k = 0; k < K; ++k) left[k] = lt[k];
                } else if (k1 < below + (uint32_t)less + (uint32_t)eq) {
                    v1 = v2 = pv;
                    if (k2 >= below + (uint32_t)less + (uint32_t)eq) {  // the next larger value
                        double next = __builtin_huge_val();
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            next = (in[k] >> lane & 1) && d[k] > pv ? fmin(next, d[k]) : next;
                        next = wave_reduce(next, __builtin_huge_val(), [](double x, double y) { return fmin(x, y); });
                        v2 = __builtin_huge_val();
                        exchange(&next, 1, [&](const double* v) { v2 = fmin(v2, v[0]); });
                    }
                    break;
                } else {
                    below += (uint32_t)less + (uint32_t)eq;
#pragma unroll
                    for (int k = 0; k < K; ++k) left[k] = gt[k];
                }
            }
            quality = (v1 + v2) / 2;
        }
        if (wv == 0 && lane == 0) a.quality[p] = quality;
    }

    const bool ok = cnt > (double)a.min_rois;
    if (wv == 0 && lane == 0 && a.mask) a.mask[p] = ok ? 1 : 0;
    if (!ok) {
        if (wv == 0 && lane < 9) {
            if (a.H) a.H[9 * (size_t)p + lane] = NAN;
            if (a.F) a.F[9 * (size_t)p + lane] = NAN;
            if (a.eps) a.eps[9 * (size_t)p + lane] = NAN;
            if (a.omega) a.omega[9 * (size_t)p + lane] = NAN;
        }
        return;
    }

    // ---- the 24 sums of the normal matrix
    double g[4][6];
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int m = 0; m < 6; ++m) g[w][m] = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool u = used[k] >> lane & 1;
        const double x = u ? ox[k] - a.cx : 0.0, y = u ? oy[k] - a.cy : 0.0;
        const double px = u ? (ox[k] + nx[k]) - a.cx : 0.0, py = u ? (oy[k] + ny[k]) - a.cy : 0.0;
        const double m[6] = {x * x, x * y, y * y, x, y, u ? 1.0 : 0.0};
        const double q = px * px + py * py;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            g[0][i] += m[i];
            g[1][i] = fma(px, m[i], g[1][i]);
            g[2][i] = fma(py, m[i], g[2][i]);
            g[3][i] = fma(q, m[i], g[3][i]);
        }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int m = 0; m < 6; ++m) g[w][m] = wave_reduce(g[w][m], 0.0, [](double x, double y) { return x + y; });
    if constexpr (NW > 1) {
        double mine[24];
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            mine[i] = g[i / 6][i % 6];
            g[i / 6][i % 6] = 0;
        }
        exchange(mine, 24, [&](const double* v) {
#pragma unroll
            for (int i = 0; i < 24; ++i) g[i / 6][i % 6] += v[i];
        });
        if (wv != 0) return;
    }

    // ---- null vector
    double x[9];
    if (!null_vector(g, z, x)) {
        double* G = jg[slot];
        double* V = jv[slot];
        if (lane == 0) {
            double* flat = V;  // the sums, addressable
#pragma unroll
            for (int e = 0; e < 24; ++e) flat[e] = g[e / 6][e % 6];
            for (int i = 0; i < 9; ++i)
                for (int j = 0; j < 9; ++j) {
                    const int bi = i / 3, bj = j / 3;
                    const int w = bi == bj ? (bi == 2 ? 3 : 0) : bi + bj == 1 ? -1 : bi + bj - 1;
                    const int r = min(i % 3, j % 3), c = max(i % 3, j % 3);
                    const int m = r == 0 ? (c == 0 ? 0 : c == 1 ? 1 : 3) : r == 1 ? (c == 1 ? 2 : 4) : 5;
                    const double zz = r == 2 ? z * z : c == 2 ? z : 1.0;
                    G[i * 9 + j] = w < 0 ? 0.0 : (w == 0 ? z * z : w == 3 ? 1.0 : -z) * zz * flat[w * 6 + m];
                }
            jacobi_eigen<9>(G, V);
            int kmin = 0;
            for (int k = 1; k < 9; ++k)
                if (G[k * 9 + k] < G[kmin * 9 + kmin]) kmin = k;
            for (int k = 0; k < 9; ++k) G[k] = V[k * 9 + kmin];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int k = 0; k < 9; ++k) x[k] = G[k];
    }
    auto store = [&](double* dst, const double (&v)[9]) {
        if (dst && lane == 0) {
#pragma unroll
            for (int k = 0; k < 9; ++k) dst[9 * (size_t)p + k] = v[k];
        }
    };
    {
#pragma clang fp contract(off)
        double h[9];  // row-major 3 x 3
#pragma unroll
        for (int k = 0; k < 9; ++k) h[k] = x[k] / x[8];
        store(a.H, h);
        const double det = x[0] * (x[4] * x[8] - x[5] * x[7]) - x[1] * (x[3] * x[8] - x[5] * x[6]) +
                           x[2] * (x[3] * x[7] - x[4] * x[6]);
        const double scale = cbrt(det);
        double f[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) f[k] = x[k] / scale;
        store(a.F, f);
        if (!a.eps && !a.omega) return;

        // ---- polar decomposition F = R U: U^2 = F^T F = V diag(l) V^T
        double c[3][3], v[3][3], ls[3], ll[3], li[3], e[9], ui[9], r[9], kk[9], ss = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) c[i][j] = f[i] * f[j] + f[3 + i] * f[3 + j] + f[6 + i] * f[6 + j];
        jacobi_eigen3(c, v);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            ls[k] = sqrt(c[k][k]);  // singular values of F
            ll[k] = log(ls[k]);
            li[k] = 1.0 / ls[k];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                double s = 0, u = 0;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    s += ll[k] * v[i][k] * v[j][k];
                    u += v[i][k] * v[j][k] * li[k];
                }
                e[i * 3 + j] = s;   // log(U)
                ui[i * 3 + j] = u;  // U^-1
            }
        store(a.eps, e);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                r[i * 3 + j] = f[i * 3] * ui[j] + f[i * 3 + 1] * ui[3 + j] + f[i * 3 + 2] * ui[6 + j];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                kk[i * 3 + j] = (r[i * 3 + j] - r[j * 3 + i]) / 2;
                ss += kk[i * 3 + j] * kk[i * 3 + j];
            }
        const double sin_t = sqrt(ss / 2);
        const double fac = asin(sin_t) / sin_t;  // 0 / 0 for no rotation, as the reference
#pragma unroll
        for (int k = 0; k < 9; ++k) kk[k] *= fac;
        store(a.omega, kk);
    }
}

template <int NW, int K>
void launch_deform_fit(const post_args& a, hipStream_t st) {
    deform_fit_kernel<NW, K><<<div_up(a.npat, (uint32_t)(kPostNT / kWave / NW)), kPostNT, 0, st>>>(a);
    EMIDA_LAUNCHED("deform_fit_kernel");
}

}  // namespace
}  // namespace emida_amd

extern "C" int emida_fit_deformation(const double* mids, int mids_per_pattern, uint32_t n_rois,
                                     const double* offsets, const double* coefs, uint32_t n_patterns,
                                     emida_calib calib, double det_min, uint32_t min_rois, int32_t* mask,
                                     double* quality, double* H, double* F, double* epsilon, double* omega,
                                     void* stream) {
    return guarded([&] {
        if (!mids || !offsets) throw arg_error("null argument");
        if (n_rois == 0 || n_rois > kPostMaxRois)
            throw arg_error("n_rois must be in 1.." + std::to_string(kPostMaxRois));
        if (!coefs && n_rois <= 4) throw arg_error("the algebraic fit needs more than 4 ROIs");
        if (n_patterns == 0) return;
        post_args a{};
        a.mids = mids;
        a.mids_stride = mids_per_pattern ? 2 * n_rois : 0;
        a.n = n_rois;
        a.offsets = offsets;
        a.coefs = coefs;
        a.npat = n_patterns;
        a.cx = calib.x;
        a.cy = calib.y;
        a.z = calib.z;
        a.det_min = det_min;
        a.min_rois = coefs ? min_rois : 4;
        a.mask = mask;
        a.quality = quality;
        a.H = H;
        a.F = F;
        a.eps = epsilon;
        a.omega = omega;
        // one wave per pattern while its ROIs fit a wave's registers, four beyond
        const hipStream_t st = (hipStream_t)stream;
        if (n_rois <= 128) launch_deform_fit<1, 2>(a, st);
        else if (n_rois <= 256) launch_deform_fit<1, 4>(a, st);
        else if (n_rois <= 448) launch_deform_fit<1, 7>(a, st);
        else if (n_rois <= 1024) launch_deform_fit<4, 4>(a, st);
        else if (n_rois <= 2048) launch_deform_fit<4, 8>(a, st);
        else launch_deform_fit<4, 32>(a, st);
    });
}
