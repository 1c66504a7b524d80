// Rayleigh-Ritz eigensolver of the Davidson projected matrix, on the device: the lowest
// nwant eigenpairs of a Hermitian m x m matrix (m <= 128, nwant <= 32) in one workgroup
// of 8 waves, so that the solver's iterations need no host round trip for it. Bound by latency:
// every part below is a chain over the m rows.
//
//  1. Householder reduction to a Hermitian tridiagonal, the same reflections as the host
//     solver (common/heev.hpp): column k below the diagonal, x, goes to alpha e_1 with
//     alpha = -phase(x_0) |x| by I - 2 v v^H, v = (x - alpha e_1) / |x - alpha e_1|, and the
//     matrix becomes (I - 2 v v^H) A (I - 2 v v^H) = A - 2 (v w^H + w v^H), p = A v,
//     w = p - (v^H p) v. Wave 0 owns no rows and computes the reflectors; waves 1..7 hold the
//     rows cw, cw + 7, ... of the matrix in registers, lane l the columns l and l + 64. A step:
//       rows    p_j over the wave's rows, sum_i conj(A_ij) v_i: the v_i are the same for all
//               lanes (v_readlane), the columns the lane's own, so nothing is reduced across
//               lanes; the seven partial sums go to LDS                             [barrier]
//       wave 0  p, v^H p, w to LDS                                                  [barrier]
//       rows    the rank-2 update of the wave's rows, meanwhile
//       wave 0  row k + 1 of the updated matrix, v_{k+1} to LDS                     [barrier]
//     Per step and wave that is 2 to 4 LDS reads of 16 bytes per lane (a layout of 8 rows per
//     wave with every wave deriving each reflector itself read 50 and was bound by them, at one
//     barrier a step: 2.7 us a step at m = 32, 3.4 at 96; now 1.3 and 2.5, most of it the rows'
//     broadcasts and multiply-adds).
//  2. A diagonal phase change makes the tridiagonal real (T_complex = Ph T Ph^H; prefix products
//     of the phases); the lowest nwant eigenvalues by multisection on Sturm counts (256 lanes in
//     all), counted as the sign changes of the leading principal minors
//     p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}, scaled by the norm and rescaled every eight
//     rows: one dependent multiply-add per row instead of a reciprocal (53 -> 24 us at m = 96).
//  3. Their eigenvectors by inverse iteration, one lane each (LU with partial pivoting of
//     T - lambda I, refactored with every forward solve so that only U is stored; from a
//     fixed pseudo-random start until the growth test of LAPACK dstein passes, then once
//     more, at most four solves; the host solver's shifts for coincident eigenvalues); the row
//     exchange is a choice of operands, with one reciprocal (two branches with a division each:
//     60 -> 41 us); each vector is then orthogonalised against the earlier vectors of its
//     cluster of close eigenvalues (modified Gram-Schmidt).
//  4. Back-transformation y = H_0 ... H_{m-3} Ph z, 16 lanes per vector, the reflectors
//     staged through LDS, the next one loaded ahead, the rows' loops sized by m.
// m = 32 / 64 / 96 / 128, 32 vectors, FP64 reduction: 159 / 323 / 522 / 756 -> 80 / 172 / 351 /
// 476 us; FP32 reduction 124 / 251 / 399 / 571 -> 63 / 133 / 283 / 384 us.
#include <cfloat>
#include <type_traits>

#include "context.hpp"
#include "cplx.hpp"
#include "wave_sums.hpp"

namespace xatu_dev {
namespace {

constexpr int kEM = 128;         // largest projected dimension
constexpr int kEThreads = 512;   // one workgroup: wave 0 and the row waves
constexpr int kERowWaves = 7;
constexpr int kEWant = 32;       // most eigenpairs
constexpr int kEPad = kEM + 1;   // padded row of the per-eigenvector arrays
constexpr int kEStage = 32;      // reflectors per LDS stage of the back-transformation

template <typename TR>
struct EigLds {
    union {
        struct {
            cx_t<TR> part[kERowWaves][kEM];  // partial sums of p
            cx_t<TR> row[2][kEM];            // row k + 1 before the update of step k, by parity of k + 1
            cx_t<TR> u[kEM], q[kEM];         // the step's vectors (see reduce_to_tridiagonal)
        } tri;
        struct {
            double ui[kEWant][kEPad], u1[kEWant][kEPad], u2[kEWant][kEPad];  // U rows; ui = 1 / u0
        } inv;
        double2 refl[kEStage][kEM];
    };
    double z[kEWant][kEPad];  // real tridiagonal eigenvectors
    double d[kEM + 8], e[kEM + 8];
    double2 st[kEM + 24];     // (d_i, e_{i-1}^2) in units of the norm, for the Sturm counts
    double2 ec[kEM], ph[kEM];
    double lam[kEWant], shift[kEWant];
    int cstart[kEWant];
    double tnorm, glo, ghi;
};

__device__ inline double2 csc(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ inline float2 csc(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// 1 / sqrt(x) for normal positive x: the hardware estimate refined by Newton steps.
__device__ inline double rsq(double x) {
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const double h = 0.5 * y;
        y = fma(h, fma(-x * y, y, 1.0), y);
    }
    return y;
}
__device__ inline float rsq(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    return fmaf(0.5f * y, fmaf(-x * y, y, 1.0f), y);
}
// Range in which the products of the reflector's scalars stay normal.
template <typename T>
__device__ inline bool safe_scalar(T x) {
    return sizeof(T) == 8 ? (x > T(1e-280) && x < T(1e280)) : (x > T(1e-34f) && x < T(1e34f));
}

// Value of lane `from` (uniform), the same in every lane.
__device__ inline double lane_value(double x, int from) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), from);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), from);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ inline float lane_value(float x, int from) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), from));
}
template <typename C>
__device__ inline C lane_value_cx(C x, int from) {
    x.x = lane_value(x.x, from);
    x.y = lane_value(x.y, from);
    return x;
}

__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Workgroup barrier that waits for this wave's LDS operations only (its global stores,
// the reflectors read after a full __syncthreads, stay in flight).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 1 / q for normal q: the hardware estimate refined by two Newton steps.
__device__ inline double recip(double q) {
    double y = __builtin_amdgcn_rcp(q);
    y = fma(y, fma(-q, y, 1.0), y);
    return fma(y, fma(-q, y, 1.0), y);
}

// Householder reduction (part 1): matrix A (lda), d, ec and the reflectors; CB column blocks of
// 64 (m <= 64 CB). The waves exchange u = |u| v (so that the row waves need not wait for its
// norm) and q = 2 w / |u|, with which the update is A -= u q^H + q u^H. Entries of u and q at or
// left of k are zero, so finished rows and columns take part without effect; groups of four
// row slots and, past column 64, the first column block are skipped once they are all finished.
template <typename TR, int CB>
__device__ inline void reduce_to_tridiagonal(EigLds<TR>& s, const double2* __restrict__ A, int lda, int m,
                                             cx_t<TR>* __restrict__ refl) {
    using CT = cx_t<TR>;
    constexpr int RA = (64 * CB + kERowWaves - 1) / kERowWaves;  // rows per row wave
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    if (wave > 0) {
        const int cw = wave - 1;
        CT B[RA][CB];  // A[cw + 7 a][lane + 64 b], Hermitian from the lower triangle
#pragma unroll
        for (int a = 0; a < RA; ++a)
#pragma unroll
            for (int b = 0; b < CB; ++b) {
                const int r = cw + kERowWaves * a, c = lane + 64 * b;
                double2 x = make_double2(0.0, 0.0);
                if (r < m && c < m) x = (r >= c) ? A[r + static_cast<size_t>(c) * lda] : cconj(A[c + static_cast<size_t>(r) * lda]);
                if (r == c) x.y = 0.0;
                B[a][b] = mk(static_cast<TR>(x.x), static_cast<TR>(x.y));
            }
        if (cw < 2) {
#pragma unroll
            for (int b = 0; b < CB; ++b) s.tri.row[cw][lane + 64 * b] = B[0][b];
        }
        // entry r = cw + 7 a of a vector held by lanes (64 entries per block)
        auto entry = [&](const CT (&x)[CB], int a) -> CT {
            const int r = cw + kERowWaves * a;
            if (CB == 1 || kERowWaves * a + kERowWaves - 1 < 64) {
                CT e = lane_value_cx(x[0], r & 63);
                if (CB == 1 && a == RA - 1 && r >= 64) e = mk(TR(0), TR(0));
                return e;
            }
            CT e = lane_value_cx(x[CB - 1], r & 63);
            if (kERowWaves * a < 64) {  // the slot on the border of the blocks
                const CT lo = lane_value_cx(x[0], r & 63);
                if (r < 64) e = lo;
            }
            if (a == RA - 1 && r >= 64 * CB) e = mk(TR(0), TR(0));
            return e;
        };
        lds_barrier();  // rows 0 and 1
        lds_barrier();  // u of step 0
        auto steps = [&](auto first_block, int k0, int k1) {
            constexpr int BL = decltype(first_block)::value;
            constexpr int AL = 64 * BL / kERowWaves;  // earlier slots hold rows below 64 BL only
            for (int k = k0; k < k1; ++k) {
                CT u[CB], p[CB];
#pragma unroll
                for (int b = 0; b < CB; ++b) {
                    u[b] = s.tri.u[lane + 64 * b];
                    p[b] = mk(TR(0), TR(0));
                }
#pragma unroll
                for (int a0 = AL; a0 < RA; a0 += 4) {
                    if (cw + kERowWaves * (a0 + 3) > k && cw + kERowWaves * a0 < m) {
#pragma unroll
                        for (int a = a0; a < a0 + 4 && a < RA; ++a) {
                            const CT ur = entry(u, a);
#pragma unroll
                            for (int b = BL; b < CB; ++b) cfma_conj(p[b], B[a][b], ur);
                        }
                    }
                }
#pragma unroll
                for (int b = BL; b < CB; ++b) s.tri.part[cw][lane + 64 * b] = p[b];
                lds_barrier();  // partial sums
                lds_barrier();  // q
                CT q[CB];
#pragma unroll
                for (int b = 0; b < CB; ++b) q[b] = s.tri.q[lane + 64 * b];
#pragma unroll
                for (int a0 = AL; a0 < RA; a0 += 4) {
                    if (cw + kERowWaves * (a0 + 3) > k + 1 && cw + kERowWaves * a0 < m) {
#pragma unroll
                        for (int a = a0; a < a0 + 4 && a < RA; ++a) {
                            const CT ur = entry(u, a), qr = entry(q, a);
#pragma unroll
                            for (int b = BL; b < CB; ++b) {
                                CT x = B[a][b];
                                x.x = fma(-ur.x, q[b].x, x.x);
                                x.x = fma(-ur.y, q[b].y, x.x);
                                x.x = fma(-qr.x, u[b].x, x.x);
                                x.x = fma(-qr.y, u[b].y, x.x);
                                x.y = fma(ur.x, q[b].y, x.y);
                                x.y = fma(-ur.y, q[b].x, x.y);
                                x.y = fma(qr.x, u[b].y, x.y);
                                x.y = fma(-qr.y, u[b].x, x.y);
                                B[a][b] = x;
                            }
                            if (cw + kERowWaves * a == k + 2) {  // the row that wave 0 needs next
#pragma unroll
                                for (int b = BL; b < CB; ++b) s.tri.row[k & 1][lane + 64 * b] = B[a][b];
                            }
                        }
                    }
                }
                lds_barrier();  // u of step k + 1
            }
        };
        steps(std::integral_constant<int, 0>{}, 0, CB == 1 ? m - 2 : min(m - 2, 64));
        if constexpr (CB > 1) steps(std::integral_constant<int, 1>{}, 64, m - 2);
#pragma unroll
        for (int a = 0; a < RA; ++a)
#pragma unroll
            for (int b = 0; b < CB; ++b)
                if (cw + kERowWaves * a == m - 1 && lane + 64 * b == m - 1) s.d[m - 1] = B[a][b].x;
        return;
    }
    // wave 0: entry j = lane + 64 b of u, q and of the current row
    CT u[CB], q[CB];
    TR inv = TR(0);  // 1 / |u|
#pragma unroll
    for (int b = 0; b < CB; ++b) u[b] = q[b] = mk(TR(0), TR(0));
    auto entry = [&](const CT (&x)[CB], int i) -> CT {
        return (CB > 1 && i >= 64) ? lane_value_cx(x[CB - 1], i - 64) : lane_value_cx(x[0], i & 63);
    };
    // reflector of step k from row k of the matrix before the update of step k - 1, which is
    // applied to it here; u to LDS, its norm afterwards
    auto reflector = [&](int k, const CT (&row)[CB]) {
        const CT uk = entry(u, k), qk = entry(q, k);
        const int k1 = k + 1;
        CT x[CB];  // conj(A[k][j])
        TR tl = TR(0);
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            const int j = lane + 64 * b;
            CT a = row[b];  // a -= u_k conj(q_j) + q_k conj(u_j)
            a.x = fma(-uk.x, q[b].x, a.x);
            a.x = fma(-uk.y, q[b].y, a.x);
            a.x = fma(-qk.x, u[b].x, a.x);
            a.x = fma(-qk.y, u[b].y, a.x);
            a.y = fma(uk.x, q[b].y, a.y);
            a.y = fma(-uk.y, q[b].x, a.y);
            a.y = fma(qk.x, u[b].y, a.y);
            a.y = fma(-qk.y, u[b].x, a.y);
            x[b] = cconj(a);
            if (j > k1 && j < m) tl += x[b].x * x[b].x + x[b].y * x[b].y;
        }
        const TR dk = entry(x, k).x;
        const CT x0 = entry(x, k1);
        tl = wave_sum(tl);  // |x|^2 without x_0
        const TR a0 = x0.x * x0.x + x0.y * x0.y;
        const TR xn2 = tl + a0;
        CT ek = x0, u0 = mk(TR(0), TR(0));
        TR un2 = TR(0);  // |u|^2
        if (!(xn2 == TR(0) || tl <= TR(0))) {
            // alpha = -x0 |x| / |x0| (= -|x| for x0 = 0), u0 = x0 - alpha
            const TR g2 = xn2 * a0;
            if (safe_scalar(g2) && safe_scalar(xn2)) {
                const TR r = rsq(g2), f = xn2 * r;  // |x| / |x0|
                ek = csc(x0, -f);
                u0 = csc(x0, TR(1) + f);
                un2 = TR(2) * fma(g2, r, xn2);  // 2 (|x|^2 + |x| |x0|)
            } else {
                if (a0 > TR(0)) {
                    const TR f = sqrt(xn2 / a0);
                    ek = csc(x0, -f);
                    u0 = csc(x0, TR(1) + f);
                } else {
                    ek = mk(-sqrt(xn2), TR(0));
                    u0 = mk(-ek.x, TR(0));
                }
                un2 = tl + u0.x * u0.x + u0.y * u0.y;
            }
        }
        const bool none = un2 == TR(0);
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            const int j = lane + 64 * b;
            u[b] = (j > k1 && j < m && !none) ? x[b] : (j == k1 ? u0 : mk(TR(0), TR(0)));
            s.tri.u[j] = u[b];
        }
        lds_barrier();  // u of step k
        inv = none ? TR(0) : (safe_scalar(un2) ? rsq(un2) : TR(1) / sqrt(un2));
        if (k + 2 < m) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
                refl[static_cast<size_t>(k) * kEM + lane + 64 * b] = b < CB ? csc(u[b < CB ? b : 0], inv) : mk(TR(0), TR(0));
        }
        if (lane == 0) {
            s.d[k] = dk;
            s.ec[k] = make_double2(ek.x, ek.y);
        }
    };
    lds_barrier();  // rows 0 and 1
    CT row[CB];
#pragma unroll
    for (int b = 0; b < CB; ++b) row[b] = s.tri.row[0][lane + 64 * b];
    if (m >= 2) reflector(0, row);
    else lds_barrier();
    for (int k = 0; k + 2 < m; ++k) {
#pragma unroll
        for (int b = 0; b < CB; ++b) row[b] = s.tri.row[(k + 1) & 1][lane + 64 * b];
        lds_barrier();  // partial sums
        CT p[CB], v[CB];
        TR c = TR(0);
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            const int j = lane + 64 * b;
            CT t[kERowWaves];
#pragma unroll
            for (int i = 0; i < kERowWaves; ++i) t[i] = s.tri.part[i][j];
            p[b] = cadd(cadd(cadd(t[0], t[1]), cadd(t[2], t[3])), cadd(cadd(t[4], t[5]), t[6]));
            p[b] = (j <= k || j >= m) ? mk(TR(0), TR(0)) : csc(p[b], inv);  // A v
            v[b] = csc(u[b], inv);
            c += v[b].x * p[b].x + v[b].y * p[b].y;
        }
        c = wave_sum(c);  // v^H p
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            q[b] = csc(mk(fma(-c, v[b].x, p[b].x), fma(-c, v[b].y, p[b].y)), TR(2) * inv);
            s.tri.q[lane + 64 * b] = q[b];
        }
        lds_barrier();  // q
        reflector(k + 1, row);  // with the barrier for its u
    }
}

// Part 4 for m <= 16 NQ: y = H_0 ... H_{m-3} Ph z, 16 lanes per vector.
template <typename TR, int NQ>
__device__ inline void back_transform(EigLds<TR>& s, int m, int nwant, const cx_t<TR>* __restrict__ refl,
                                      double* __restrict__ theta, double2* __restrict__ Y, int ldy) {
    const int t = threadIdx.x, vec = t >> 4, ls = t & 15;
    double2 x[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = ls + 16 * q;
        x[q] = (vec < nwant && i < m) ? csc(s.ph[i], s.z[vec < nwant ? vec : 0][i]) : make_double2(0.0, 0.0);
    }
    for (int k1 = m - 2; k1 > 0; k1 -= kEStage) {  // reflectors k1 - 1 down to max(0, k1 - kEStage)
        const int k0 = max(0, k1 - kEStage);
        __syncthreads();  // the previous stage (or z) is no longer read
        for (int e = t; e < (k1 - k0) * kEM; e += kEThreads) {
            const int kk = e / kEM, i = e % kEM;
            const cx_t<TR> rv = refl[static_cast<size_t>(k0 + kk) * kEM + i];
            s.refl[kk][i] = make_double2(rv.x, rv.y);
        }
        __syncthreads();
        double2 nx[NQ];  // the next reflector, loaded ahead
#pragma unroll
        for (int q = 0; q < NQ; ++q) nx[q] = s.refl[k1 - 1 - k0][ls + 16 * q];
        for (int k = k1 - 1; k >= k0; --k) {
            double2 v[NQ], s0 = make_double2(0.0, 0.0), s1 = make_double2(0.0, 0.0);
            const int kn = max(k - 1, k0) - k0;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                v[q] = nx[q];
                nx[q] = s.refl[kn][ls + 16 * q];
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) cfma_conj((q & 1) ? s1 : s0, v[q], x[q]);
            const double2 f = make_double2(-2.0 * sum16_row(s0.x + s1.x), -2.0 * sum16_row(s0.y + s1.y));
#pragma unroll
            for (int q = 0; q < NQ; ++q) cfma(x[q], v[q], f);
        }
    }
    if (vec < nwant) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int i = ls + 16 * q;
            if (i < m) Y[i + static_cast<size_t>(vec) * ldy] = x[q];
        }
        if (ls == 0) theta[vec] = s.lam[vec];
    }
}

// TR: arithmetic of the tridiagonalisation (float or double); the eigenvalues, eigenvectors
// and back-transformation are FP64.
template <typename TR>
__global__ __launch_bounds__(kEThreads) void projected_eigen_kernel(const double2* __restrict__ A, int lda, int m,
                                                                    int nwant, cx_t<TR>* __restrict__ refl,
                                                                    double* __restrict__ theta,
                                                                    double2* __restrict__ Y, int ldy,
                                                                    unsigned long long* __restrict__ stamp) {
    if (threadIdx.x == 0) *stamp = wall_clock64();
    using CT = cx_t<TR>;
    // working accuracy of the tridiagonal: the eigenvalues are resolved to it (multisection
    // tolerance, shift separation, inverse-iteration growth test), not beyond
    constexpr double kTolEps = sizeof(TR) == 4 ? static_cast<double>(FLT_EPSILON) : DBL_EPSILON;
    __shared__ EigLds<TR> s;
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;

    // ---- 1. tridiagonalisation -------------------------------------------------------
    if (m <= 64) reduce_to_tridiagonal<TR, 1>(s, A, lda, m, refl);
    else reduce_to_tridiagonal<TR, 2>(s, A, lda, m, refl);
    __syncthreads();

    // ---- 2. real tridiagonal, bounds; lowest eigenvalues -------------------------------
    if (w == 0) {
        // entries i = 2 lane, 2 lane + 1: moduli and phases of the off-diagonal, the prefix
        // products of the phases, the Gershgorin bounds
        double ae[2];
        double2 q[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = 2 * lane + u;
            const double2 c = i + 1 < m ? s.ec[i] : make_double2(0.0, 0.0);
            ae[u] = hypot(c.x, c.y);
            q[u] = ae[u] > 0.0 ? csc(c, 1.0 / ae[u]) : make_double2(1.0, 0.0);
            s.e[i] = ae[u];
        }
        double2 run = cmul(q[0], q[1]);  // inclusive products over the lanes' pairs
#pragma unroll
        for (int st = 1; st < 64; st <<= 1) {
            const double2 o = make_double2(__shfl_up(run.x, st), __shfl_up(run.y, st));
            if (lane >= st) run = cmul(o, run);
        }
        const double2 before = make_double2(__shfl_up(run.x, 1), __shfl_up(run.y, 1));
        const double2 p0 = lane ? before : make_double2(1.0, 0.0);
        s.ph[2 * lane] = p0;
        s.ph[2 * lane + 1] = cmul(p0, q[0]);
        const double left = __shfl_up(ae[1], 1);
        double tn = 0.0, lo = s.d[0], hi = s.d[0];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = 2 * lane + u;
            if (i < m) {
                const double off = ae[u] + (u ? ae[0] : (lane ? left : 0.0));
                tn = fmax(tn, fabs(s.d[i]) + off);
                lo = fmin(lo, s.d[i] - off);
                hi = fmax(hi, s.d[i] + off);
            }
        }
#pragma unroll
        for (int st = 1; st < 64; st <<= 1) {
            tn = fmax(tn, __shfl_xor(tn, st));
            lo = fmin(lo, __shfl_xor(lo, st));
            hi = fmax(hi, __shfl_xor(hi, st));
        }
        // Sturm rows in units of the norm; an off-diagonal is not taken below 1e-20 of it, so
        // that a vanishing minor is always followed by one of the opposite sign of the one before
        const double scale = tn > 0.0 ? 1.0 / tn : 1.0;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = 2 * lane + u;
            const double el = (u ? ae[0] : (lane ? left : 0.0)) * scale;
            // rows past m change no sign of the counts
            s.st[i] = i < m ? make_double2(s.d[i] * scale, fmax(el * el, 1e-40)) : make_double2(4.0, 0.0);
            if (i >= m) s.d[i] = 4.0 * tn;  // decoupled rows for the solves' padding
        }
        if (lane < 24) s.st[kEM + lane] = make_double2(4.0, 0.0);
        if (lane < 8) {
            s.d[kEM + lane] = 4.0 * tn;
            s.e[kEM + lane] = 0.0;
        }
        if (lane == 0) {
            const double fudge = 1e-12 * tn;
            s.tnorm = tn;
            s.glo = lo - fudge;
            s.ghi = hi + fudge;
        }
    }
    __syncthreads();
    {
        int nwp = 1;
        while (nwp < nwant) nwp <<= 1;
        // lanes per eigenvalue, a power of two: 256 lanes in all, a wave per SIMD (the counts are
        // bound by instruction issue, so more lanes cost more than the iterations they save)
        const int G = min(64, 256 / nwp);
        const int ev = t / G, gs = t % G;
        const double tnorm = s.tnorm, scale = tnorm > 0.0 ? 1.0 / tnorm : 1.0;
        if (ev < nwant) {
            double lo = s.glo, hi = s.ghi;
            const int gshift = lane - gs;  // first lane of the group in the wave
            const unsigned long long gmask = (G == 64) ? ~0ull : ((1ull << G) - 1ull);
            for (int it = 0; it < 64; ++it) {
                if (hi - lo <= kTolEps * (2.0 * fmax(fabs(lo), fabs(hi)) + tnorm)) break;
                const double step = (hi - lo) / (G + 1);
                const double x = (lo + step * (gs + 1)) * scale;
                // Sturm count: sign changes of the leading minors = eigenvalues below x
                double p0 = 1.0, p1 = s.st[0].x - x;
                unsigned cnt = static_cast<unsigned>(__double2hiint(p1)) >> 31;
                double2 r[8];  // eight rows, the next eight loaded ahead
#pragma unroll
                for (int u = 0; u < 8; ++u) r[u] = s.st[1 + u];
                for (int i0 = 1; i0 < m; i0 += 8) {
                    double2 c[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        c[u] = r[u];
                        r[u] = s.st[i0 + 8 + u];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const double pn = fma(c[u].x - x, p1, -(c[u].y * p0));
                        cnt += static_cast<unsigned>(__double2hiint(pn) ^ __double2hiint(p1)) >> 31;
                        p0 = p1;
                        p1 = pn;
                    }
                    const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(p1)));
                    p0 = __builtin_amdgcn_ldexp(p0, ex);
                    p1 = __builtin_amdgcn_ldexp(p1, ex);
                }
                const unsigned long long bal = __ballot(static_cast<int>(cnt) >= ev + 1);
                const unsigned long long mine = (bal >> gshift) & gmask;
                const int first = mine ? __ffsll(static_cast<long long>(mine)) - 1 : G;
                const double nlo = first == 0 ? lo : lo + step * first;
                const double nhi = first == G ? hi : lo + step * (first + 1);
                lo = nlo;
                hi = nhi;
            }
            if (gs == 0) s.lam[ev] = 0.5 * (lo + hi);
        }
    }
    __syncthreads();
    if (t == 0) {
        // clusters of close eigenvalues and separated shifts for coincident ones
        const double cluster = 1e-3 * fmax(s.tnorm, 1e-300);
        const double sep = 10.0 * kTolEps * s.tnorm;
        int cs = 0;
        for (int i = 0; i < nwant; ++i) {
            if (i > 0 && s.lam[i] - s.lam[i - 1] > cluster) cs = i;
            s.cstart[i] = cs;
            double sh = s.lam[i];
            if (i > cs && sh - s.shift[i - 1] < sep) sh = s.shift[i - 1] + sep;
            s.shift[i] = sh;
        }
    }
    __syncthreads();

    // ---- 3. inverse iteration, one lane per eigenvector --------------------------------
    // (the recurrences carry their running values in registers, four rows per pass with the
    // pass's loads ahead of its stores; LDS holds U and z)
    if (t < nwant) {
        double* ui = s.inv.ui[t];
        double* u1 = s.inv.u1[t];
        double* u2 = s.inv.u2[t];
        double* z = s.z[t];
        const double lam = s.shift[t];
        const double eps = DBL_EPSILON * fmax(s.tnorm, DBL_MIN);
        auto guard = [&](double x) { return (fabs(x) < eps) ? (x < 0.0 ? -eps : eps) : x; };
        unsigned sd = static_cast<unsigned>(t + 1) * 2654435761u + 12345u;
        // the recurrences run over mp = 4 j + 1 >= m rows: the ones past m are decoupled (zero
        // off-diagonal, diagonal away from the shifts) and start at zero
        const int mp = ((m + 2) & ~3) + 1;
        for (int i = 0; i < mp; ++i) {
            sd = sd * 1664525u + 1013904223u;
            z[i] = i < m ? 0.5 + (sd >> 8) * (1.0 / 16777216.0) : 0.0;
        }
        double scale = 1.0;  // the previous solve's normalisation, applied on the way in
        // a solve whose growth |(T - lam I)^-1 z| reaches 1 / (64 sqrt(m) eps |T|), eps the
        // working accuracy, has converged (the test of LAPACK dstein); one more solve follows
        // it, at most four
        const double grow = 1.0 / (64.0 * sqrt(static_cast<double>(m)) * kTolEps * fmax(s.tnorm, DBL_MIN));
        int extra = -1;
        for (int it = 0; it < 4 && extra != 0; ++it) {
            // LU with partial pivoting of T - lam I (pending row: alpha at i, beta at i + 1)
            // and L y = z by the same row operations
            double alpha = s.d[0] - lam, beta = s.e[0];
            double cur = z[0] * scale;
            for (int i0 = 0; i0 + 1 < mp; i0 += 4) {
                double nz[4], sb[4], nd[4], ns[4], out[4], oi[4], o1[4], o2[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    nz[u] = z[i0 + u + 1] * scale;
                    sb[u] = s.e[i0 + u];
                    nd[u] = s.d[i0 + u + 1] - lam;
                    ns[u] = s.e[i0 + u + 1];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // the larger of the pending row's pivot and of the next row's leading entry
                    // becomes the pivot (a row exchange for the latter)
                    const bool swap = fabs(alpha) < fabs(sb[u]);
                    if (!swap) alpha = guard(alpha);
                    const double ip = recip(swap ? sb[u] : alpha);
                    const double mult = (swap ? alpha : sb[u]) * ip;
                    const double pz = swap ? nz[u] : cur;
                    oi[u] = ip;
                    o1[u] = swap ? nd[u] : beta;
                    o2[u] = swap ? ns[u] : 0.0;
                    alpha = (swap ? beta : nd[u]) - mult * o1[u];
                    beta = swap ? -mult * ns[u] : ns[u];
                    out[u] = pz;
                    cur = (swap ? cur : nz[u]) - mult * pz;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    z[i0 + u] = out[u];
                    ui[i0 + u] = oi[u];
                    u1[i0 + u] = o1[u];
                    u2[i0 + u] = o2[u];
                }
            }
            // U x = y from the last row, the two following entries in registers
            double z1 = cur * recip(guard(alpha)), z2 = 0.0, nrm = z1 * z1;
            z[mp - 1] = z1;
            for (int i0 = mp - 2; i0 >= 0; i0 -= 4) {
                double yy[4], a1[4], a2[4], ia[4], out[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    yy[u] = z[i0 - u];
                    a1[u] = u1[i0 - u];
                    a2[u] = u2[i0 - u];
                    ia[u] = ui[i0 - u];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const double zi = fma(-a1[u], z1, fma(-a2[u], z2, yy[u])) * ia[u];
                    out[u] = zi;
                    nrm = fma(zi, zi, nrm);
                    z2 = z1;
                    z1 = zi;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) z[i0 - u] = out[u];
            }
            if (!(nrm > 0.0)) {
                for (int i = 0; i < m; ++i) z[i] = (i == (t + 1) % m) ? 1.0 : 0.0;
                nrm = 1.0;
            }
            scale = 1.0 / sqrt(nrm);
            if (extra > 0) --extra;
            if (extra < 0 && sqrt(nrm) >= grow) extra = 1;
        }
        for (int i = 0; i < m; ++i) z[i] *= scale;
    }
    __syncthreads();
    // modified Gram-Schmidt inside clusters (wave 0; entries lane and lane + 64)
    if (w == 0) {
        for (int i = 1; i < nwant; ++i) {
            const int cs = s.cstart[i];
            if (cs == i) continue;
            double* zi = s.z[i];
            const bool ia = lane < m, ib = lane + 64 < m;
            for (int j = cs; j < i; ++j) {
                const double* zj = s.z[j];
                double dp = 0.0;
                if (ia) dp += zj[lane] * zi[lane];
                if (ib) dp += zj[lane + 64] * zi[lane + 64];
                dp = wave_sum(dp);
                if (ia) zi[lane] -= dp * zj[lane];
                if (ib) zi[lane + 64] -= dp * zj[lane + 64];
                wave_lds_fence();
            }
            double nn = 0.0;
            if (ia) nn += zi[lane] * zi[lane];
            if (ib) nn += zi[lane + 64] * zi[lane + 64];
            nn = wave_sum(nn);
            const double in = nn > 0.0 ? 1.0 / sqrt(nn) : 0.0;
            if (ia) zi[lane] *= in;
            if (ib) zi[lane + 64] *= in;
            wave_lds_fence();
        }
    }
    __syncthreads();

    // ---- 4. back-transformation ------------------------------------------------------
    if (m <= 32) back_transform<TR, 2>(s, m, nwant, refl, theta, Y, ldy);
    else if (m <= 64) back_transform<TR, 4>(s, m, nwant, refl, theta, Y, ldy);
    else if (m <= 96) back_transform<TR, 6>(s, m, nwant, refl, theta, Y, ldy);
    else back_transform<TR, 8>(s, m, nwant, refl, theta, Y, ldy);
}

}  // namespace

int projected_eigen_max_dim() { return kEM; }
int projected_eigen_max_want() { return kEWant; }

void launch_projected_eigen(const double2* T, int ldt, int m, int nwant, double2* refl, double* theta, double2* Y,
                            int ldy, bool fp32_reduction, unsigned long long* stamp, hipStream_t s) {
    if (m < 1 || m > kEM || nwant < 1 || nwant > kEWant || nwant > m || ldt < m || ldy < m)
        throw Error(XATU_ERR_INVALID_ARGUMENT, "projected eigensolver: unsupported dimensions");
    if (fp32_reduction) {
        hipLaunchKernelGGL(projected_eigen_kernel<float>, dim3(1), dim3(kEThreads), 0, s, T, ldt, m, nwant,
                           reinterpret_cast<float2*>(refl), theta, Y, ldy, stamp);
    } else {
        hipLaunchKernelGGL(projected_eigen_kernel<double>, dim3(1), dim3(kEThreads), 0, s, T, ldt, m, nwant, refl,
                           theta, Y, ldy, stamp);
    }
    XATU_HIP(hipGetLastError());
}

}  // namespace xatu_dev
