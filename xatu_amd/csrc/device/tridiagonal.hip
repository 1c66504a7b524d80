// Reduction of a dense Hermitian matrix to a real tridiagonal one, A = Q T Q^H, for the full
// diagonalisation of small operators. Reflectors H_j = 1 - tau_j v_j v_j^H, Q = H_0 H_1 ..., with v_j zero up to
// row j, one in row j + 1 and its remaining rows stored below that in column j of R (the
// storage that the library's back-transformation takes).
//
// The reduction is a chain of n steps with little work in each (n = 400: 2.5 MB, which stay in
// the last-level cache), so it is bound by what a step costs in launches and latency: the
// library takes five to six kernels per column. Here a step is one kernel: every workgroup
// repeats the small part for itself (the rank-2 update's second vector from the last product, the updated
// column, its reflector) and then, for its own columns, applies the update and multiplies by
// the new reflector in one pass over the column. The loads of the columns are issued before
// the small part. A column always belongs to the same workgroup number, hence to the same XCD's L2.
// n = 400: 5.0 us a step (5.5 with the sums over a wave by shuffles instead of DPP), the reduction about
// 8 -> 2.0 ms; all eigenpairs with apply_reflectors_kernel 10.8 -> 4.1 ms, n = 1024 28.6 -> 12.7, n = 2025 68
// -> 45 ms. A lane keeps its rows of a column in registers, which ends at
// 32 (n = 2048; a step then moves 64 MB through the last-level cache and costs as much as the library's).
#include "context.hpp"
#include "cplx.hpp"
#include "wave_sums.hpp"

namespace xatu_dev {

namespace {

// Step j. v (column j - 1 of R with its unit entry) and p = A v of step j - 1 give w = tau p -
// (tau / 2) (tau p)^H v v; A <- A - v w^H - w v^H on rows and columns j and above; column j then gives D[j],
// reflector j, E[j], tau[j]; next = A v_j. Q: rows per lane, n <= 64 Q. Wave per column, grid ceil(n / WAVES).
// The workgroup of the last column stores the step's results.
template <int Q, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void tridiagonal_step_kernel(double2* __restrict__ A, int n, int j,
                                                                      const double2* __restrict__ p,
                                                                      double2* __restrict__ next,
                                                                      double2* __restrict__ R,
                                                                      double2* __restrict__ tau,
                                                                      double* __restrict__ D, double* __restrict__ E) {
    constexpr int kThreads = 64 * WAVES;
    constexpr int K = 64 * Q / kThreads;  // rows per thread of the small part
    __shared__ double2 s_v[64 * Q], s_w[64 * Q], s_n[64 * Q];
    __shared__ double s_red[2][WAVES][2];
    __shared__ double2 s_alpha;
    const int c = blockIdx.x * WAVES + (threadIdx.x >> 6);
    const bool last = blockIdx.x == gridDim.x - 1;
    if (static_cast<int>((blockIdx.x + 1) * WAVES) <= j + 1 && !last) return;  // all columns done
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool mine = c > j && c < n;

    double2 col[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = lane + 64 * q;
        col[q] = mk(0.0, 0.0);
        if (mine && r > j && r < n) col[q] = A[r + static_cast<int64_t>(c) * n];
    }
    double2 v[K], w[K], a[K];
    double sr = 0.0, si = 0.0;
    const double2 tp = j > 0 ? tau[j - 1] : mk(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int r = threadIdx.x + kThreads * k;
        v[k] = w[k] = a[k] = mk(0.0, 0.0);
        if (r >= j && r < n) {
            a[k] = A[r + static_cast<int64_t>(j) * n];
            if (j > 0) {
                v[k] = r == j ? mk(1.0, 0.0) : R[r + static_cast<int64_t>(j - 1) * n];
                w[k] = p[r];
            }
        }
        sr += w[k].x * v[k].x + w[k].y * v[k].y;  // conj(p) v
        si += w[k].x * v[k].y - w[k].y * v[k].x;
    }
    if (j > 0) {
        sr = wave_sum(sr);
        si = wave_sum(si);
        if (lane == 0) {
            s_red[0][wave][0] = sr;
            s_red[0][wave][1] = si;
        }
        __syncthreads();
        sr = si = 0.0;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) {
            sr += s_red[0][k][0];
            si += s_red[0][k][1];
        }
        // -(tau / 2) conj(tau) (p^H v)
        const double h = -0.5 * (tp.x * tp.x + tp.y * tp.y);
        const double2 f = mk(h * sr, h * si);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double2 x = cmul(tp, w[k]);
            cfma(x, f, v[k]);
            w[k] = x;
            const int r = threadIdx.x + kThreads * k;
            if (r < n) {
                s_v[r] = v[k];
                s_w[r] = w[k];
            }
        }
        __syncthreads();
        const double2 wj = s_w[j];  // v_j is one
#pragma unroll
        for (int k = 0; k < K; ++k) a[k] = csub(csub(a[k], cmul(v[k], cconj(wj))), w[k]);
    }
    // reflector of the updated column: beta real with H^H (alpha, x) = (beta, 0)
    double norm = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int r = threadIdx.x + kThreads * k;
        if (r >= j + 2 && r < n) norm += a[k].x * a[k].x + a[k].y * a[k].y;
        if (r == j + 1 && r < n) s_alpha = a[k];
        if (r == j && last) D[j] = a[k].x;
    }
    norm = wave_sum(norm);
    if (lane == 0) s_red[1][wave][0] = norm;
    __syncthreads();
    if (j + 1 >= n) return;
    norm = 0.0;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) norm += s_red[1][k][0];
    double2 alpha = s_alpha;
    double back = 1.0;  // from the units of the reflector's scalars to the matrix's
    const double sum = alpha.x * alpha.x + alpha.y * alpha.y + norm;
    if (__builtin_expect(!(sum > 1e-280 && sum < 1e280), 0)) {
        // squares that left the normal numbers (or nothing but zeros): the column in units of a power of two
        // near its largest entry. The whole workgroup comes here or none of it.
        double most = fmax(fabs(alpha.x), fabs(alpha.y));
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int r = threadIdx.x + kThreads * k;
            if (r >= j + 2 && r < n) most = fmax(most, fmax(fabs(a[k].x), fabs(a[k].y)));
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) most = fmax(most, __shfl_xor(most, d));
        if (lane == 0) s_red[0][wave][0] = most;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < WAVES; ++k) most = fmax(most, s_red[0][k][0]);
        double unit = 1.0;
        if (most > 0.0) {
            const int ex = max(-1000, min(1000, ilogb(most)));
            unit = ldexp(1.0, -ex);
            back = ldexp(1.0, ex);
        }
        norm = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int r = threadIdx.x + kThreads * k;
            a[k] = mk(a[k].x * unit, a[k].y * unit);
            if (r >= j + 2 && r < n) norm += a[k].x * a[k].x + a[k].y * a[k].y;
        }
        norm = wave_sum(norm);
        if (lane == 0) s_red[1][wave][0] = norm;
        __syncthreads();
        norm = 0.0;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) norm += s_red[1][k][0];
        alpha = mk(alpha.x * unit, alpha.y * unit);
    }
    double beta = alpha.x;
    double2 t = mk(0.0, 0.0), scale = mk(0.0, 0.0);
    if (norm > 0.0 || alpha.y != 0.0) {
        const double len = sqrt(alpha.x * alpha.x + alpha.y * alpha.y + norm);
        beta = alpha.x >= 0.0 ? -len : len;
        t = mk((beta - alpha.x) / beta, -alpha.y / beta);
        const double2 d = mk(alpha.x - beta, alpha.y);  // |d| >= len
        const double inv = 1.0 / (d.x * d.x + d.y * d.y);
        scale = mk(d.x * inv, -d.y * inv);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int r = threadIdx.x + kThreads * k;
        if (r < n) {
            const double2 x = r > j + 1 ? cmul(a[k], scale) : mk(r == j + 1 ? 1.0 : 0.0, 0.0);
            s_n[r] = x;
            if (last && r > j + 1) R[r + static_cast<int64_t>(j) * n] = x;
        }
    }
    if (last && threadIdx.x == 0) {
        tau[j] = t;
        E[j] = beta * back;
    }
    __syncthreads();
    if (!mine) return;
    double pr = 0.0, pi = 0.0;
    const double2 vc = j > 0 ? s_v[c] : mk(0.0, 0.0), wc = j > 0 ? s_w[c] : mk(0.0, 0.0);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = lane + 64 * q;
        if (r > j && r < n) {
            double2 x = col[q];
            if (j > 0) {
                x = csub(csub(x, cmul(s_v[r], cconj(wc))), cmul(s_w[r], cconj(vc)));
                A[r + static_cast<int64_t>(c) * n] = x;
            }
            const double2 y = s_n[r];
            pr += x.x * y.x + x.y * y.y;  // conj(A(r, c)) v(r) = A(c, r) v(r)
            pi += x.x * y.y - x.y * y.x;
        }
    }
    pr = wave_sum(pr);
    pi = wave_sum(pi);
    if (lane == 0) next[c] = mk(pr, pi);
}

// C <- Q C: a wave holds one column of C in registers and applies the reflectors to it from the last
// one on, each as a dot product over the wave and an update; the next few reflectors are on their way
// meanwhile. Bound by that chain, 0.5 us a reflector, while the reflectors, which every wave
// reads, come from the caches: n = 400 1.3 ms by the library's blocked products -> 0.21 (0.38 with
// one reflector ahead and branches around the finished rows). To n = 1024, where all of them are 16 MB.
template <int Q>
__global__ __launch_bounds__(256) void apply_reflectors_kernel(const double2* __restrict__ R,
                                                               const double2* __restrict__ tau, int n,
                                                               double2* __restrict__ C) {
    const int lane = threadIdx.x & 63;
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (c >= n) return;
    double2* col = C + static_cast<int64_t>(c) * n;
    constexpr int D = 4;  // reflectors in flight
    double2 x[Q], v[D][Q], t[D];
    // without branches, so that the loads of several reflectors can be counted: R is zero where no
    // reflector is stored
    auto load = [&](double2 (&dst)[Q], double2& tj, int j) {
        const int64_t jj = j < 0 ? 0 : j;
        tj = tau[jj];
#pragma unroll
        for (int q = 0; q < Q; ++q) dst[q] = R[min(lane + 64 * q, n - 1) + jj * n];
    };
    auto apply = [&](double2 (&u)[Q], double2 tj, int j) {
        double sr = 0.0, si = 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int r = lane + 64 * q;
            const bool in = r < n;
            u[q].x = r == j + 1 ? 1.0 : in ? u[q].x : 0.0;
            u[q].y = in ? u[q].y : 0.0;  // zero at j + 1
            sr += u[q].x * x[q].x + u[q].y * x[q].y;  // conj(v) x
            si += u[q].x * x[q].y - u[q].y * x[q].x;
        }
        const double2 f = cmul(tj, mk(wave_sum(sr), wave_sum(si)));
#pragma unroll
        for (int q = 0; q < Q; ++q) x[q] = csub(x[q], cmul(f, u[q]));
    };
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = lane + 64 * q;
        x[q] = r < n ? col[r] : mk(0.0, 0.0);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d) load(v[d], t[d], n - 2 - d);
    int j = n - 2;
    for (; j >= D - 1; j -= D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(v[(d + D - 1) % D], t[(d + D - 1) % D], j - d - (D - 1));
            apply(v[d], t[d], j - d);
        }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (j - d >= 0) apply(v[d], t[d], j - d);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = lane + 64 * q;
        if (r < n) col[r] = x[q];
    }
}

template <int Q, int WAVES>
void run_steps(double2* A, int n, double2* p, double2* R, double2* tau, double* D, double* E, hipStream_t s) {
    const unsigned grid = (n + WAVES - 1) / WAVES;
    for (int j = 0; j < n; ++j)
        hipLaunchKernelGGL((tridiagonal_step_kernel<Q, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, A, n, j,
                           p + static_cast<size_t>(n) * (j & 1), p + static_cast<size_t>(n) * (1 - (j & 1)), R, tau, D, E);
}

}  // namespace

int tridiagonal_max_dim() { return 2048; }
int reflectors_max_dim() { return 1024; }

void launch_apply_reflectors(const double2* R, const double2* tau, int n, double2* C, hipStream_t s) {
    if (n < 2 || n > reflectors_max_dim()) throw Error(XATU_ERR_INVALID_ARGUMENT, "reflectors: unsupported dimension");
    const dim3 grid((n + 3) / 4), block(256);
    if (n <= 256) hipLaunchKernelGGL((apply_reflectors_kernel<4>), grid, block, 0, s, R, tau, n, C);
    else if (n <= 512) hipLaunchKernelGGL((apply_reflectors_kernel<8>), grid, block, 0, s, R, tau, n, C);
    else hipLaunchKernelGGL((apply_reflectors_kernel<16>), grid, block, 0, s, R, tau, n, C);
    XATU_HIP(hipGetLastError());
}

void launch_tridiagonal(double2* A, int n, double2* p, double2* R, double2* tau, double* D, double* E, hipStream_t s) {
    if (n < 1 || n > tridiagonal_max_dim()) throw Error(XATU_ERR_INVALID_ARGUMENT, "tridiagonal reduction: unsupported dimension");
    if (n <= 256) run_steps<4, 4>(A, n, p, R, tau, D, E, s);
    else if (n <= 512) run_steps<8, 4>(A, n, p, R, tau, D, E, s);
    else if (n <= 1024) run_steps<16, 4>(A, n, p, R, tau, D, E, s);
    else run_steps<32, 8>(A, n, p, R, tau, D, E, s);
    XATU_HIP(hipGetLastError());
}

}  // namespace xatu_dev
