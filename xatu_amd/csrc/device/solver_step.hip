// The vector kernels of one iteration of the device Davidson solver, fused so that an
// iteration is few launches: at N = 900 an iteration is bound by the launches and by the
// host's share of it, not by its arithmetic (22 launches -> 14; 330 -> 270 us an iteration with
// what the host did in it, 25 x 25 with the convolution product 140 -> 100 us).
//   ritz_block_kernel   X = V Y, AX = W Y, residual norms, preconditioned corrections, restart
//                       (was two products, residual, precondition, two copies and a restart
//                       kernel; reads V and W once, stores no residuals)
//   whiten_kernel       S with (T S)^H (T S) = 1 from the corrections' Gram matrix (was on the host,
//                       between two waits)
//   whiten_apply_kernel T = T S in place (was a product to a scratch block and a copy), and the
//                       iteration's report to the host
// The kernels also leave the device's clock at their start, which times the phases without
// events: an event between two kernels keeps the second from starting for several microseconds.
#include "context.hpp"
#include "cplx.hpp"
#include "solver_step.hpp"
#include "wave_sums.hpp"

#include <algorithm>

namespace xatu_dev {

namespace {

constexpr int kCols = 4;           // columns per wave
constexpr int kRows = 64;          // rows per workgroup

__device__ inline double2 cscale(double2 a, double s) { return mk(a.x * s, a.y * s); }
__device__ inline unsigned long long device_clock() { return wall_clock64(); }

// Four uniform entries of row k of a small matrix (scalar loads); a column past nb repeats the
// last one present and is not stored.
__device__ inline void load_coefs(const double2* __restrict__ B, int ld, int k, int jn, double2 (&b)[kCols]) {
#pragma unroll
    for (int j = 0; j < kCols; ++j) b[j] = B[k + static_cast<int64_t>(min(j, jn - 1)) * ld];
}

// One row per lane, kCols columns per wave, ceil(b / kCols) waves. partial[j blocks + block] =
// sum of |r_j|^2 over the block's rows. T: nb <= b columns, r_j / (theta_j - d) with the denominator
// kept away from zero (nb = 0: none). restart: V and W begin with X and AX afterwards and
// the projected matrix Tm with diag(theta); T may then lie in the columns of V that were read,
// so every store waits for the loads of all the workgroup's waves.
// Bound by reading V and W once (HBM) when N is large, by the latency of a lane's m loads of both when it is
// small, hence eight columns of both in flight (N = 900, block 16, basis 16 to 64: 28 us of separate
// kernels -> 13 us; coefficients passed as a restricted pointer so that they are scalar loads, else 28).
__global__ __launch_bounds__(64 * kStepMaxBlock / kCols) __attribute__((amdgpu_waves_per_eu(2, 4))) void ritz_block_kernel(
    RitzBlockArgs a, const double2* __restrict__ Y) {
    const unsigned long long t0 = device_clock();
    const int lane = threadIdx.x & 63;
    const int cg = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kRows + lane;
    const bool ok = i < a.N;
    const int64_t ia = ok ? i : a.N - 1;  // rows past N load row N-1 and are not stored
    const int j0 = kCols * cg, jn = a.b - j0;
    double2 x[kCols], w[kCols];
#pragma unroll
    for (int j = 0; j < kCols; ++j) x[j] = w[j] = mk(0.0, 0.0);
    {
        const double2* Yc = Y + static_cast<int64_t>(j0) * a.m;
        const double2 *v = a.V + ia, *av = a.W + ia;
        constexpr int U = 8;
        int k = 0;
        for (; k + U <= a.m; k += U) {
            double2 vk[U], wk[U];
#pragma unroll
            for (int q = 0; q < U; ++q) {
                vk[q] = v[static_cast<int64_t>(k + q) * a.N];
                wk[q] = av[static_cast<int64_t>(k + q) * a.N];
            }
#pragma unroll
            for (int q = 0; q < U; ++q) {
                double2 y[kCols];
                load_coefs(Yc, a.m, k + q, jn, y);
#pragma unroll
                for (int j = 0; j < kCols; ++j) {
                    cfma(x[j], vk[q], y[j]);
                    cfma(w[j], wk[q], y[j]);
                }
            }
        }
        for (; k < a.m; ++k) {
            const double2 vk = v[static_cast<int64_t>(k) * a.N], wk = av[static_cast<int64_t>(k) * a.N];
            double2 y[kCols];
            load_coefs(Yc, a.m, k, jn, y);
#pragma unroll
            for (int j = 0; j < kCols; ++j) {
                cfma(x[j], vk, y[j]);
                cfma(w[j], wk, y[j]);
            }
        }
    }
    const double d = a.diag[ia];
    double theta[kCols];
#pragma unroll
    for (int j = 0; j < kCols; ++j) theta[j] = a.theta[j0 + min(j, jn - 1)];
    if (a.restart) __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x == 0) a.stamps[kStampRitz] = t0;
#pragma unroll
    for (int j = 0; j < kCols; ++j) {
        if (j < jn) {
            const int jj = j0 + j;
            const double th = theta[j];
            const double2 r = mk(w[j].x - th * x[j].x, w[j].y - th * x[j].y);
            double s = ok ? r.x * r.x + r.y * r.y : 0.0;
            s = wave_sum(s);
            if (lane == 0) a.partial[static_cast<int64_t>(jj) * gridDim.x + blockIdx.x] = s;
            if (ok) {
                const int64_t at = i + static_cast<int64_t>(jj) * a.N;
                a.X[at] = x[j];
                a.AX[at] = w[j];
                if (a.restart) {
                    a.V[at] = x[j];
                    a.W[at] = w[j];
                }
                if (jj < a.nb) {
                    double den = th - d;
                    if (fabs(den) < 1e-3) den = (den >= 0.0) ? 1e-3 : -1e-3;
                    a.T[at] = mk(r.x / den, r.y / den);
                }
            }
        }
    }
    if (a.restart && blockIdx.x == 0) {
        for (int e = threadIdx.x; e < a.b * a.b; e += blockDim.x) {
            const int p = e % a.b, q = e / a.b;
            a.Tm[p + static_cast<int64_t>(q) * a.ldt] = mk(p == q ? a.theta[p] : 0.0, 0.0);
        }
    }
}

// One workgroup of 256. With P the rows of the block in its Gram matrix (ld ldp, nb <= 32 columns):
// D^2 = 1 / diag P, G = D P D = L L^H, S = D L^-H, if every pivot^2 of G is above 1e-6 (cond(G)
// stays below ~1e6); else *flag = 0 and the caller orthonormalises the block another way. The
// factorisation and the inverse go on together in one nb x nb array, one column of G turning
// into one of L^-1 per step, four entries per thread in registers, the step's row and column
// exchanged through LDS with one barrier. Bound by the latency of these nb steps: 15 us for 16.
__global__ __launch_bounds__(256) void whiten_kernel(WhitenArgs a) {
    __shared__ double2 s_col[2][32], s_row[2][32];
    __shared__ double s_d[32];
    const unsigned long long t0 = device_clock();
    const int i = threadIdx.x & 31, c0 = threadIdx.x >> 5;
    if (threadIdx.x < a.nb) {
        const double g = a.P[threadIdx.x + static_cast<int64_t>(threadIdx.x) * a.ldp].x;
        s_d[threadIdx.x] = g > 0.0 ? 1.0 / sqrt(g) : 0.0;
    }
    __syncthreads();
    double2 e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = c0 + 8 * q;
        e[q] = mk(0.0, 0.0);
        if (i < a.nb && c < a.nb) e[q] = cscale(a.P[i + static_cast<int64_t>(c) * a.ldp], s_d[i] * s_d[c]);
    }
    bool good = true;
    for (int j = 0; j < a.nb; ++j) {
        double2 *col = s_col[j & 1], *row = s_row[j & 1];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = c0 + 8 * q;
            if (c == j) col[i] = e[q];
            if (i == j) row[c] = e[q];
        }
        __syncthreads();
        const double d = col[j].x;
        if (!(d > 1e-6)) {
            good = false;
            break;
        }
        const double inv = rsqrt(d);
        const double2 li = cscale(col[i], inv);
        double2 cc[4], rc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            cc[q] = col[c0 + 8 * q];
            rc[q] = row[c0 + 8 * q];
        }
        // selections instead of branches: they would leave one LDS latency after the other
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = c0 + 8 * q;
            // row j of L^-1 left of column j, its diagonal at j, conjugated column j of L right of it
            // (component by component: selections of whole structures went through scratch memory)
            const double fx = c == j ? inv : (c < j ? rc[q].x : cc[q].x) * inv;
            const double fy = c == j ? 0.0 : (c < j ? rc[q].y : -cc[q].y) * inv;
            const double bx = (c == j ? 0.0 : e[q].x) - (li.x * fx - li.y * fy);
            const double by = (c == j ? 0.0 : e[q].y) - (li.x * fy + li.y * fx);
            const bool pivot = i == j && c <= j;
            e[q].x = i > j ? bx : pivot ? fx : e[q].x;
            e[q].y = i > j ? by : pivot ? fy : e[q].y;
        }
    }
    if (good) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = c0 + 8 * q;
            // S[c, i] = D_c conj(L^-1[i, c]), c <= i
            if (i < a.nb && c < a.nb)
                a.S[c + static_cast<int64_t>(i) * a.nb] = c <= i ? cscale(cconj(e[q]), s_d[c]) : mk(0.0, 0.0);
        }
    }
    if (threadIdx.x == 0) {
        *a.flag = good ? 1 : 0;
        a.stamps[kStampWhiten] = t0;
    }
}

// T = T S in place unless the whitening failed: a workgroup holds its 64 rows in registers
// before any wave stores. The workgroup after those of the rows writes the report. A store to the
// host takes some ten microseconds to be acknowledged and a kernel's end waits for it, so it stands
// here, beside the host's own reaction to it, and needs no second store that says it is complete:
// each value has its check beside it (solver_step.hpp). (Written by the whitening kernel with
// the sequence number behind a fence it held up the stream for 20 us.)
__global__ __launch_bounds__(64 * kStepMaxBlock / kCols) void whiten_apply_kernel(WhitenArgs a, const double2* __restrict__ S) {
    if (blockIdx.x == gridDim.x - 1) {
        for (int t = threadIdx.x; t < kReportEntries; t += blockDim.x) {
            unsigned long long v = 0;
            if (t < kStepMaxBlock) {
                if (t < a.b) v = __double_as_longlong(a.theta[t]);
            } else if (t < 2 * kStepMaxBlock) {
                if (t - kStepMaxBlock < a.b) v = __double_as_longlong(a.norm2[t - kStepMaxBlock]);
            } else if (t < 2 * kStepMaxBlock + kStamps) {
                v = a.stamps[t - 2 * kStepMaxBlock];
            } else {
                v = *a.flag;
            }
            a.host->entry[t] = make_ulonglong2(v, v ^ a.sequence);
        }
        return;
    }
    if (*a.flag) {
        const int lane = threadIdx.x & 63;
        const int cg = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
        const int64_t i = static_cast<int64_t>(blockIdx.x) * kRows + lane;
        const int64_t ia = i < a.N ? i : a.N - 1;
        const int j0 = kCols * cg, jn = a.nb - j0;
        double2 acc[kCols];
#pragma unroll
        for (int j = 0; j < kCols; ++j) acc[j] = mk(0.0, 0.0);
        if (jn > 0) {
#pragma unroll 8
            for (int k = 0; k < a.nb; ++k) {
                const double2 t = a.T[ia + static_cast<int64_t>(k) * a.N];
                double2 y[kCols];
                load_coefs(S + static_cast<int64_t>(j0) * a.nb, a.nb, k, jn, y);
#pragma unroll
                for (int j = 0; j < kCols; ++j) cfma(acc[j], t, y[j]);
            }
        }
        __syncthreads();
        if (i < a.N) {
#pragma unroll
            for (int j = 0; j < kCols; ++j)
                if (j < jn) a.T[i + static_cast<int64_t>(j0 + j) * a.N] = acc[j];
        }
    }
}

unsigned step_blocks(int64_t N) { return static_cast<unsigned>((N + kRows - 1) / kRows); }
unsigned step_threads(int b) { return 64 * ((b + kCols - 1) / kCols); }

}  // namespace

int ritz_block_partials(int64_t N) { return static_cast<int>(step_blocks(N)); }

void launch_ritz_block(const RitzBlockArgs& a, hipStream_t s) {
    if (a.b < 1 || a.b > kStepMaxBlock || a.nb < 0 || a.nb > a.b || a.m < 1)
        throw Error(XATU_ERR_INVALID_ARGUMENT, "Ritz block: unsupported dimensions");
    hipLaunchKernelGGL(ritz_block_kernel, dim3(step_blocks(a.N)), dim3(step_threads(a.b)), 0, s, a, a.Y);
    XATU_HIP(hipGetLastError());
}

void launch_whiten(const WhitenArgs& a, hipStream_t s) {
    if (a.nb < 0 || a.nb > kStepMaxBlock || a.b > kStepMaxBlock)
        throw Error(XATU_ERR_INVALID_ARGUMENT, "whitening: unsupported dimensions");
    hipLaunchKernelGGL(whiten_kernel, dim3(1), dim3(256), 0, s, a);
    // without a block only the report's workgroup
    hipLaunchKernelGGL(whiten_apply_kernel, dim3(a.nb > 0 ? step_blocks(a.N) + 1 : 1), dim3(step_threads(std::max(a.nb, 1))),
                       0, s, a, a.S);
    XATU_HIP(hipGetLastError());
}

}  // namespace xatu_dev
