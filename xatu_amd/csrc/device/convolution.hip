// Matrix-free BSE products by k-space convolution.
//
// The direct term of the reference's matrix (src/ExcitonTB.cpp:520-548, 840-921),
//   D(kcv, k'c'v') = sum_ab rho^c_a M_ab(k'-k) rho^v_b,
//   rho^c_a = sum_{al in a} conj(C_kc,al) C_k'c',al,  rho^v_b = sum_{be in b} conj(V_k'v',be) V_kv,be,
// depends on the pair (k, k') only through the lattice-sum table M(k'-k), so its
// product with a vector factorises:
//   z_{al be}(k')  = sum_{c'v'} C_k'c',al conj(V_k'v',be) x(k'c'v')
//   w_{al be}(k)   = sum_k' M_{a(al) b(be)}(k'-k) z_{al be}(k')        (a correlation on the mesh)
//   (D x)(kcv)     = sum_{al be} conj(C_kc,al) V_kv,be w_{al be}(k).
// The correlation is evaluated with FFTs on the mesh of the lattice sums (mesh_n points
// per axis; k-points sit at their integer offsets, so reduced and shifted meshes work
// unchanged): w = IFFT( P_ab . FFT(z) ) with P_ab the backward transform of the table
// M_ab(Delta) = ft[q(Delta)] (q the same mesh index the assembly uses), scaled by 1/mesh.
// Cost per vector: norb^2 FFT pairs of mesh size plus O(nk norb^2 nc) contractions,
// instead of O(nk^2) pair evaluations for a recomputed tile.
//
// Off the diagonal the reference fills only the upper triangle and mirrors it. The
// direct formula is Hermitian under the exchange of the pair because the table obeys
// M(-q) = conj M(q) (including the conjugated diagonal the reference stores), so the
// full correlation equals the mirrored matrix up to rounding. The exchange term
// X(i,j) = sum_a E1_a(i) E2_a(j) is not Hermitian when V(Q) has a complex diagonal, so
// it follows the triangle: (X_tri x)_i = sum_a [E1_a(i) sum_{j>i} E2_a(j) x_j
// + conj(E2_a(i)) sum_{j<i} conj(E1_a(j)) x_j] + Re(sum_a E1_a(i) E2_a(i)) x_i, with the
// partial sums from a blocked scan in a fixed order. The diagonal energies enter as
// e_i x_i, so H x = e x - D x + X_tri x exactly as the assembled matrix.
//
// FFTs: on 2-D meshes with sides A B (fft_stages.hpp) the row and column kernels of
// conv_rows.hpp, which never store z or w on the mesh; otherwise rocFFT (batched, in place,
// interleaved complex; plans cached per precision and batch size). The exchange part runs in
// FP64 for both precisions.
#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include <rocfft/rocfft.h>

#include "context.hpp"
#include "conv_rows.hpp"
#include "cplx.hpp"
#include "mfma.hpp"
#include "wave_sums.hpp"

#define XATU_FFT(call)                                                                                    \
    do {                                                                                                  \
        rocfft_status s_ = (call);                                                                        \
        if (s_ != rocfft_status_success) {                                                                \
            throw ::xatu_dev::Error(XATU_ERR_DEVICE,                                                      \
                                    std::string(#call) + ": rocfft status " + std::to_string(static_cast<int>(s_))); \
        }                                                                                                 \
    } while (0)

namespace xatu_dev {

namespace {

constexpr int kScanRows = 64;   // rows of one block of the exchange scans: a wave
constexpr int kScanWaves = 4;   // waves per workgroup of the scans

// Layout of the correlation buffer G (batch entries b of M mesh points g = o0 + mesh_n o1).
// Entry-major: G[b M + g]. Row-interleaved (2-D meshes): G[(o1 batch + b) mesh_n + o0],
// so that the FFTs along o0 (unit stride, rows of mesh_n) and along o1 (stride
// batch mesh_n, consecutive transforms adjacent) are each one uniform batched 1-D pass
// with no transposition between them.
struct GLayout {
    int64_t bstride;    // distance between consecutive batch entries
    int rowlen;         // 0: entry-major; mesh_n: row-interleaved
    int64_t rowstride;  // row-interleaved: batch mesh_n
    __device__ int64_t at(int64_t b, int g) const {
        return b * bstride + (rowlen ? static_cast<int64_t>(g / rowlen) * rowstride + g % rowlen : g);
    }
};

__device__ inline int atom_of(const LatticeDesc& lat, int orb) {
    int a = 0;
    while (a + 1 < lat.natoms && orb >= lat.orb_begin[a + 1]) ++a;
    return a;
}

// Mt[ab][g] = ft[q(g) NA^2 + ab], g = sum_j d_j m^j, q = sum_j ((d_j + m/2) mod m) m^j.
__global__ void table_grid_kernel(LatticeDesc lat, const double2* __restrict__ ft, double2* __restrict__ Mt) {
    const int64_t M = lat.nmesh;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int na2 = lat.natoms * lat.natoms;
    if (idx >= M * na2) return;
    const int ab = static_cast<int>(idx / M);
    int64_t g = idx % M;
    const int m = lat.mesh_n;
    int64_t q = 0, mul = 1;
    for (int j = 0; j < lat.ndim; ++j) {
        const int d = static_cast<int>(g % m);
        g /= m;
        q += static_cast<int64_t>((d + m / 2) % m) * mul;
        mul *= m;
    }
    Mt[idx] = ft[q * na2 + ab];
}

template <typename R>
__global__ void scale_spectrum_kernel(const double2* __restrict__ in, int64_t n, double scale, cx_t<R>* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) out[i] = mk(static_cast<R>(in[i].x * scale), static_cast<R>(in[i].y * scale));
}

// Kernel spectrum of the atom pair (a, b) on the window of the first axis, real:
// P[((a + NA b) n + xi_1) W + j] = sum of V_ab(R) / T over the cells R = -xi (a < b) or R = xi
// (a >= b) modulo the mesh, xi_0 = (w0 + j) mod n. head[xi_0 + n xi_1] is the first cell of a
// residue, next[R] the following one (-1: none).
template <typename R>
__global__ void window_spectrum_kernel(LatticeDesc lat, int W, int w0, const int* __restrict__ head,
                                       const int* __restrict__ next, int nR, const double* __restrict__ vtab,
                                       double inv_total, R* __restrict__ P) {
    const int n = lat.mesh_n;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<int64_t>(lat.natoms) * lat.natoms * n * W) return;
    const int j = static_cast<int>(idx % W);
    const int x1 = static_cast<int>((idx / W) % n);
    const int ab = static_cast<int>(idx / (static_cast<int64_t>(W) * n));
    const int a = ab % lat.natoms, b = ab / lat.natoms;
    int m0 = (w0 + j) % n, m1 = x1;
    if (a < b) {
        m0 = m0 ? n - m0 : 0;
        m1 = m1 ? n - m1 : 0;
    }
    const int lo = min(a, b), hi = max(a, b);
    const int p = lo * lat.natoms - lo * (lo - 1) / 2 + hi - lo;  // pairs (lo, hi >= lo), row by row
    double sum = 0.0;
    for (int r = head[m0 + n * m1]; r >= 0; r = next[r]) sum += vtab[static_cast<size_t>(p) * nR + r];
    P[idx] = static_cast<R>(sum * inv_total);
}

// Band stacks transposed for coalesced access across k: Ct[(c norb + al) nk + k] =
// C^{k+Q}_{nv+c}(k)[al] (conduction) and Vt[(v norb + be) nk + k] = C^{k}_{v}(k)[be] (valence).
template <typename R>
__global__ void transpose_stacks_kernel(int nk, int nv, int nc, int norb, const double2* __restrict__ evk,
                                        const double2* __restrict__ evkq, cx_t<R>* __restrict__ Ct,
                                        cx_t<R>* __restrict__ Vt) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int col = blockIdx.y;  // 0..nc*norb-1 conduction, then nv*norb valence
    if (k >= nk) return;
    const int nb = nv + nc;
    if (col < nc * norb) {
        const int c = col / norb, al = col % norb;
        const double2 v = evkq[(static_cast<size_t>(k) * nb + nv + c) * norb + al];
        Ct[static_cast<size_t>(col) * nk + k] = mk(static_cast<R>(v.x), static_cast<R>(v.y));
    } else {
        const int cv = col - nc * norb;
        const int v = cv / norb, be = cv % norb;
        const double2 w = evk[(static_cast<size_t>(k) * nb + v) * norb + be];
        Vt[static_cast<size_t>(cv) * nk + k] = mk(static_cast<R>(w.x), static_cast<R>(w.y));
    }
}

// orbitals al per thread in the z contraction: each group re-reads u (FP64 at 18 orbitals:
// 6 took the product's z step from 176 to 158 us against 4; FP32 at 36 orbitals: 12 made it
// slower, 1.92 against 1.77 ms, the G stores of more orbitals per thread outweighing the
// fewer passes over u)
template <typename R>
constexpr int conv_orb_group() { return sizeof(R) == 8 ? 6 : 4; }

// vectors per thread in the u and y contractions (register budget: FP64 halves it)
template <typename R>
constexpr int conv_vec_group() { return sizeof(R) == 8 ? 2 : 4; }
// vectors per thread of the y contraction: one, for enough threads to cover the latency of
// its norb^2 loads per vector (the band coefficients it re-reads hit the caches)
template <typename R>
constexpr int conv_y_group() { return 1; }
// orbitals be per pass over al in the y contraction (their partial sums stay in registers)
template <typename R>
constexpr int conv_y_be_block() { return sizeof(R) == 8 ? 6 : 12; }

// u[((n NC + c) norb + be) nk + k] = sum_v conj(V_k[be, v]) x[k NCV + c NV + v, n]
// thread per k, blockIdx.y = group of vectors; the device clock to stamp, if any
template <typename R, int NC, int NV>
__global__ __launch_bounds__(256) void conv_u_kernel(int nk, int norb, int nvec, const cx_t<R>* __restrict__ Vt,
                                                     const double2* __restrict__ X, int64_t N, cx_t<R>* __restrict__ U,
                                                     unsigned long long* __restrict__ stamp) {
    if (stamp && blockIdx.x + blockIdx.y == 0 && threadIdx.x == 0) *stamp = wall_clock64();
    constexpr int VG = conv_vec_group<R>();
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int n0 = blockIdx.y * VG;
    if (k >= nk) return;
    constexpr int ncv = NC * NV;
    cx_t<R> x[VG][NC][NV];
#pragma unroll
    for (int g = 0; g < VG; ++g)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int n = n0 + g;
                const double2 xv = n < nvec ? X[static_cast<size_t>(k) * ncv + c * NV + v + n * N] : mk(0.0, 0.0);
                x[g][c][v] = mk(static_cast<R>(xv.x), static_cast<R>(xv.y));
            }
    for (int be = 0; be < norb; ++be) {
        cx_t<R> vb[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) vb[v] = Vt[(static_cast<size_t>(v) * norb + be) * nk + k];
#pragma unroll
        for (int g = 0; g < VG; ++g) {
            const int n = n0 + g;
            if (n < nvec) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    cx_t<R> s = mk(R(0), R(0));
#pragma unroll
                    for (int v = 0; v < NV; ++v) cfma_conj(s, vb[v], x[g][c][v]);
                    U[((static_cast<size_t>(n) * NC + c) * norb + be) * nk + k] = s;
                }
            }
        }
    }
}

// G[entry (al norb + be) nvec + n][g(k)] = sum_c C_k[al, c] u[n][c][be][k]
// thread per k, blockIdx.y = group of conv_orb_group<R>() orbitals al, blockIdx.z = vector n
template <typename R, int NC>
__global__ __launch_bounds__(256) void conv_z_kernel(int nk, int norb, int nvec, GLayout lay, const int* __restrict__ gk,
                                                     const cx_t<R>* __restrict__ Ct, const cx_t<R>* __restrict__ U,
                                                     cx_t<R>* __restrict__ G) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    constexpr int AG = conv_orb_group<R>();
    const int al0 = blockIdx.y * AG;
    const int n = blockIdx.z;
    if (k >= nk) return;
    cx_t<R> Ca[AG][NC];
#pragma unroll
    for (int a = 0; a < AG; ++a)
#pragma unroll
        for (int c = 0; c < NC; ++c)
            Ca[a][c] = al0 + a < norb ? Ct[(static_cast<size_t>(c) * norb + al0 + a) * nk + k] : mk(R(0), R(0));
    const int g = gk[k];
    for (int be = 0; be < norb; ++be) {
        cx_t<R> ub[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) ub[c] = U[((static_cast<size_t>(n) * NC + c) * norb + be) * nk + k];
#pragma unroll
        for (int a = 0; a < AG; ++a) {
            if (al0 + a < norb) {
                cx_t<R> s = mk(R(0), R(0));
#pragma unroll
                for (int c = 0; c < NC; ++c) cfma(s, Ca[a][c], ub[c]);
                G[lay.at((static_cast<int64_t>(al0 + a) * norb + be) * nvec + n, g)] = s;
            }
        }
    }
}

// G[b][xi] *= P[a(al) + NA b(be)][xi], batch b = (al norb + be) nvec + n
template <typename R>
__global__ void conv_multiply_kernel(LatticeDesc lat, int nvec, int64_t M, GLayout lay, const cx_t<R>* __restrict__ P,
                                     cx_t<R>* __restrict__ G) {
    const int64_t xi = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int b = blockIdx.y;
    if (xi >= M) return;
    const int ab = b / nvec;
    const int al = ab / lat.norb, be = ab % lat.norb;
    const int pa = atom_of(lat, al) + lat.natoms * atom_of(lat, be);
    const int64_t i = lay.at(b, static_cast<int>(xi));
    G[i] = cmul(G[i], P[static_cast<int64_t>(pa) * M + xi]);
}

// Y[k NCV + c NV + v, n] = e(kcv) x - sum_be V_k[be, v] sum_al conj(C_k[al, c]) w[(al norb + be) nvec + n][g(k)]
// thread per k, blockIdx.y = group of vectors (the band coefficients are loaded once per group)
template <typename R, int NC, int NV>
__global__ __launch_bounds__(256) void conv_y_kernel(int nk, int norb, int nvec, GLayout lay, const int* __restrict__ gk,
                                                     const cx_t<R>* __restrict__ Ct, const cx_t<R>* __restrict__ Vt,
                                                     const double* __restrict__ eval_k, const double* __restrict__ eval_kq,
                                                     double scissor, const cx_t<R>* __restrict__ W,
                                                     const double2* __restrict__ X, int64_t N, double2* __restrict__ Y) {
    constexpr int VG = conv_y_group<R>();
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int n0 = blockIdx.y * VG;
    if (k >= nk) return;
    constexpr int nb = NV + NC, ncv = NC * NV;
    const int ng = min(VG, nvec - n0);
    const int g = gk[k];
    cx_t<R> acc[VG][NC][NV];
#pragma unroll
    for (int q = 0; q < VG; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[q][c][v] = mk(R(0), R(0));
    // BE orbitals be per pass over al, so that C_k[al, c] is loaded once per pass instead of
    // once per be; every t(be) = sum_al conj(C) w and acc += V t(be) keeps its order (al, then
    // be increasing), so the result does not depend on BE
    constexpr int BE = conv_y_be_block<R>();
    for (int be0 = 0; be0 < norb; be0 += BE) {
        const int nbe = min(BE, norb - be0);
        cx_t<R> t[VG][BE][NC];
#pragma unroll
        for (int q = 0; q < VG; ++q)
#pragma unroll
            for (int j = 0; j < BE; ++j)
#pragma unroll
                for (int c = 0; c < NC; ++c) t[q][j][c] = mk(R(0), R(0));
        for (int al = 0; al < norb; ++al) {
            cx_t<R> ca[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) ca[c] = Ct[(static_cast<size_t>(c) * norb + al) * nk + k];
#pragma unroll
            for (int j = 0; j < BE; ++j) {
                if (j < nbe) {
                    const cx_t<R>* w = W + lay.at((static_cast<int64_t>(al) * norb + be0 + j) * nvec + n0, g);
#pragma unroll
                    for (int q = 0; q < VG; ++q) {
                        if (q < ng) {
                            const cx_t<R> wq = w[q * lay.bstride];
#pragma unroll
                            for (int c = 0; c < NC; ++c) cfma_conj(t[q][j][c], ca[c], wq);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < BE; ++j) {
            if (j < nbe) {
                const int be = be0 + j;
                cx_t<R> vb[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) vb[v] = Vt[(static_cast<size_t>(v) * norb + be) * nk + k];
#pragma unroll
                for (int q = 0; q < VG; ++q)
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int v = 0; v < NV; ++v) cfma(acc[q][c][v], vb[v], t[q][j][c]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < VG; ++q) {
        if (q < ng) {
            const int n = n0 + q;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const int64_t row = static_cast<int64_t>(k) * ncv + c * NV + v;
                    const double e = (scissor + eval_kq[static_cast<size_t>(k) * nb + NV + c]) -
                                     eval_k[static_cast<size_t>(k) * nb + v];
                    const double2 x = X[row + n * N];
                    Y[row + n * N] = mk(e * x.x - static_cast<double>(acc[q][c][v].x),
                                        e * x.y - static_cast<double>(acc[q][c][v].y));
                }
        }
    }
}

// Y[k NCV + c NV + v, n] = e(kcv) x - sum_be V_k[be, v] t[n][c][be][k] with t the sum of the
// parts that conv_rows_out_kernel left (T[((part nvec + n) NC + c) norb + be][k]). grid (k, vector);
// S threads of a workgroup share a k-point, each with the orbitals be = its number modulo S, and their sums
// meet in LDS. Reads T once, so bound by HBM when there are many k-points and vectors (S = 1) and
// by the latency of the loads of one thread when there are few (S = kBandsShare; 25 x 25, 4 vectors,
// 18 orbitals, FP64: 76 -> 14 us; 48 x 48, 8 vectors, 8 orbitals: 20 -> 10 us).
constexpr int kBandsShare = 8;
template <typename R, int NC, int NV, int S>
__global__ __launch_bounds__(256) void conv_bands_y_kernel(int nk, int norb, int nvec, int parts,
                                                           const cx_t<R>* __restrict__ Vt,
                                                           const double* __restrict__ eval_k,
                                                           const double* __restrict__ eval_kq, double scissor,
                                                           const cx_t<R>* __restrict__ T,
                                                           const double2* __restrict__ X, int64_t N,
                                                           double2* __restrict__ Y) {
    constexpr int KB = 256 / S;
    __shared__ cx_t<R> sums[S > 1 ? S : 1][NV][S > 1 ? KB : 1];
    const int share = threadIdx.x / KB;
    const int k = blockIdx.x * KB + threadIdx.x % KB;
    const int n = blockIdx.y;
    const bool ok = k < nk;
    if (S == 1 && !ok) return;
    constexpr int nb = NV + NC, ncv = NC * NV;
    cx_t<R> acc[NC][NV];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[c][v] = mk(R(0), R(0));
    const size_t part_stride = static_cast<size_t>(nvec) * NC * norb * nk;
    const cx_t<R>* tn = T + static_cast<size_t>(n) * NC * norb * nk + k;
    for (int be = share; ok && be < norb; be += S) {
        cx_t<R> vb[NV], t[NC];
#pragma unroll
        for (int v = 0; v < NV; ++v) vb[v] = Vt[(static_cast<size_t>(v) * norb + be) * nk + k];
#pragma unroll
        for (int c = 0; c < NC; ++c) t[c] = tn[(static_cast<size_t>(c) * norb + be) * nk];
#pragma unroll 4
        for (int q = 1; q < parts; ++q)
#pragma unroll
            for (int c = 0; c < NC; ++c) t[c] = cadd(t[c], tn[q * part_stride + (static_cast<size_t>(c) * norb + be) * nk]);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < NV; ++v) cfma(acc[c][v], vb[v], t[c]);
    }
    auto store = [&](int c, int v, cx_t<R> sum) {
        const int64_t row = static_cast<int64_t>(k) * ncv + c * NV + v;
        const double e = (scissor + eval_kq[static_cast<size_t>(k) * nb + NV + c]) - eval_k[static_cast<size_t>(k) * nb + v];
        const double2 x = X[row + n * N];
        Y[row + n * N] = mk(e * x.x - static_cast<double>(sum.x), e * x.y - static_cast<double>(sum.y));
    };
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (S == 1) {
#pragma unroll
            for (int v = 0; v < NV; ++v) store(c, v, acc[c][v]);
        } else {
            if (c > 0) __syncthreads();
#pragma unroll
            for (int v = 0; v < NV; ++v) sums[share][v][threadIdx.x % KB] = acc[c][v];
            __syncthreads();
            if (ok && share < NV) {
                cx_t<R> sum = sums[0][share][threadIdx.x % KB];
#pragma unroll
                for (int q = 1; q < S; ++q) sum = cadd(sum, sums[q][share][threadIdx.x % KB]);
                store(c, share, sum);
            }
        }
    }
}

// Launch the contraction kernels for the context's band counts (nc, nv in 1..4).
template <typename R, typename Fn>
void with_bands(const Context& c, Fn&& fn) {
#define XATU_CONV_BANDS(NC, NV)                          \
    if (c.nc == NC && c.nv == NV) {                       \
        fn(std::integral_constant<int, NC>{}, std::integral_constant<int, NV>{}); \
        return;                                          \
    }
    XATU_CONV_BANDS(1, 1) XATU_CONV_BANDS(1, 2) XATU_CONV_BANDS(1, 3) XATU_CONV_BANDS(1, 4)
    XATU_CONV_BANDS(2, 1) XATU_CONV_BANDS(2, 2) XATU_CONV_BANDS(2, 3) XATU_CONV_BANDS(2, 4)
    XATU_CONV_BANDS(3, 1) XATU_CONV_BANDS(3, 2) XATU_CONV_BANDS(3, 3) XATU_CONV_BANDS(3, 4)
    XATU_CONV_BANDS(4, 1) XATU_CONV_BANDS(4, 2) XATU_CONV_BANDS(4, 3) XATU_CONV_BANDS(4, 4)
#undef XATU_CONV_BANDS
    throw Error(XATU_ERR_INVALID_ARGUMENT, "convolution products support 1 <= nc, nv <= 4");
}

// ---- exchange term along the upper triangle (FP64) ----
// A block is the 64 rows of one wave, so that its sums and scans stay in registers (DPP) and need no
// barrier; the price, four times as many blocks as with 256 rows, falls on the scan over the
// blocks, which 64 threads share per series. N = 129600, 32 vectors, 4 atoms: sums, offsets and application
// 109 + 127 + 169 -> 86 + 17 + 107 us (the vector units busy with the sums); N = 1875, 8 vectors: 7.5 + 5 + 10.6
// -> 4.3 + 4.2 + 4.4 us.
// Block sums of A_a(i) = E2_a(i) x_i and B_a(i) = conj(E1_a(i)) x_i:
// part[((n nblk + blk) NA + a) 2 + s], a wave's values in one store; grid (workgroups, vectors)
__global__ __launch_bounds__(64 * kScanWaves) void xscan_partial_kernel(int na, int ncv, const double2* __restrict__ e1,
                                                                        const double2* __restrict__ e2,
                                                                        const double2* __restrict__ X, int64_t N,
                                                                        int nblk, double2* __restrict__ part) {
    const int n = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t blk = static_cast<int64_t>(blockIdx.x) * kScanWaves + (threadIdx.x >> 6);
    const int64_t i = blk * kScanRows + lane;
    if (blk * kScanRows >= N) return;
    const bool ok = i < N;
    const double2 x = ok ? X[i + n * N] : mk(0.0, 0.0);
    const int64_t k = ok ? i / ncv : 0;
    const int cv = ok ? static_cast<int>(i % ncv) : 0;
    double mr = 0.0, mi = 0.0;  // of the series that this lane stores
    for (int a = 0; a < na; ++a) {
        const size_t off = (static_cast<size_t>(k) * na + a) * ncv + cv;
        const double2 va = cmul(e2[off], x), vb = cmul(cconj(e1[off]), x);
        const double ar = wave_sum(va.x), ai = wave_sum(va.y), br = wave_sum(vb.x), bi = wave_sum(vb.y);
        mr = lane == 2 * a ? ar : lane == 2 * a + 1 ? br : mr;
        mi = lane == 2 * a ? ai : lane == 2 * a + 1 ? bi : mi;
    }
    if (lane < 2 * na) part[(static_cast<size_t>(n) * nblk + blk) * 2 * na + lane] = mk(mr, mi);
}

// Exclusive prefix over the blocks, in place, and the totals. Series t = (n, a, s), ns of them per vector: a workgroup has 16 of them,
// each shared by 64 threads with a run of blocks, whose sums are scanned in LDS. block 1024
constexpr int kOffSeries = 16, kOffRuns = 64;
__global__ __launch_bounds__(kOffSeries* kOffRuns) void xscan_offsets_kernel(int nblk, int nseries, int ns,
                                                                             double2* __restrict__ part,
                                                                             double2* __restrict__ total) {
    __shared__ double2 s_run[kOffRuns][kOffSeries];
    const int c = threadIdx.x % kOffSeries, q = threadIdx.x / kOffSeries;
    const int t = blockIdx.x * kOffSeries + c;
    const int run = (nblk + kOffRuns - 1) / kOffRuns, b0 = min(nblk, q * run), b1 = t < nseries ? min(nblk, b0 + run) : b0;
    double2* p = part + (static_cast<size_t>(t / ns) * nblk) * ns + t % ns;
    double2 sum = mk(0.0, 0.0);
#pragma unroll 8
    for (int b = b0; b < b1; ++b) sum = cadd(sum, p[static_cast<size_t>(b) * ns]);
    s_run[q][c] = sum;
    __syncthreads();
    for (int d = 1; d < kOffRuns; d <<= 1) {
        const double2 v = q >= d ? s_run[q - d][c] : mk(0.0, 0.0);
        __syncthreads();
        s_run[q][c] = cadd(s_run[q][c], v);
        __syncthreads();
    }
    double2 at = q > 0 ? s_run[q - 1][c] : mk(0.0, 0.0);
    if (q == kOffRuns - 1 && t < nseries) total[t] = s_run[q][c];
#pragma unroll 8
    for (int b = b0; b < b1; ++b) {
        const size_t i = static_cast<size_t>(b) * ns;
        const double2 v = p[i];
        p[i] = at;
        at = cadd(at, v);
    }
}

// y_i += sum_a [E1_a(i) (A_tot - sum_{j<=i} A_a(j)) + conj(E2_a(i)) sum_{j<i} B_a(j)] + Re(sum_a E1_a E2_a) x_i
__global__ __launch_bounds__(64 * kScanWaves) void xscan_apply_kernel(int na, int ncv, const double2* __restrict__ e1,
                                                                      const double2* __restrict__ e2,
                                                                      const double2* __restrict__ X, int64_t N, int nblk,
                                                                      const double2* __restrict__ part,
                                                                      const double2* __restrict__ total,
                                                                      double2* __restrict__ Y) {
    const int n = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t blk = static_cast<int64_t>(blockIdx.x) * kScanWaves + (threadIdx.x >> 6);
    const int64_t i = blk * kScanRows + lane;
    if (blk * kScanRows >= N) return;
    const bool ok = i < N;
    const double2 x = ok ? X[i + n * N] : mk(0.0, 0.0);
    const int64_t k = ok ? i / ncv : 0;
    const int cv = ok ? static_cast<int>(i % ncv) : 0;
    const double2* before = part + (static_cast<size_t>(n) * nblk + blk) * 2 * na;  // sums over earlier blocks
    const double2* tot = total + static_cast<size_t>(n) * 2 * na;
    double2 y = mk(0.0, 0.0);
    double diag = 0.0;
    for (int a = 0; a < na; ++a) {
        const size_t off = (static_cast<size_t>(k) * na + a) * ncv + cv;
        const double2 E1 = e1[off], E2 = e2[off];
        if (ok) diag += E1.x * E2.x - E1.y * E2.y;
        const double2 va = cmul(E2, x), vb = cmul(cconj(E1), x);
        const double2 A = cadd(before[2 * a], mk(wave_scan(va.x), wave_scan(va.y)));
        const double2 B = cadd(before[2 * a + 1], mk(wave_scan(vb.x), wave_scan(vb.y)));
        cfma(y, E1, csub(tot[2 * a], A));        // sum_{j>i} A_a(j)
        cfma(y, cconj(E2), csub(B, vb));             // sum_{j<i} B_a(j)
    }
    if (ok) {
        double2 o = Y[i + n * N];
        o.x += y.x + diag * x.x;
        o.y += y.y + diag * x.y;
        Y[i + n * N] = o;
    }
}

// Pw[(n NA^2 + a + NA b) M + xi] = sum_{al in a, be in b} |G[((al norb + be) ns + n) M + xi]|^2
__global__ void power_sum_kernel(LatticeDesc lat, int ns, int64_t M, const double2* __restrict__ G,
                                 double2* __restrict__ Pw) {
    const int64_t xi = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int ab = blockIdx.y, n = blockIdx.z;
    if (xi >= M) return;
    const int a = ab % lat.natoms, b = ab / lat.natoms;
    double sum = 0.0;
    for (int al = lat.orb_begin[a]; al < lat.orb_begin[a + 1]; ++al)
        for (int be = lat.orb_begin[b]; be < lat.orb_begin[b + 1]; ++be) {
            const double2 z = G[((static_cast<int64_t>(al) * lat.norb + be) * ns + n) * M + xi];
            sum += z.x * z.x + z.y * z.y;
        }
    Pw[(static_cast<int64_t>(n) * lat.natoms * lat.natoms + ab) * M + xi] = mk(sum, 0.0);
}

// Scans of the exchange adjoint, from the block sums of xscan_partial_kernel with x = psi:
//   S_a(i) = 2 sum_{j>i} A_a(j) + A_a(i),  F_a(i) = conj(2 sum_{j<i} B_a(j) + B_a(i)),
// A_a = E2_a psi, B_a = conj(E1_a) psi; S[(n NA + a) N + i] and F likewise. grid (blocks, nvec).
__global__ __launch_bounds__(64 * kScanWaves) void xscan_adjoint_kernel(int na, int ncv, const double2* __restrict__ e1,
                                                                        const double2* __restrict__ e2,
                                                                        const double2* __restrict__ X, int64_t N,
                                                                        int nblk, const double2* __restrict__ part,
                                                                        const double2* __restrict__ total,
                                                                        double2* __restrict__ S, double2* __restrict__ F) {
    const int n = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t blk = static_cast<int64_t>(blockIdx.x) * kScanWaves + (threadIdx.x >> 6);
    const int64_t i = blk * kScanRows + lane;
    if (blk * kScanRows >= N) return;
    const bool ok = i < N;
    const double2 x = ok ? X[i + n * N] : mk(0.0, 0.0);
    const int64_t k = ok ? i / ncv : 0;
    const int cv = ok ? static_cast<int>(i % ncv) : 0;
    const double2* before = part + (static_cast<size_t>(n) * nblk + blk) * 2 * na;
    const double2* tot = total + static_cast<size_t>(n) * 2 * na;
    for (int a = 0; a < na; ++a) {
        const size_t off = (static_cast<size_t>(k) * na + a) * ncv + cv;
        const double2 va = cmul(e2[off], x), vb = cmul(cconj(e1[off]), x);
        const double2 A = cadd(before[2 * a], mk(wave_scan(va.x), wave_scan(va.y)));
        const double2 B = cadd(before[2 * a + 1], mk(wave_scan(vb.x), wave_scan(vb.y)));
        if (ok) {
            const size_t out = (static_cast<size_t>(n) * na + a) * N + i;
            const double2 after = csub(tot[2 * a], A), prior = csub(B, vb);
            S[out] = mk(2.0 * after.x + va.x, 2.0 * after.y + va.y);
            F[out] = mk(2.0 * prior.x + vb.x, -(2.0 * prior.y + vb.y));
        }
    }
}

// Band-vector derivatives of one state per blockIdx.y (see conv_band_adjoint): thread per
// (k, orbital), the orbital fastest. g[((n 2 + stack) nk + k) nb + b) norb + orbital].
__global__ __launch_bounds__(256) void band_adjoint_kernel(LatticeDesc lat, int nk, int nv, int nc, int nvec, int parts1,
                                                           int parts2, const double2* __restrict__ Ct,
                                                           const double2* __restrict__ Vt,
                                                           const double2* __restrict__ psi, int64_t N,
                                                           const double2* __restrict__ T1,
                                                           const double2* __restrict__ T2, int exchange,
                                                           const double2* __restrict__ ftq,
                                                           const double2* __restrict__ S,
                                                           const double2* __restrict__ F, double2* __restrict__ g) {
    const int norb = lat.norb, na = lat.natoms, nb = nv + nc, ncv = nc * nv;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<int64_t>(nk) * norb) return;
    const int al = static_cast<int>(idx % norb), k = static_cast<int>(idx / norb);
    const int n = blockIdx.y;
    const int a = atom_of(lat, al);
    const double2* p = psi + static_cast<int64_t>(n) * N + static_cast<int64_t>(k) * ncv;
    const size_t stack = static_cast<size_t>(nk) * nb * norb;
    double2* gk = g + static_cast<size_t>(n) * 2 * stack + static_cast<size_t>(k) * nb * norb + al;
    double2* gq = gk + stack;
    auto term = [&](const double2* T, int parts, int nch, int ch) {
        double2 t = mk(0.0, 0.0);
        for (int q = 0; q < parts; ++q)
            t = cadd(t, T[(((static_cast<size_t>(q) * nvec + n) * nch + ch) * norb + al) * nk + k]);
        return t;
    };
    // H_a = S_a + conj(sum_b F_b MQ_ba) of a row
    auto row_h = [&](int cv) {
        const size_t i = static_cast<size_t>(k) * ncv + cv;
        double2 f = mk(0.0, 0.0);
        for (int b = 0; b < na; ++b) cfma(f, F[(static_cast<size_t>(n) * na + b) * N + i], ftq[b + na * a]);
        return cadd(S[(static_cast<size_t>(n) * na + a) * N + i], cconj(f));
    };
    for (int c = 0; c < nc; ++c) {
        double2 s = mk(0.0, 0.0);
        for (int v = 0; v < nv; ++v) {
            const double2 q = cconj(p[c * nv + v]);
            double2 t = term(T2, parts2, nv, v);
            t = mk(-t.x, -t.y);
            if (exchange) {
                const double2 h = cmul(row_h(c * nv + v), Vt[(static_cast<size_t>(v) * norb + al) * nk + k]);
                t = mk(t.x + 0.5 * h.x, t.y + 0.5 * h.y);
            }
            cfma(s, q, t);
        }
        gq[(nv + c) * norb] = s;
        gk[(nv + c) * norb] = mk(0.0, 0.0);
    }
    for (int v = 0; v < nv; ++v) {
        double2 s = mk(0.0, 0.0);
        for (int c = 0; c < nc; ++c) {
            double2 t = cconj(term(T1, parts1, nc, c));
            t = mk(-t.x, -t.y);
            if (exchange) {
                const double2 h = cmul(cconj(row_h(c * nv + v)), Ct[(static_cast<size_t>(c) * norb + al) * nk + k]);
                t = mk(t.x + 0.5 * h.x, t.y + 0.5 * h.y);
            }
            cfma(s, p[c * nv + v], t);
        }
        gk[v * norb] = s;
        gq[v * norb] = mk(0.0, 0.0);
    }
}

// shat[(s npairs + p) nR + R] from the forward transforms G[(xi_1 batch + (al norb + be) ns + s) W + j]
// (see conv_cell_density); grid (ceil(nR / 256), npairs, ns)
__global__ void cell_power_kernel(LatticeDesc lat, int W, int w0, const int* __restrict__ cells, int nR, int npairs,
                                  int ns, const double2* __restrict__ G, double* __restrict__ shat) {
    const int R = blockIdx.x * blockDim.x + threadIdx.x;
    const int p = blockIdx.y, st = blockIdx.z;
    if (R >= nR) return;
    int a = 0, rem = p;
    while (rem >= lat.natoms - a) {
        rem -= lat.natoms - a;
        ++a;
    }
    const int b = a + rem;
    const int n = lat.mesh_n, norb = lat.norb;
    const int64_t batch = static_cast<int64_t>(norb) * norb * ns;
    auto power = [&](int ra, int rb, int sign) {  // sum over al in ra, be in rb at xi = sign R
        int x[2];
        for (int j = 0; j < 2; ++j) x[j] = (((sign * cells[3 * R + j]) % n) + n) % n;
        int j = x[0] - w0;
        if (j < 0) j += n;
        const double2* g = G + (x[1] * batch + st) * W + j;
        double sum = 0.0;
        for (int al = lat.orb_begin[ra]; al < lat.orb_begin[ra + 1]; ++al)
            for (int be = lat.orb_begin[rb]; be < lat.orb_begin[rb + 1]; ++be) {
                const double2 z = g[static_cast<int64_t>(al * norb + be) * ns * W];
                sum += z.x * z.x + z.y * z.y;
            }
        return sum;
    };
    shat[(static_cast<size_t>(st) * npairs + p) * nR + R] = a < b ? power(a, b, -1) + power(b, a, 1) : power(a, a, 1);
}

// S[(n nmesh + q) NA^2 + ab] = W[(n NA^2 + ab) M + g(Delta(q))] / M with Delta_j = (q_j - m/2) mod m
__global__ void scatter_pair_density_kernel(LatticeDesc lat, int ns, const double2* __restrict__ W,
                                            double2* __restrict__ S) {
    const int64_t M = lat.nmesh;
    const int na2 = lat.natoms * lat.natoms;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= M * na2 * ns) return;
    const int ab = static_cast<int>(idx % na2);
    const int64_t q = (idx / na2) % M;
    const int n = static_cast<int>(idx / (na2 * M));
    const int m = lat.mesh_n;
    int64_t g = 0, mul = 1, rem = q;
    for (int j = 0; j < lat.ndim; ++j) {
        const int d = static_cast<int>(rem % m);
        rem /= m;
        g += static_cast<int64_t>(((d - m / 2) % m + m) % m) * mul;
        mul *= m;
    }
    const double2 w = W[(static_cast<int64_t>(n) * na2 + ab) * M + g];
    const double inv = 1.0 / static_cast<double>(M);
    S[idx] = mk(w.x * inv, w.y * inv);
}

template <typename R>
constexpr rocfft_precision fft_precision() {
    return sizeof(R) == 8 ? rocfft_precision_double : rocfft_precision_single;
}

}  // namespace

struct ConvState {
    int gen = -1;
    int64_t M = 0;
    DevBuf<int> d_gk;
    DevBuf<double2> P64;
    DevBuf<float2> P32;
    DevBuf<double2> G64, U64, Ct64, Vt64;
    DevBuf<float2> G32, U32, Ct32, Vt32;
    DevBuf<double2> part, total;
    DevBuf<double2> S, F, T64b;  // exchange scans and second contraction of the band adjoint
    DevBuf<double2> Mt;  // interaction table on the mesh (set-up scratch, kept between set-ups)
    // row and column transforms (2-D meshes with a supported side): window of the first axis, real
    // spectra on it, cell lists of the spectrum, k-point of each mesh point (-1: none)
    bool rows = false;
    bool full = false;  // every mesh point has a k-point
    int W = 0, w0 = 0;
    DevBuf<double> Pw64;
    DevBuf<float> Pw32;
    DevBuf<int> d_head, d_next, d_kmap;
    DevBuf<double2> T64;
    DevBuf<float2> T32;
    // A transform over the whole mesh: one rocFFT plan per direction (entry-major layout),
    // or for the row-interleaved layout two batched 1-D plans per direction (along o0,
    // then along o1)
    struct Plan {
        rocfft_plan fwd = nullptr, bwd = nullptr, fwd2 = nullptr, bwd2 = nullptr;
        rocfft_execution_info info = nullptr;
        void* work = nullptr;
    };
    std::map<std::tuple<int, int, int>, Plan> plans;  // (bytes per real, batch, row-interleaved)
    int plan_ndim = 0, plan_side = 0;  // the mesh that the plans are for
    void drop_plans() {
        for (auto& kv : plans) {
            for (rocfft_plan q : {kv.second.fwd, kv.second.bwd, kv.second.fwd2, kv.second.bwd2})
                if (q) rocfft_plan_destroy(q);
            if (kv.second.info) rocfft_execution_info_destroy(kv.second.info);
            if (kv.second.work) (void)hipFree(kv.second.work);
        }
        plans.clear();
    }
    ~ConvState() { drop_plans(); }
};

void destroy_conv_state(ConvState* s) { delete s; }

namespace {

void fft_setup_once() {
    static std::once_flag flag;
    static rocfft_status st = rocfft_status_success;
    std::call_once(flag, [] { st = rocfft_setup(); });
    if (st != rocfft_status_success) throw Error(XATU_ERR_DEVICE, "rocfft_setup failed");
}

// Batched 1-D plan of length n with the given stride and distance.
template <typename R>
rocfft_plan strided_plan(rocfft_transform_type dir, size_t n, size_t count, size_t stride, size_t dist) {
    rocfft_plan_description d = nullptr;
    XATU_FFT(rocfft_plan_description_create(&d));
    size_t st[1] = {stride};
    rocfft_status r = rocfft_plan_description_set_data_layout(d, rocfft_array_type_complex_interleaved,
                                                             rocfft_array_type_complex_interleaved, nullptr, nullptr,
                                                             1, st, dist, 1, st, dist);
    rocfft_plan q = nullptr;
    if (r == rocfft_status_success) r = rocfft_plan_create(&q, rocfft_placement_inplace, dir, fft_precision<R>(), 1, &n, count, d);
    rocfft_plan_description_destroy(d);
    XATU_FFT(r);
    return q;
}

// Plans over `batch` mesh transforms; interleaved (2-D meshes only): the row-interleaved
// layout of GLayout.
template <typename R>
ConvState::Plan& get_plan(Context& c, ConvState& cs, int batch, bool interleaved = false) {
    const auto key = std::make_tuple(static_cast<int>(sizeof(R)), batch, interleaved ? 1 : 0);
    auto it = cs.plans.find(key);
    if (it != cs.plans.end()) return it->second;
    fft_setup_once();
    ConvState::Plan p;
    const size_t m = static_cast<size_t>(c.lat.mesh_n);
    size_t lengths[3] = {m, m, m};
    if (interleaved) {
        const size_t count = static_cast<size_t>(batch) * m;
        p.fwd = strided_plan<R>(rocfft_transform_type_complex_forward, m, count, 1, m);
        p.fwd2 = strided_plan<R>(rocfft_transform_type_complex_forward, m, count, count, 1);
        p.bwd = strided_plan<R>(rocfft_transform_type_complex_inverse, m, count, 1, m);
        p.bwd2 = strided_plan<R>(rocfft_transform_type_complex_inverse, m, count, count, 1);
    } else {
        XATU_FFT(rocfft_plan_create(&p.fwd, rocfft_placement_inplace, rocfft_transform_type_complex_forward,
                                    fft_precision<R>(), c.lat.ndim, lengths, batch, nullptr));
        XATU_FFT(rocfft_plan_create(&p.bwd, rocfft_placement_inplace, rocfft_transform_type_complex_inverse,
                                    fft_precision<R>(), c.lat.ndim, lengths, batch, nullptr));
    }
    size_t w = 0;
    for (rocfft_plan q : {p.fwd, p.bwd, p.fwd2, p.bwd2}) {
        size_t wq = 0;
        if (q) XATU_FFT(rocfft_plan_get_work_buffer_size(q, &wq));
        w = std::max(w, wq);
    }
    XATU_FFT(rocfft_execution_info_create(&p.info));
    XATU_FFT(rocfft_execution_info_set_stream(p.info, c.stream));
    if (w > 0) {
        XATU_HIP(hipMalloc(&p.work, w));
        XATU_FFT(rocfft_execution_info_set_work_buffer(p.info, p.work, w));
    }
    return cs.plans.emplace(key, p).first->second;
}

// Largest correlation buffer of one pass of the row and column transforms: a product takes its
// vectors in chunks that keep the buffer within it (N = 129600, 32 FP32 vectors, 2.3 GB in one
// pass: 16.0 ms a call; passes of 512 MB 16.6 ms, of 128 MB, which the last-level cache
// holds, 19.7 ms: the kernels are not bound by that traffic).
constexpr size_t kRowsBufferBytes = size_t(4) << 30;

// Band stacks transposed, the mesh point of every k-point, and the kernel spectra: on 2-D
// meshes with a supported side directly from the potential on the window of the transforms,
// otherwise P_ab = (1/M) backward FFT of the table on the mesh; rebuilt after each preparation
// of the operator.
void ensure_conv(Context& c) {
    if (!c.conv) c.conv = std::unique_ptr<ConvState, void (*)(ConvState*)>(new ConvState, destroy_conv_state);
    ConvState& cs = *c.conv;
    if (cs.gen == c.prep_gen) return;
    if (c.lat.ndim < 1 || c.lat.ndim > 2) throw Error(XATU_ERR_INVALID_ARGUMENT, "convolution products need ndim 1 or 2");
    const int64_t M = c.lat.nmesh;
    cs.M = M;
    const int m = c.lat.mesh_n;
    if (cs.plan_ndim != c.lat.ndim || cs.plan_side != m) {
        // the lattice was set again: plans of another mesh have other lengths
        if (!cs.plans.empty()) XATU_HIP(hipStreamSynchronize(c.stream));
        cs.drop_plans();
        cs.plan_ndim = c.lat.ndim;
        cs.plan_side = m;
    }
    const int norb = c.lat.norb;
    const int na2 = c.lat.natoms * c.lat.natoms;
    std::vector<int> gk(c.nk), kmap(M, -1);
    bool distinct = true;
    for (int k = 0; k < c.nk; ++k) {
        int64_t g = 0, mul = 1;
        for (int j = 0; j < c.lat.ndim; ++j) {
            int o = c.h_koff[static_cast<size_t>(k) * c.lat.ndim + j] % m;
            if (o < 0) o += m;
            g += o * mul;
            mul *= m;
        }
        gk[k] = static_cast<int>(g);
        distinct = distinct && kmap[g] < 0;
        kmap[g] = k;
    }
    cs.Ct64.alloc(static_cast<size_t>(c.nc) * norb * c.nk);
    cs.Vt64.alloc(static_cast<size_t>(c.nv) * norb * c.nk);
    cs.Ct32.alloc(cs.Ct64.n);
    cs.Vt32.alloc(cs.Vt64.n);
    const dim3 tg((c.nk + 255) / 256, (c.nc + c.nv) * norb);
    hipLaunchKernelGGL((transpose_stacks_kernel<double>), tg, dim3(256), 0, c.stream, c.nk, c.nv, c.nc, norb,
                       c.d_evec_k.p, c.d_evec_kq.p, cs.Ct64.p, cs.Vt64.p);
    hipLaunchKernelGGL((transpose_stacks_kernel<float>), tg, dim3(256), 0, c.stream, c.nk, c.nv, c.nc, norb,
                       c.d_evec_k.p, c.d_evec_kq.p, cs.Ct32.p, cs.Vt32.p);
    XATU_HIP(hipGetLastError());
    int fa = 0, fb = 0;
    fft_factors(m, fa, fb);
    cs.full = distinct && static_cast<int64_t>(c.nk) == M;
    // k-points that share a mesh point (offsets that differ by whole periods) stay on the general path
    cs.rows = c.lat.ndim == 2 && fa > 0 && distinct;
    if (cs.rows) {
        int w = 0;
        std::vector<int> head(M, -1), next(c.nR, -1);
        for (int r = c.nR - 1; r >= 0; --r) {
            int o[2];
            for (int j = 0; j < 2; ++j) {
                const int mj = c.h_cells[2 * static_cast<size_t>(r) + j];
                w = std::max(w, j == 0 ? std::abs(mj) : 0);
                o[j] = ((mj % m) + m) % m;
            }
            const int g = o[0] + m * o[1];
            next[r] = head[g];
            head[g] = r;
        }
        cs.W = std::min(m, 2 * w + 1);
        cs.w0 = cs.W == m ? 0 : m - w;
        cs.d_head.alloc(head.size());
        cs.d_next.alloc(next.size());
        cs.d_kmap.alloc(kmap.size());
        XATU_HIP(hipMemcpyAsync(cs.d_head.p, head.data(), head.size() * sizeof(int), hipMemcpyHostToDevice, c.stream));
        XATU_HIP(hipMemcpyAsync(cs.d_next.p, next.data(), next.size() * sizeof(int), hipMemcpyHostToDevice, c.stream));
        XATU_HIP(hipMemcpyAsync(cs.d_kmap.p, kmap.data(), kmap.size() * sizeof(int), hipMemcpyHostToDevice, c.stream));
        const size_t np = static_cast<size_t>(na2) * m * cs.W;
        cs.Pw64.alloc(np);
        cs.Pw32.alloc(np);
        const double inv_total = 1.0 / static_cast<double>(c.inter.total_cells);
        hipLaunchKernelGGL((window_spectrum_kernel<double>), dim3((np + 255) / 256), dim3(256), 0, c.stream, c.lat, cs.W,
                           cs.w0, cs.d_head.p, cs.d_next.p, c.nR, c.d_vtab.p, inv_total, cs.Pw64.p);
        hipLaunchKernelGGL((window_spectrum_kernel<float>), dim3((np + 255) / 256), dim3(256), 0, c.stream, c.lat, cs.W,
                           cs.w0, cs.d_head.p, cs.d_next.p, c.nR, c.d_vtab.p, inv_total, cs.Pw32.p);
        XATU_HIP(hipGetLastError());
        cs.gen = c.prep_gen;
        return;
    }
    cs.d_gk.alloc(c.nk);
    XATU_HIP(hipMemcpyAsync(cs.d_gk.p, gk.data(), gk.size() * sizeof(int), hipMemcpyHostToDevice, c.stream));
    DevBuf<double2>& Mt = cs.Mt;
    Mt.alloc(static_cast<size_t>(na2) * M);
    hipLaunchKernelGGL(table_grid_kernel, dim3((Mt.n + 255) / 256), dim3(256), 0, c.stream, c.lat, c.d_ft.p, Mt.p);
    XATU_HIP(hipGetLastError());
    ConvState::Plan& p = get_plan<double>(c, cs, na2);
    void* buf[1] = {Mt.p};
    XATU_FFT(rocfft_execute(p.bwd, buf, nullptr, p.info));
    cs.P64.alloc(Mt.n);
    cs.P32.alloc(Mt.n);
    const double scale = 1.0 / static_cast<double>(M);
    hipLaunchKernelGGL((scale_spectrum_kernel<double>), dim3((Mt.n + 255) / 256), dim3(256), 0, c.stream, Mt.p,
                       static_cast<int64_t>(Mt.n), scale, cs.P64.p);
    hipLaunchKernelGGL((scale_spectrum_kernel<float>), dim3((Mt.n + 255) / 256), dim3(256), 0, c.stream, Mt.p,
                       static_cast<int64_t>(Mt.n), scale, cs.P32.p);
    XATU_HIP(hipGetLastError());
    cs.gen = c.prep_gen;
}

// The precision's buffers of a ConvState.
template <typename R>
struct ConvBuffers;
template <>
struct ConvBuffers<double> {
    DevBuf<double2>&G, &U, &T;
    const double2 *P, *Ct, *Vt;
    const double* Pw;
    explicit ConvBuffers(ConvState& s) : G(s.G64), U(s.U64), T(s.T64), P(s.P64.p), Ct(s.Ct64.p), Vt(s.Vt64.p), Pw(s.Pw64.p) {}
};
template <>
struct ConvBuffers<float> {
    DevBuf<float2>&G, &U, &T;
    const float2 *P, *Ct, *Vt;
    const float* Pw;
    explicit ConvBuffers(ConvState& s) : G(s.G32), U(s.U32), T(s.T32), P(s.P32.p), Ct(s.Ct32.p), Vt(s.Vt32.p), Pw(s.Pw32.p) {}
};

// u of nv vectors (band contraction with the valence vectors) to b.U.
template <typename R>
void conv_bands_in(Context& c, ConvBuffers<R>& b, const double2* X, int nv, hipStream_t s) {
    const int norb = c.lat.norb;
    b.U.reserve(static_cast<size_t>(nv) * c.nc * norb * c.nk);
    const unsigned kb = (c.nk + 255) / 256;
    const int vg = (nv + conv_vec_group<R>() - 1) / conv_vec_group<R>();
    unsigned long long* stamp = c.take_product_stamp();
    with_bands<R>(c, [&](auto ncc, auto nvc) {
        constexpr int NC = decltype(ncc)::value, NV = decltype(nvc)::value;
        hipLaunchKernelGGL((conv_u_kernel<R, NC, NV>), dim3(kb, vg), dim3(256), 0, s, c.nk, norb, nv, b.Vt, X, c.N, b.U.p,
                           stamp);
    });
    XATU_HIP(hipGetLastError());
}

// Arguments of the row kernels for nv vectors: fixed orbital be, looped orbital al.
RowsArgs rows_args(const Context& c, const ConvState& cs, int nv) {
    const int norb = c.lat.norb;
    RowsArgs a{};
    a.n = c.lat.mesh_n;
    a.W = cs.W;
    a.w0 = cs.w0;
    a.nk = c.nk;
    a.nvec = nv;
    a.nfix = a.nloop = norb;
    a.conj = 1;
    a.batch = static_cast<int64_t>(norb) * norb * nv;
    a.sl = static_cast<int64_t>(norb) * nv;
    a.sf = nv;
    return a;
}

// The transformed z of nv vectors (b.U) on the window: rows, then columns (with the spectrum and
// back, or forward only) in b.G.
template <typename R>
void conv_rows_forward(Context& c, ConvState& cs, ConvBuffers<R>& b, int nv, bool spectrum, hipStream_t s) {
    const RowsArgs a = rows_args(c, cs, nv);
    const int64_t count = a.batch * cs.W;
    b.G.reserve(static_cast<size_t>(count) * a.n);
    launch_rows_in<R>(a, c.nc, cs.d_kmap.p, c.d_twiddle.p, b.Ct, b.U.p, b.G.p, s);
    launch_columns<R>(c.lat, cs.W, count, nv, c.d_twiddle.p, b.Pw, b.G.p, spectrum, s);
}

// Direct term and energies of nv vectors by row and column transforms.
template <typename R>
void conv_rows_product(Context& c, ConvState& cs, ConvBuffers<R>& b, const double2* X, double2* Y, int nv, hipStream_t s) {
    conv_bands_in<R>(c, b, X, nv, s);
    conv_rows_forward<R>(c, cs, b, nv, true, s);
    const RowsArgs a = rows_args(c, cs, nv);
    const int parts = rows_out_chunks(a);
    b.T.reserve(static_cast<size_t>(parts) * nv * c.nc * c.lat.norb * c.nk);
    launch_rows_out<R>(a, c.nc, parts, cs.d_kmap.p, c.d_twiddle.p, b.Ct, b.G.p, b.T.p, s);
    with_bands<R>(c, [&](auto ncc, auto nvc) {
        constexpr int NC = decltype(ncc)::value, NV = decltype(nvc)::value;
        // shared k-points while they leave CUs without a workgroup otherwise
        if (static_cast<int64_t>(c.nk) * nv <= 65536)
            hipLaunchKernelGGL((conv_bands_y_kernel<R, NC, NV, kBandsShare>), dim3((c.nk * kBandsShare + 255) / 256, nv),
                               dim3(256), 0, s, c.nk, c.lat.norb, nv, parts, b.Vt, c.d_eval_k.p, c.d_eval_kq.p,
                               c.scissor, b.T.p, X, c.N, Y);
        else
            hipLaunchKernelGGL((conv_bands_y_kernel<R, NC, NV, 1>), dim3((c.nk + 255) / 256, nv), dim3(256), 0, s, c.nk,
                               c.lat.norb, nv, parts, b.Vt, c.d_eval_k.p, c.d_eval_kq.p, c.scissor, b.T.p, X, c.N, Y);
    });
    XATU_HIP(hipGetLastError());
}

// The same with whole meshes in the buffer and rocFFT: 1-D meshes, sides without a factor pair,
// k-points that share a mesh point.
template <typename R>
void conv_mesh_product(Context& c, ConvState& cs, ConvBuffers<R>& b, const double2* X, double2* Y, int nv, hipStream_t s) {
    const int norb = c.lat.norb;
    const int64_t M = cs.M;
    const int batch = norb * norb * nv;
    // 2-D meshes: row-interleaved layout, two 1-D passes without transpositions
    const bool inter = c.lat.ndim == 2;
    const GLayout lay = inter ? GLayout{c.lat.mesh_n, c.lat.mesh_n, static_cast<int64_t>(batch) * c.lat.mesh_n}
                              : GLayout{M, 0, 0};
    b.G.reserve(static_cast<size_t>(batch) * M);
    conv_bands_in<R>(c, b, X, nv, s);
    if (!cs.full) XATU_HIP(hipMemsetAsync(b.G.p, 0, static_cast<size_t>(batch) * M * sizeof(cx_t<R>), s));
    const dim3 kb((c.nk + 255) / 256);
    with_bands<R>(c, [&](auto ncc, auto nvc) {
        constexpr int NC = decltype(ncc)::value, NV = decltype(nvc)::value;
        (void)NV;
        hipLaunchKernelGGL((conv_z_kernel<R, NC>), dim3(kb.x, (norb + conv_orb_group<R>() - 1) / conv_orb_group<R>(), nv),
                           dim3(256), 0, s, c.nk, norb, nv, lay, cs.d_gk.p, b.Ct, b.U.p, b.G.p);
    });
    XATU_HIP(hipGetLastError());
    ConvState::Plan& p = get_plan<R>(c, cs, batch, inter);
    void* buf[1] = {b.G.p};
    XATU_FFT(rocfft_execute(p.fwd, buf, nullptr, p.info));
    if (p.fwd2) XATU_FFT(rocfft_execute(p.fwd2, buf, nullptr, p.info));
    hipLaunchKernelGGL((conv_multiply_kernel<R>), dim3((M + 255) / 256, batch), dim3(256), 0, s, c.lat, nv, M, lay, b.P,
                       b.G.p);
    XATU_HIP(hipGetLastError());
    if (p.bwd2) XATU_FFT(rocfft_execute(p.bwd2, buf, nullptr, p.info));
    XATU_FFT(rocfft_execute(p.bwd, buf, nullptr, p.info));
    with_bands<R>(c, [&](auto ncc, auto nvc) {
        constexpr int NC = decltype(ncc)::value, NV = decltype(nvc)::value;
        const int yg = (nv + conv_y_group<R>() - 1) / conv_y_group<R>();
        hipLaunchKernelGGL((conv_y_kernel<R, NC, NV>), dim3(kb.x, yg), dim3(256), 0, s, c.nk, norb, nv, lay, cs.d_gk.p,
                           b.Ct, b.Vt, c.d_eval_k.p, c.d_eval_kq.p, c.scissor, b.G.p, X, c.N, Y);
    });
    XATU_HIP(hipGetLastError());
}

// Vectors per pass of the row and column transforms (their buffer within kRowsBufferBytes).
template <typename R>
int rows_vectors(const Context& c, const ConvState& cs, int nvec) {
    const size_t per = sizeof(cx_t<R>) * static_cast<size_t>(c.lat.norb) * c.lat.norb * cs.W * c.lat.mesh_n;
    const int most = static_cast<int>(std::max<size_t>(1, std::min<size_t>(kBlockVectors, kRowsBufferBytes / per)));
    const int passes = (nvec + most - 1) / most;
    return (nvec + passes - 1) / passes;
}

int scan_blocks(int64_t N) { return static_cast<int>((N + kScanRows - 1) / kScanRows); }

// Block sums of the exchange scans of nv vectors, as offsets (cs.part) and totals; returns the
// number of workgroups for the blocks.
int exchange_scans(Context& c, ConvState& cs, const double2* X, int nv, hipStream_t s) {
    const int nblk = scan_blocks(c.N), wgs = (nblk + kScanWaves - 1) / kScanWaves;
    const int nseries = c.lat.natoms * 2 * nv;
    cs.part.reserve(static_cast<size_t>(nblk) * nseries);
    cs.total.reserve(static_cast<size_t>(nseries));
    hipLaunchKernelGGL(xscan_partial_kernel, dim3(wgs, nv), dim3(64 * kScanWaves), 0, s, c.lat.natoms, c.nc * c.nv,
                       c.d_e1.p, c.d_e2.p, X, c.N, nblk, cs.part.p);
    hipLaunchKernelGGL(xscan_offsets_kernel, dim3((nseries + kOffSeries - 1) / kOffSeries), dim3(kOffSeries * kOffRuns), 0,
                       s, nblk, nseries, 2 * c.lat.natoms, cs.part.p, cs.total.p);
    XATU_HIP(hipGetLastError());
    return wgs;
}

template <typename R>
void conv_product(Context& c, const double2* X, double2* Y, int nvec, hipStream_t s) {
    ConvState& cs = *c.conv;
    ConvBuffers<R> b(cs);
    const int64_t N = c.N;
    const int step = cs.rows ? rows_vectors<R>(c, cs, nvec) : kBlockVectors;
    for (int v0 = 0; v0 < nvec; v0 += step) {
        const int nv = std::min(step, nvec - v0);
        const double2* Xb = X + static_cast<int64_t>(v0) * N;
        double2* Yb = Y + static_cast<int64_t>(v0) * N;
        if (cs.rows) conv_rows_product<R>(c, cs, b, Xb, Yb, nv, s);
        else conv_mesh_product<R>(c, cs, b, Xb, Yb, nv, s);
    }
    if (!c.inter.exchange) return;
    for (int v0 = 0; v0 < nvec; v0 += kBlockVectors) {
        const int nv = std::min(kBlockVectors, nvec - v0);
        const double2* Xb = X + static_cast<int64_t>(v0) * N;
        double2* Yb = Y + static_cast<int64_t>(v0) * N;
        const int na = c.lat.natoms;
        const int ncv = c.nc * c.nv;
        const int wgs = exchange_scans(c, cs, Xb, nv, s);
        hipLaunchKernelGGL(xscan_apply_kernel, dim3(wgs, nv), dim3(64 * kScanWaves), 0, s, na, ncv, c.d_e1.p, c.d_e2.p, Xb, N,
                           scan_blocks(N), cs.part.p, cs.total.p, Yb);
        XATU_HIP(hipGetLastError());
    }
}

}  // namespace

// Whether the operator's convolution runs on the row and column transforms.
bool conv_rows_available(Context& c) {
    ensure_conv(c);
    return c.conv->rows;
}

// Adjoint of the lattice sums for the Hellmann-Feynman gradients, on the cells directly:
//   Shat_p(R) = sum_q [S_ab(q) e^{iqR} + S_ba(q) e^{-iqR}] (a < b),  sum_q S_aa(q) e^{-iqR} (a = b)
// with S_ab(q) the pair densities of conv_pair_density. Their transform is the power spectrum of
// z, so Shat_p(R) = sum_{al in a, be in b} |Z_{al be}(-R)|^2 + sum_{al in b, be in a} |Z_{al be}(R)|^2
// (a = b: one sum, at R), Z the forward transform of z on the window that holds every cell.
// shat[(s npairs + p) nR + R] for the ns <= 32 states of psi (N x ns), taken in passes that keep the buffer
// within kRowsBufferBytes.
void conv_cell_density(Context& c, const double2* psi, int ns, double* shat) {
    ensure_conv(c);
    ConvState& cs = *c.conv;
    ConvBuffers<double> b(cs);
    hipStream_t s = c.stream;
    const int npairs = c.lat.natoms * (c.lat.natoms + 1) / 2;
    const int step = rows_vectors<double>(c, cs, ns);
    for (int v0 = 0; v0 < ns; v0 += step) {
        const int nv = std::min(step, ns - v0);
        conv_bands_in<double>(c, b, psi + static_cast<int64_t>(v0) * c.N, nv, s);
        conv_rows_forward<double>(c, cs, b, nv, false, s);
        hipLaunchKernelGGL(cell_power_kernel, dim3((c.nR + 255) / 256, npairs, nv), dim3(256), 0, s, c.lat, cs.W, cs.w0,
                           c.d_cells.p, c.nR, npairs, nv, b.G.p, shat + static_cast<size_t>(v0) * npairs * c.nR);
        XATU_HIP(hipGetLastError());
    }
}

// Adjoint of the assembly with respect to the band vectors by the same transforms: with
// z_{al be} = sum_cv C_al conj(V_be) psi_cv and w = M (*) z the direct term's energy is
// -sum_k conj(z) w, so that (Wirtinger derivatives by the conjugated coefficients, M Hermitian)
//   g_C(c, al) = -sum_v conj(psi_cv) sum_be V_be,v w_{al be},
//   g_V(v, be) = -sum_c psi_cv conj(sum_al conj(C_al,c) w_{al be}):
// the contraction of the product and the same with the orbitals exchanged. The exchange term
// along the upper triangle, Re sum_a [2 sum_{i<j} f_a(i) A_a(j) + sum_i f_a(i) A_a(i)] with
// f_a = conj(psi) E1_a and A_a = E2_a psi, adds with its scans S and F (xscan_adjoint_kernel) and
// H_a = S_a + conj(sum_b F_b MQ_ba)
//   g_C(c, al) += 1/2 sum_v conj(psi_cv) V_al,v H_a,  g_V(v, al) += 1/2 sum_c psi_cv C_al,c conj(H_a).
// Cost per state: the transforms of one product, against nk^2 / 2 pairs of k-points with atomic
// adds (36 x 36, 18 orbitals, 8 states: 0.2 ms for 104 ms). g: ns states of 2 stacks.
void conv_band_adjoint(Context& c, const double2* psi, int ns, double2* g) {
    ensure_conv(c);
    ConvState& cs = *c.conv;
    ConvBuffers<double> b(cs);
    hipStream_t s = c.stream;
    const int norb = c.lat.norb, na = c.lat.natoms;
    const size_t stack = static_cast<size_t>(norb) * c.nb * c.nk;
    const int step = rows_vectors<double>(c, cs, std::min(ns, kBlockVectors));
    for (int v0 = 0; v0 < ns; v0 += step) {
        const int nv = std::min(step, ns - v0);
        const double2* X = psi + static_cast<int64_t>(v0) * c.N;
        conv_bands_in<double>(c, b, X, nv, s);
        conv_rows_forward<double>(c, cs, b, nv, true, s);
        const RowsArgs a1 = rows_args(c, cs, nv);
        RowsArgs a2 = a1;  // fixed al, looped be
        a2.conj = 0;
        a2.sl = nv;
        a2.sf = static_cast<int64_t>(norb) * nv;
        const int parts = rows_out_chunks(a1);
        b.T.reserve(static_cast<size_t>(parts) * nv * c.nc * norb * c.nk);
        cs.T64b.reserve(static_cast<size_t>(parts) * nv * c.nv * norb * c.nk);
        launch_rows_out<double>(a1, c.nc, parts, cs.d_kmap.p, c.d_twiddle.p, b.Ct, b.G.p, b.T.p, s);
        launch_rows_out<double>(a2, c.nv, parts, cs.d_kmap.p, c.d_twiddle.p, b.Vt, b.G.p, cs.T64b.p, s);
        if (c.inter.exchange) {
            const int wgs = exchange_scans(c, cs, X, nv, s);
            cs.S.reserve(static_cast<size_t>(nv) * na * c.N);
            cs.F.reserve(static_cast<size_t>(nv) * na * c.N);
            hipLaunchKernelGGL(xscan_adjoint_kernel, dim3(wgs, nv), dim3(64 * kScanWaves), 0, s, na, c.nc * c.nv, c.d_e1.p,
                               c.d_e2.p, X, c.N, scan_blocks(c.N), cs.part.p, cs.total.p, cs.S.p, cs.F.p);
        }
        hipLaunchKernelGGL(band_adjoint_kernel, dim3((static_cast<size_t>(c.nk) * norb + 255) / 256, nv), dim3(256), 0, s,
                           c.lat, c.nk, c.nv, c.nc, nv, parts, parts, b.Ct, b.Vt, X, c.N, b.T.p, cs.T64b.p,
                           c.inter.exchange, c.d_ftq.p, cs.S.p, cs.F.p, g + 2 * stack * v0);
        XATU_HIP(hipGetLastError());
    }
}

// Pair-density adjoint of the direct term for the Hellmann-Feynman gradients:
//   S_ab(q) = sum_k G_ab(k, k+q),  G_ab(k,k') = sum_{al in a, be in b} conj(z_ab(k)) z_ab(k'),
// with z_{al be}(k) = sum_{cv} C_kc,al conj(V_kv,be) psi_kcv (the vector the convolution
// product forms from x = psi). The sum over k is an autocorrelation on the mesh:
// S_ab(Delta) = (1/M) backward( sum_{al in a, be in b} |forward(z_{al be})|^2 )(Delta).
// Output layout S[(n nmesh + q) NA^2 + a + NA b] for the ns states of psi (N x ns).
void conv_pair_density(Context& c, const double2* psi, int ns, double2* S) {
    ensure_conv(c);
    ConvState& cs = *c.conv;
    const int norb = c.lat.norb;
    const int na2 = c.lat.natoms * c.lat.natoms;
    const int64_t M = cs.M;
    const int64_t N = c.N;
    hipStream_t s = c.stream;
    if (ns < 1 || ns > kBlockVectors) throw Error(XATU_ERR_INVALID_ARGUMENT, "pair density: 1..32 states per call");
    const int batch = norb * norb * ns;
    cs.G64.alloc(std::max<size_t>(cs.G64.n, static_cast<size_t>(batch) * M));
    cs.U64.alloc(std::max<size_t>(cs.U64.n, static_cast<size_t>(ns) * c.nc * norb * c.nk));
    if (!cs.full) XATU_HIP(hipMemsetAsync(cs.G64.p, 0, static_cast<size_t>(batch) * M * sizeof(double2), s));
    const dim3 kb((c.nk + 255) / 256);
    with_bands<double>(c, [&](auto ncc, auto nvc) {
        constexpr int NC = decltype(ncc)::value, NV = decltype(nvc)::value;
        constexpr int VG = conv_vec_group<double>();
        hipLaunchKernelGGL((conv_u_kernel<double, NC, NV>), dim3(kb.x, (ns + VG - 1) / VG), dim3(256), 0, s, c.nk, norb,
                           ns, cs.Vt64.p, psi, N, cs.U64.p, nullptr);
        hipLaunchKernelGGL((conv_z_kernel<double, NC>), dim3(kb.x, (norb + conv_orb_group<double>() - 1) / conv_orb_group<double>(), ns),
                           dim3(256), 0, s, c.nk, norb, ns, GLayout{M, 0, 0}, cs.d_gk.p, cs.Ct64.p, cs.U64.p,
                           cs.G64.p);
    });
    XATU_HIP(hipGetLastError());
    ConvState::Plan& pf = get_plan<double>(c, cs, batch);
    void* buf[1] = {cs.G64.p};
    XATU_FFT(rocfft_execute(pf.fwd, buf, nullptr, pf.info));
    DevBuf<double2> Pw;
    Pw.alloc(static_cast<size_t>(ns) * na2 * M);
    hipLaunchKernelGGL(power_sum_kernel, dim3((M + 255) / 256, na2, ns), dim3(256), 0, s, c.lat, ns, M, cs.G64.p, Pw.p);
    XATU_HIP(hipGetLastError());
    ConvState::Plan& pb = get_plan<double>(c, cs, na2 * ns);
    void* buf2[1] = {Pw.p};
    XATU_FFT(rocfft_execute(pb.bwd, buf2, nullptr, pb.info));
    hipLaunchKernelGGL(scatter_pair_density_kernel, dim3((Pw.n + 255) / 256), dim3(256), 0, s, c.lat, ns, Pw.p, S);
    XATU_HIP(hipGetLastError());
    XATU_HIP(hipStreamSynchronize(s));  // Pw goes out of scope
}

void launch_conv64(Context& c, const double2* X, double2* Y, int nvec, hipStream_t s) {
    ensure_conv(c);
    conv_product<double>(c, X, Y, nvec, s);
}

void launch_conv32(Context& c, const double2* X, double2* Y, int nvec, hipStream_t s) {
    ensure_conv(c);
    conv_product<float>(c, X, Y, nvec, s);
}

}  // namespace xatu_dev
