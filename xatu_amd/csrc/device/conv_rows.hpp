// Transforms of the convolution product on 2-D meshes with sides n = A B (fft_stages.hpp): three
// kernels between which the correlation buffer holds only the window of first-axis frequencies
// where the kernel spectrum is not zero.
//
// The spectrum of the lattice-sum table on the mesh is the potential itself: the table is
// M_ab(Delta) = (1/T) sum_R V_ab(R) e^{i Delta R}, so its transform at frequency xi is
// V_ab(R)/T for the cells R = -xi (a < b) or R = +xi (a >= b, stored conjugated), real, and
// zero outside the cutoff: |xi_0| <= w of the n frequencies of an axis matter (N = 36864,
// cutoff 25 cells: 57 of 96). The buffer is
//   G[(o1 batch + b) W + j],  o1 the mesh row, b = (al norb + be) nvec + v, xi_0 = (w0 + j) mod n.
//  conv_rows_in_kernel   z_{al be}(k) = sum_c C_k[al, c] u[v][c][be][k] along a mesh row and its
//                        transform, in registers, the window to G
//  conv_columns_kernel   per (b, j): transform along o1, times the spectrum, inverse (in place)
//  conv_rows_out_kernel  inverse transform along a row from the window, contracted at once with
//                        the band coefficients: t[v][c][be][k] = sum_al conj(C_k[al, c]) w(k)
// so that z and w at the mesh points never go to memory: the buffer is written and read twice
// at W / n of its size. Measured against one kernel that held whole planes in LDS between a
// contraction that wrote z and one that read w (32 FP32 vectors, 36 orbitals, 120 x 120; 16 FP64
// vectors, 18 orbitals, 96 x 96): 1.77 + 4.12 + 1.65 -> 1.55 + 1.14 + 1.72 + 0.16 ms and
// 0.17 + 0.56 + 0.25 -> 0.18 + 0.19 + 0.24 + 0.02 ms. The columns run at 4 TB/s; the rows are
// bound by the latency of the loop over l (LDS reads, exchange, two DFTs) at two waves per
// SIMD: their vector instructions alone take about half the time.
#pragma once
#include <cstdint>
#include <type_traits>

#include "context.hpp"
#include "cplx.hpp"
#include "fft_stages.hpp"

namespace xatu_dev {

constexpr int kRowWaves = 4;   // waves per workgroup of the row kernels
// Adjacent columns per workgroup of the column kernel: fewer for the long prime factors, whose
// workgroups would have too many waves for the registers of their DFT (62 x 62, FP64, 16 columns: 1.70 ms
// a product, 8: 1.23; 124 x 124: 4.8 and 5.5).
constexpr int col_group(int A, int B) { return B <= 16 ? 32 : A <= 2 && B > 23 ? 8 : 16; }

// Waves per SIMD of the row kernels (three made the FP32 ones spill: 1.72 -> 1.84 ms).
constexpr int kRowOccupancy = 2;

// Arguments of the row kernels. A group of B lanes owns one (fixed orbital f, vector v) of one
// mesh row and loops over the other orbital l; its row of G starts at
// (o1 batch + f sf + l sl + v) W.
struct RowsArgs {
    int n;
    int W, w0;           // window of the first-axis frequencies
    int nk, nvec;
    int nfix, nloop;     // fixed and looped orbitals
    int lchunk, stage;   // looped orbitals per workgroup (grid z) and per LDS stage
    int conj;            // rows_out: conjugate the coefficients
    int64_t batch, sf, sl;
};

// LDS: twiddles, staged coefficients [l][channel][o0], then a buffer per wave for the exchange
// between the two steps (8-byte words; FP64 exchanges real and imaginary parts in turn).
template <typename R, int A, int B, int NCH>
constexpr size_t rows_lds_bytes(int stage) {
    constexpr int n = A * B;
    return sizeof(cx_t<R>) * (static_cast<size_t>(n) + static_cast<size_t>(stage) * NCH * n) +
           8 * static_cast<size_t>(kRowWaves) * (64 / B) * B * (A | 1);
}

// Orders the LDS accesses of one wave (the groups of a row never cross a wave).
__device__ inline void rows_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Exchange of a group through its LDS buffer: lane `wl` (if wr) writes v[i] to slot(i), lane
// `rl` (if rd) reads x[i] from its slots.
template <typename R, int NW, int NR, typename WS, typename RS>
__device__ inline void rows_exchange(void* buf, bool wr, const cx_t<R> (&v)[NW], WS&& ws, bool rd, cx_t<R> (&x)[NR],
                                     RS&& rs) {
    if constexpr (sizeof(R) == 8) {
        double* e = static_cast<double*>(buf);
        if (wr) {
#pragma unroll
            for (int i = 0; i < NW; ++i) e[ws(i)] = v[i].x;
        }
        rows_wave_sync();
        if (rd) {
#pragma unroll
            for (int i = 0; i < NR; ++i) x[i].x = e[rs(i)];
        }
        rows_wave_sync();
        if (wr) {
#pragma unroll
            for (int i = 0; i < NW; ++i) e[ws(i)] = v[i].y;
        }
        rows_wave_sync();
        if (rd) {
#pragma unroll
            for (int i = 0; i < NR; ++i) x[i].y = e[rs(i)];
        }
        rows_wave_sync();
    } else {
        float2* e = static_cast<float2*>(buf);
        if (wr) {
#pragma unroll
            for (int i = 0; i < NW; ++i) e[ws(i)] = v[i];
        }
        rows_wave_sync();
        if (rd) {
#pragma unroll
            for (int i = 0; i < NR; ++i) x[i] = e[rs(i)];
        }
        rows_wave_sync();
    }
}

// The step of a long prime length B with a short A, spread over the B lanes of a group: each lane
// forms one frequency of every of the A transforms from the entries of all lanes, which it reads from
// LDS (the same address for the whole group), with its own B - 1 cosines and sines in registers. In the
// other form A lanes hold a whole transform each and the others wait: 2 (B - 1)^2 against 4 A (B - 1)
// multiply-adds (62 = 2 x 31: 1800 on two lanes against 240 on all).
template <int A, int B>
constexpr bool rows_spread() {
    return B >= 11 && B != 12 && B != 14 && B != 15 && B != 16 && 4 * A <= B;
}
// Steps of the sum whose LDS reads may be in flight together (more of them spilled: the compiler
// moved all reads to the front).
constexpr int kSpreadLoads = 4;
template <typename R, int B>
struct SpreadRoots {
    static constexpr int H = (B - 1) / 2;
    R c[H], s[H];  // of e^{-2 pi i j k / B}, j = 1 .. H, k the lane's
    __device__ void load(const cx_t<R>* tw, int A, int k) {
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const cx_t<R> t = tw[(j * k % B) * A];
            c[j - 1] = t.x;
            s[j - 1] = t.y;
        }
    }
};
// p + i q (SG -1) or p - i q (SG 1): the sums of the entries with the roots or their conjugates.
template <typename R, int SG>
__device__ inline cx_t<R> spread_value(cx_t<R> p, cx_t<R> q) {
    return SG < 0 ? mk(p.x - q.y, p.y + q.x) : mk(p.x + q.y, p.y - q.x);
}
// z[k1] of the lanes k2 = 0 .. B - 1 of a group -> out[k1] = sum_k2 z_k2[k1] e^{SG 2 pi i k2 s / B}
template <typename R, int A, int B, int SG>
__device__ inline void rows_spread_dft(void* buf, bool on, int s, const cx_t<R> (&z)[A], const SpreadRoots<R, B>& w,
                                       cx_t<R> (&out)[A]) {
    constexpr int H = (B - 1) / 2, AP = A | 1;
    cx_t<R> p[A], q[A];
    if constexpr (sizeof(R) == 8) {
        double* e = static_cast<double*>(buf);
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            if (on) {
#pragma unroll
                for (int k = 0; k < A; ++k) e[s * AP + k] = part ? z[k].y : z[k].x;
            }
            rows_wave_sync();
            if (on) {
                double a[A], d[A];
#pragma unroll
                for (int k = 0; k < A; ++k) {
                    a[k] = e[k];
                    d[k] = 0.0;
                }
#pragma unroll
                for (int j = 1; j <= H; ++j) {
                    if (j % kSpreadLoads == 0) asm volatile("" ::: "memory");
#pragma unroll
                    for (int k = 0; k < A; ++k) {
                        const double x = e[j * AP + k], y = e[(B - j) * AP + k];
                        a[k] += w.c[j - 1] * (x + y);
                        d[k] += w.s[j - 1] * (x - y);
                    }
                }
#pragma unroll
                for (int k = 0; k < A; ++k) {
                    if (part) {
                        p[k].y = a[k];
                        q[k].y = d[k];
                    } else {
                        p[k].x = a[k];
                        q[k].x = d[k];
                    }
                }
            }
            rows_wave_sync();
        }
    } else {
        float2* e = static_cast<float2*>(buf);
        if (on) {
#pragma unroll
            for (int k = 0; k < A; ++k) e[s * AP + k] = z[k];
        }
        rows_wave_sync();
        if (on) {
#pragma unroll
            for (int k = 0; k < A; ++k) {
                p[k] = e[k];
                q[k] = mk(0.0f, 0.0f);
            }
#pragma unroll
            for (int j = 1; j <= H; ++j) {
                if (j % kSpreadLoads == 0) asm volatile("" ::: "memory");
#pragma unroll
                for (int k = 0; k < A; ++k) {
                    const float2 x = e[j * AP + k], y = e[(B - j) * AP + k];
                    p[k] = mk(p[k].x + w.c[j - 1] * (x.x + y.x), p[k].y + w.c[j - 1] * (x.y + y.y));
                    q[k] = mk(q[k].x + w.s[j - 1] * (x.x - y.x), q[k].y + w.s[j - 1] * (x.y - y.y));
                }
            }
        }
        rows_wave_sync();
    }
#pragma unroll
    for (int k = 0; k < A; ++k) out[k] = on ? spread_value<R, SG>(p[k], q[k]) : mk(R(0), R(0));
}
// Offsets of the frequencies k1 + A s of a lane of the spread form.
template <int A, int B>
__device__ inline void spread_offsets(const RowsArgs& a, int s, int at, bool on, int (&off)[A]) {
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        int j = k1 + A * s - a.w0;
        if (j < 0) j += A * B;
        off[k1] = (on && j < a.W) ? at + j : -1;
    }
}

// Coefficients Coef[(c nloop + l) nk + k] of the looped orbitals l0 .. l0 + count - 1 on mesh row
// o1 to sc[(l NCH + c) n + o0] (zero where the mesh point has no k-point).
template <typename R, int NCH>
__device__ inline void stage_row_coefficients(cx_t<R>* sc, const cx_t<R>* __restrict__ Coef, const int* __restrict__ kmap,
                                              const RowsArgs& a, int o1, int l0, int count) {
    const int total = count * NCH * a.n;
    for (int e = threadIdx.x; e < total; e += 64 * kRowWaves) {
        const int o0 = e % a.n, lc = e / a.n;
        const int c = lc % NCH, l = l0 + lc / NCH;
        const int k = kmap[o0 + a.n * o1];
        sc[e] = k >= 0 ? Coef[(static_cast<size_t>(c) * a.nloop + l) * a.nk + k] : mk(R(0), R(0));
    }
}

// Offsets within a mesh row of G of a lane's frequencies s + A k2, from `at` on; -1 outside the
// window or for an idle lane.
template <int A, int B>
__device__ inline void row_offsets(const RowsArgs& a, int s, int at, bool on, int (&off)[B]) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
        int j = s + A * k2 - a.w0;
        if (j < 0) j += A * B;
        off[k2] = (on && j < a.W) ? at + j : -1;
    }
}

// Twiddles e^{-2 pi i k / n} from the lattice sums' table of e^{i pi p / n}.
template <typename R>
__device__ inline void load_twiddles(cx_t<R>* tw, const double2* __restrict__ root, int n, int nthreads) {
    for (int k = threadIdx.x; k < n; k += nthreads) {
        const double2 r = root[2 * k];
        tw[k] = mk(static_cast<R>(r.x), static_cast<R>(-r.y));
    }
}

// Forward rows. U[((v NCH + c) nfix + f) nk + k]. grid (row groups, n, chunks of l), block 256.
template <typename R, int A, int B, int NCH>
__global__ __launch_bounds__(64 * kRowWaves, kRowOccupancy) void conv_rows_in_kernel(RowsArgs a, const int* __restrict__ kmap,
                                                                      const double2* __restrict__ root,
                                                                      const cx_t<R>* __restrict__ Coef,
                                                                      const cx_t<R>* __restrict__ U,
                                                                      cx_t<R>* __restrict__ G) {
    using C = cx_t<R>;
    constexpr int n = A * B, GW = 64 / B, AP = A | 1;
    extern __shared__ unsigned char rows_raw[];
    C* tw = reinterpret_cast<C*>(rows_raw);
    C* sc = tw + n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gi = lane / B, s = lane - gi * B;
    const int o1 = blockIdx.y;
    const int task = (blockIdx.x * kRowWaves + wave) * GW + gi;
    const bool live = gi < GW && task < a.nfix * a.nvec;
    const int f = live ? task / a.nvec : 0, v = live ? task - f * a.nvec : 0;
    unsigned char* xb = rows_raw + sizeof(C) * (n + static_cast<size_t>(a.stage) * NCH * n) +
                        8 * static_cast<size_t>(wave * GW + (gi < GW ? gi : 0)) * B * AP;
    load_twiddles<R>(tw, root, n, 64 * kRowWaves);
    C u[A][NCH];
#pragma unroll
    for (int j = 0; j < A; ++j) {
        const int k = live ? kmap[B * j + s + n * o1] : -1;
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            u[j][c] = k >= 0 ? U[((static_cast<size_t>(v) * NCH + c) * a.nfix + f) * a.nk + k] : mk(R(0), R(0));
    }
    const int l0 = blockIdx.z * a.lchunk, l1 = min(a.nloop, l0 + a.lchunk);
    // uniform base of the mesh row, 32-bit offsets of the lane's window entries (-1: outside)
    C* grow = G + static_cast<int64_t>(o1) * a.batch * a.W;
    constexpr bool kSpread = rows_spread<A, B>();
    int off[kSpread ? A : B];
    SpreadRoots<R, kSpread ? B : 1> roots;
    if constexpr (kSpread) {
        spread_offsets<A, B>(a, s, static_cast<int>(f * a.sf + v) * a.W, live, off);
        __syncthreads();  // the twiddles
        roots.load(tw, A, s);
    } else {
        row_offsets<A, B>(a, s, static_cast<int>(f * a.sf + v) * a.W, live && s < A, off);
    }
    for (int ls = l0; ls < l1; ls += a.stage) {
        const int count = min(a.stage, l1 - ls);
        __syncthreads();
        stage_row_coefficients<R, NCH>(sc, Coef, kmap, a, o1, ls, count);
        __syncthreads();
        for (int l = 0; l < count; ++l) {
            C z[A];
#pragma unroll
            for (int j = 0; j < A; ++j) {
                z[j] = mk(R(0), R(0));
#pragma unroll
                for (int c = 0; c < NCH; ++c) cfma(z[j], sc[(l * NCH + c) * n + B * j + s], u[j][c]);
            }
            dft_len<R, A, -1>(z);
#pragma unroll
            for (int k1 = 1; k1 < A; ++k1) z[k1] = cmul(z[k1], tw[s * k1]);
            if constexpr (kSpread) {
                C x[A];
                rows_spread_dft<R, A, B, -1>(xb, gi < GW, s, z, roots, x);
                C* out = grow + static_cast<int64_t>(ls + l) * a.sl * a.W;
#pragma unroll
                for (int k1 = 0; k1 < A; ++k1)
                    if (off[k1] >= 0) out[static_cast<unsigned>(off[k1])] = x[k1];
            } else {
                C x[B];
                rows_exchange<R, A, B>(
                    xb, gi < GW, z, [&](int i) { return s * AP + i; }, gi < GW && s < A, x,
                    [&](int i) { return i * AP + s; });
                if (live && s < A) {
                    dft_len<R, B, -1>(x);
                    C* out = grow + static_cast<int64_t>(ls + l) * a.sl * a.W;
#pragma unroll
                    for (int k2 = 0; k2 < B; ++k2)
                        if (off[k2] >= 0) out[static_cast<unsigned>(off[k2])] = x[k2];
                }
            }
        }
    }
}

// Inverse rows and contraction: T[(((part nvec + v) NCH + c) nfix + f) nk + k] = sum over the l of
// this chunk (part) of Coef_l (conjugated if a.conj) times the row. grid as above, block 256.
template <typename R, int A, int B, int NCH>
__global__ __launch_bounds__(64 * kRowWaves, kRowOccupancy) void conv_rows_out_kernel(RowsArgs a, const int* __restrict__ kmap,
                                                                       const double2* __restrict__ root,
                                                                       const cx_t<R>* __restrict__ Coef,
                                                                       const cx_t<R>* __restrict__ G,
                                                                       cx_t<R>* __restrict__ T) {
    using C = cx_t<R>;
    constexpr int n = A * B, GW = 64 / B, AP = A | 1;
    extern __shared__ unsigned char rows_raw[];
    C* tw = reinterpret_cast<C*>(rows_raw);
    C* sc = tw + n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gi = lane / B, s = lane - gi * B;
    const int o1 = blockIdx.y;
    const int task = (blockIdx.x * kRowWaves + wave) * GW + gi;
    const bool live = gi < GW && task < a.nfix * a.nvec;
    const int f = live ? task / a.nvec : 0, v = live ? task - f * a.nvec : 0;
    unsigned char* xb = rows_raw + sizeof(C) * (n + static_cast<size_t>(a.stage) * NCH * n) +
                        8 * static_cast<size_t>(wave * GW + (gi < GW ? gi : 0)) * B * AP;
    load_twiddles<R>(tw, root, n, 64 * kRowWaves);
    C t[A][NCH];
#pragma unroll
    for (int j = 0; j < A; ++j)
#pragma unroll
        for (int c = 0; c < NCH; ++c) t[j][c] = mk(R(0), R(0));
    const int l0 = blockIdx.z * a.lchunk, l1 = min(a.nloop, l0 + a.lchunk);
    const C* grow = G + static_cast<int64_t>(o1) * a.batch * a.W;
    const R cs = a.conj ? R(-1) : R(1);
    constexpr bool kSpread = rows_spread<A, B>();
    constexpr int NX = kSpread ? A : B;  // window entries of a lane
    int off[NX];
    SpreadRoots<R, kSpread ? B : 1> roots;
    if constexpr (kSpread) {
        spread_offsets<A, B>(a, s, static_cast<int>(f * a.sf + v) * a.W, live, off);
        __syncthreads();  // the twiddles
        roots.load(tw, A, s);
    } else {
        row_offsets<A, B>(a, s, static_cast<int>(f * a.sf + v) * a.W, live && s < A, off);
    }
    // the next row's window is loaded one row ahead where the registers allow it
    // (a long prime's DFT holds its entries twice)
    constexpr bool kAhead = kSpread || sizeof(R) * (A * NCH + (B > 16 ? 5 : 3) * B) <= 8 * 56;
    C x[NX];
    auto load = [&](int l) {
        const C* in = grow + static_cast<int64_t>(l) * a.sl * a.W;
#pragma unroll
        for (int k2 = 0; k2 < NX; ++k2) x[k2] = off[k2] >= 0 ? in[static_cast<unsigned>(off[k2])] : mk(R(0), R(0));
    };
    if (kAhead && l0 < l1) load(l0);
    for (int ls = l0; ls < l1; ls += a.stage) {
        const int count = min(a.stage, l1 - ls);
        __syncthreads();
        stage_row_coefficients<R, NCH>(sc, Coef, kmap, a, o1, ls, count);
        __syncthreads();
        for (int l = 0; l < count; ++l) {
            if (!kAhead) load(ls + l);
            C y[NX], w[A];
#pragma unroll
            for (int i = 0; i < NX; ++i) y[i] = x[i];
            if (kAhead && ls + l + 1 < l1) load(ls + l + 1);
            if constexpr (kSpread) {
                rows_spread_dft<R, A, B, 1>(xb, gi < GW, s, y, roots, w);
#pragma unroll
                for (int k1 = 1; k1 < A; ++k1) w[k1] = cmul(w[k1], cconj(tw[s * k1]));
            } else {
                dft_len<R, B, 1>(y);
                if (s < A) {
#pragma unroll
                    for (int i = 1; i < B; ++i) y[i] = cmul(y[i], cconj(tw[i * s]));
                }
                rows_exchange<R, B, A>(
                    xb, gi < GW && s < A, y, [&](int i) { return i * AP + s; }, gi < GW, w,
                    [&](int i) { return s * AP + i; });
            }
            dft_len<R, A, 1>(w);
#pragma unroll
            for (int j = 0; j < A; ++j)
#pragma unroll
                for (int c = 0; c < NCH; ++c) {
                    C q = sc[(l * NCH + c) * n + B * j + s];
                    q.y *= cs;
                    cfma(t[j][c], q, w[j]);
                }
        }
    }
    if (live) {
        const size_t base = (static_cast<size_t>(blockIdx.z) * a.nvec + v) * NCH;
#pragma unroll
        for (int j = 0; j < A; ++j) {
            const int k = kmap[B * j + s + n * o1];
            if (k < 0) continue;
#pragma unroll
            for (int c = 0; c < NCH; ++c) T[((base + c) * a.nfix + f) * a.nk + k] = t[j][c];
        }
    }
}

// The spectrum of column u = b W + j: entry xi_1 at [xi_1 W].
template <typename R>
__device__ inline const R* spectrum_of(const LatticeDesc& lat, int W, int nvec, int64_t u, int n, const R* P) {
    const int64_t b = u / W;
    const int j = static_cast<int>(u - b * W);
    const int ab = static_cast<int>(b / nvec);
    const int al = ab / lat.norb, be = ab - al * lat.norb;
    int pa = 0, pb = 0;
    while (al >= lat.orb_begin[pa + 1]) ++pa;
    while (be >= lat.orb_begin[pb + 1]) ++pb;
    return P + static_cast<int64_t>(pa + lat.natoms * pb) * n * W + j;
}

// Columns u = b W + j of G (length n, stride count = batch W): transform along o1, times the real
// spectrum P[(pa n + xi_1) W + j] of the atom pair of b, inverse; in place. SPECTRUM false:
// forward transform only, frequency xi_1 left at row xi_1. Lane (s, column) holds rows B j2 + s,
// then frequency k1 = s of the first step. T = col_group(A, B): grid ceil(count / T), block T B, dynamic LDS
// (n + T n) entries.
template <typename R, int A, int B, bool SPECTRUM>
__global__ __launch_bounds__(col_group(A, B) * B) void conv_columns_kernel(LatticeDesc lat, int W, int64_t count, int nvec,
                                                                    const double2* __restrict__ root,
                                                                    const R* __restrict__ P, cx_t<R>* __restrict__ G) {
    using C = cx_t<R>;
    constexpr int n = A * B, T = col_group(A, B);
    extern __shared__ unsigned char rows_raw[];
    C* tw = reinterpret_cast<C*>(rows_raw);
    C* ex = tw + n;
    const int c = threadIdx.x % T, s = threadIdx.x / T;
    const int64_t u = static_cast<int64_t>(blockIdx.x) * T + c;
    const bool live = u < count;
    C* g = G + (live ? u : count - 1);
    load_twiddles<R>(tw, root, n, T * B);
    {
        C v[A];
#pragma unroll
        for (int j = 0; j < A; ++j) v[j] = g[static_cast<int64_t>(B * j + s) * count];
        __syncthreads();  // the twiddles
        dft_len<R, A, -1>(v);
#pragma unroll
        for (int k = 0; k < A; ++k) ex[(s * A + k) * T + c] = k ? cmul(v[k], tw[s * k]) : v[k];
    }
    __syncthreads();
    if constexpr (rows_spread<A, B>() && A <= 2) {
        // the long prime's step spread over the lanes of a column (as in the row kernels; from A = 3 on
        // the whole transforms per lane are the faster ones here: 87 x 87 and 124 x 124 products
        // 3.0 against 3.6 ms and 6.2 against 7.8)
        SpreadRoots<R, B> roots;
        roots.load(tw, A, s);
        C v[A];
        auto spread = [&](auto sign) {
            constexpr int SG = decltype(sign)::value;
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) {
                C p = ex[k1 * T + c], q = mk(R(0), R(0));
#pragma unroll
                for (int j = 1; j <= (B - 1) / 2; ++j) {
                    const C x = ex[(j * A + k1) * T + c], y = ex[((B - j) * A + k1) * T + c];
                    p = mk(p.x + roots.c[j - 1] * (x.x + y.x), p.y + roots.c[j - 1] * (x.y + y.y));
                    q = mk(q.x + roots.s[j - 1] * (x.x - y.x), q.y + roots.s[j - 1] * (x.y - y.y));
                }
                v[k1] = spread_value<R, SG>(p, q);
            }
        };
        spread(std::integral_constant<int, -1>{});
        if constexpr (SPECTRUM) {
            const R* p = spectrum_of(lat, W, nvec, live ? u : count - 1, n, P);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) {
                const R f = p[static_cast<int64_t>(k1 + A * s) * W];
                v[k1].x *= f;
                v[k1].y *= f;
            }
            __syncthreads();  // every lane has read the entries
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) ex[(s * A + k1) * T + c] = v[k1];
            __syncthreads();
            spread(std::integral_constant<int, 1>{});
#pragma unroll
            for (int k1 = 1; k1 < A; ++k1) v[k1] = cmul(v[k1], cconj(tw[s * k1]));
            dft_len<R, A, 1>(v);
            if (live) {
#pragma unroll
                for (int j = 0; j < A; ++j) g[static_cast<int64_t>(B * j + s) * count] = v[j];
            }
        } else if (live) {
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) g[static_cast<int64_t>(k1 + A * s) * count] = v[k1];
        }
        return;
    } else {
        C v[B];
        if (s < A) {
#pragma unroll
            for (int i = 0; i < B; ++i) v[i] = ex[(i * A + s) * T + c];
            dft_len<R, B, -1>(v);
            if constexpr (SPECTRUM) {
                const R* p = spectrum_of(lat, W, nvec, live ? u : count - 1, n, P);
#pragma unroll
                for (int k = 0; k < B; ++k) {
                    const R q = p[static_cast<int64_t>(s + A * k) * W];
                    v[k].x *= q;
                    v[k].y *= q;
                }
                dft_len<R, B, 1>(v);
#pragma unroll
                for (int i = 1; i < B; ++i) v[i] = cmul(v[i], cconj(tw[i * s]));
            } else if (live) {
#pragma unroll
                for (int k = 0; k < B; ++k) g[static_cast<int64_t>(s + A * k) * count] = v[k];
            }
        }
        if constexpr (SPECTRUM) {
            // a lane writes the slots that it read itself
            if (s < A) {
#pragma unroll
                for (int i = 0; i < B; ++i) ex[(i * A + s) * T + c] = v[i];
            }
            __syncthreads();
            C w[A];
#pragma unroll
            for (int k = 0; k < A; ++k) w[k] = ex[(s * A + k) * T + c];
            dft_len<R, A, 1>(w);
            if (live) {
#pragma unroll
                for (int j = 0; j < A; ++j) g[static_cast<int64_t>(B * j + s) * count] = w[j];
            }
        }
    }
}

// Launchers (one source file per precision and kernel, to build them in parallel). A side
// without a factor pair or more than four channels throws.
template <typename R>
void launch_rows_in(RowsArgs a, int nch, const int* kmap, const double2* root, const cx_t<R>* Coef, const cx_t<R>* U,
                    cx_t<R>* G, hipStream_t s);
// chunks: chunks of the looped orbitals, each with its own part of T (see rows_out_chunks).
template <typename R>
void launch_rows_out(RowsArgs a, int nch, int chunks, const int* kmap, const double2* root, const cx_t<R>* Coef,
                     const cx_t<R>* G, cx_t<R>* T, hipStream_t s);
template <typename R>
void launch_columns(const LatticeDesc& lat, int W, int64_t count, int nvec, const double2* root, const R* P,
                    cx_t<R>* G, bool spectrum, hipStream_t s);

// Chunks of the looped orbitals for about `aim` workgroups.
inline int rows_chunks(const RowsArgs& a, int aim, int most) {
    int A = 0, B = 0;
    fft_factors(a.n, A, B);
    const int per = kRowWaves * (64 / B);
    const int64_t wgs = static_cast<int64_t>((a.nfix * a.nvec + per - 1) / per) * a.n;
    const int c = static_cast<int>((aim + wgs - 1) / wgs);
    const int chunks = c < 1 ? 1 : (c > most ? most : c);
    const int len = (a.nloop + chunks - 1) / chunks;
    return (a.nloop + len - 1) / len;
}
// Parts of T: one per chunk, so few.
inline int rows_out_chunks(const RowsArgs& a) { return rows_chunks(a, 512, a.nloop < 6 ? a.nloop : 6); }

// Stages of the looped orbitals that keep the LDS near 40 KB (four workgroups per CU).
template <typename R, int A, int B, int NCH>
int rows_stage(int lchunk) {
    const size_t fixed = rows_lds_bytes<R, A, B, NCH>(0), per = sizeof(cx_t<R>) * NCH * A * B;
    const size_t room = fixed < 40 * 1024 ? 40 * 1024 - fixed : 0;
    const int fit = static_cast<int>(room / per);
    const int most = fit < 1 ? 1 : (fit < lchunk ? fit : lchunk);
    const int stages = (lchunk + most - 1) / most;
    return (lchunk + stages - 1) / stages;
}

}  // namespace xatu_dev
