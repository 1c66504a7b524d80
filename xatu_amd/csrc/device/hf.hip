// Hellmann-Feynman gradients of exciton energies with respect to the screening
// parameters (r0, eps_m, eps_s), without forming dH.
//
// For a normalised eigenvector psi, dE/dtheta = psi^H (dH/dtheta) psi with
// dH = -(dD - dX). The direct term's formula is Hermitian under swapping the pair
// (the lattice sums satisfy M(-q) = conj M(q) with the reference's conjugation
// convention), so psi^H dD psi is the full double sum
//   sum_{k,k'} sum_ab dM_ab(k'-k) G_ab(k,k'),
//   G_ab(k,k') = sum_{c v c' v'} conj(psi_kcv) rho^c_a(ck,c'k') rho^v_b(v'k',vk) psi_k'c'v'.
// Grouping the pairs by q = k'-k gives the adjoint of the pair densities,
// S_ab(q) = sum_k G_ab(k, k+q) (one workgroup per mesh point q, deterministic);
// the adjoint of the lattice sum then maps S to the cell table,
//   Shat_p(R) = sum_q [S_ab(q) e^{iqR} + S_ba(q) e^{-iqR}]  (a < b),
//   Shat_p(R) = sum_q S_aa(q) e^{-iqR}                        (a = b),
// and psi^H dD psi = (1/T) sum_p sum_R dV_p(R) Shat_p(R) for any parameter, with
// dV from the analytic derivative of the potential (FP64). The exchange formula
// X(i,j) = sum_ab f_a(i) MQ_ab g_b(j) is not Hermitian when V(Q) has a complex
// diagonal (Q != 0 with a cell set that is not inversion-symmetric), so it follows
// the reference's construction H = A + A^H from the upper triangle:
//   psi^H dX psi = Re sum_ab dMQ_ab (2 P_ab + G_ab),
//   P_ab = sum_j (sum_{i<j} f_a(i)) g_b(j),  G_ab = sum_i f_a(i) g_b(i),
// with f_a(i) = conj(psi_i) rho1_a(i), g_b(j) = rho2_b(j) psi_j (prefixes by runs of rows).
#include <cmath>
#include <vector>

#include "context.hpp"
#include "cplx.hpp"
#include "wave_sums.hpp"
#include "potential_dev.hpp"

namespace xatu_dev {

namespace {

constexpr int kHfThreads = 256;
constexpr int kHfStates = 4;  // states per pass of the pair-density adjoint
constexpr int kHfRowStates = 8;  // ... when it runs on the row and column transforms

// dV/dtheta for pair p and cell R. which: 0 r0, 1 eps (m or s: identical).
__global__ void dpotential_table_kernel(LatticeDesc lat, PotDesc pot, const int* __restrict__ cells, int nR, int npairs,
                                        int which, const double* __restrict__ gl, double* __restrict__ out) {
    const int R = blockIdx.x * blockDim.x + threadIdx.x;
    const int p = blockIdx.y;
    if (R >= nR || p >= npairs) return;
    int a = 0, rem = p;
    while (rem >= lat.natoms - a) {
        rem -= lat.natoms - a;
        ++a;
    }
    const int b = a + rem;
    const double r = cell_distance(lat, cells + 3 * R, a, b);
    double d = 0.0;
    if (pot.kind == XATU_POTENTIAL_KELDYSH) {
        d = (which == 0) ? keldysh_dr0(r, pot, gl) : -potential(r, pot) / (2.0 * pot.eps_bar);
    }
    out[static_cast<size_t>(p) * nR + R] = d;
}

// S[s][q][a + na b] for states [s0, s0 + ns): one workgroup per mesh point q.
// kmap[linear mesh offset] = k index or -1; psi: N x nstates column-major.
__global__ __launch_bounds__(kHfThreads) void pair_adjoint_kernel(LatticeDesc lat, int nk, int nv, int nc,
                                                                  const double2* __restrict__ evk,
                                                                  const double2* __restrict__ evkq,
                                                                  const int* __restrict__ kcoord,
                                                                  const int* __restrict__ kmap,
                                                                  const double2* __restrict__ psi, int64_t N, int s0,
                                                                  int ns, double2* __restrict__ S) {
    const int q = blockIdx.x;
    const int n = lat.mesh_n;
    const int na = lat.natoms;
    const int nb = nv + nc;
    const int ncv = nc * nv;
    const int norb = lat.norb;
    // mesh coordinates of q -> offset delta (q = (delta + n/2) mod n per axis)
    int dq[3] = {0, 0, 0};
    {
        int rem = q;
        for (int j = 0; j < lat.ndim; ++j) {
            dq[j] = rem % n - n / 2;
            rem /= n;
        }
    }
    __shared__ double2 red[kHfThreads];
    for (int a = 0; a < na; ++a) {
        for (int b = 0; b < na; ++b) {
            double2 acc[kHfStates];
#pragma unroll
            for (int st = 0; st < kHfStates; ++st) acc[st] = mk(0.0, 0.0);
            for (int k = threadIdx.x; k < nk; k += blockDim.x) {
                int lin = 0, mul = 1;
                for (int j = 0; j < lat.ndim; ++j) {
                    int o = (kcoord[3 * k + j] + dq[j]) % n;
                    if (o < 0) o += n;
                    lin += o * mul;
                    mul *= n;
                }
                const int k2 = kmap[lin];
                if (k2 < 0) continue;
                const double2* Ck = evkq + static_cast<size_t>(k) * nb * norb;
                const double2* Vk = evk + static_cast<size_t>(k) * nb * norb;
                const double2* Ck2 = evkq + static_cast<size_t>(k2) * nb * norb;
                const double2* Vk2 = evk + static_cast<size_t>(k2) * nb * norb;
                // G_ab = sum_{c,c'} rho^c_a(c,c') sum_{v,v'} conj(psi_kcv) rho^v_b(v',v) psi_k'c'v'
                for (int c = 0; c < nc; ++c) {
                    for (int c2 = 0; c2 < nc; ++c2) {
                        double2 rc = mk(0.0, 0.0);
                        for (int al = lat.orb_begin[a]; al < lat.orb_begin[a + 1]; ++al)
                            cfma_conj(rc, Ck[(nv + c) * norb + al], Ck2[(nv + c2) * norb + al]);
                        for (int v = 0; v < nv; ++v) {
                            for (int v2 = 0; v2 < nv; ++v2) {
                                double2 rv = mk(0.0, 0.0);
                                for (int be = lat.orb_begin[b]; be < lat.orb_begin[b + 1]; ++be)
                                    cfma_conj(rv, Vk2[v2 * norb + be], Vk[v * norb + be]);
                                const double2 w = cmul(rc, rv);
                                const int64_t i = static_cast<int64_t>(k) * ncv + c * nv + v;
                                const int64_t j = static_cast<int64_t>(k2) * ncv + c2 * nv + v2;
#pragma unroll
                                for (int st = 0; st < kHfStates; ++st) {
                                    if (st < ns) {
                                        const double2 pi = psi[i + static_cast<int64_t>(s0 + st) * N];
                                        const double2 pj = psi[j + static_cast<int64_t>(s0 + st) * N];
                                        double2 t = mk(0.0, 0.0);
                                        cfma_conj(t, pi, pj);
                                        cfma(acc[st], t, w);
                                    }
                                }
                            }
                        }
                    }
                }
            }
            // block reduction, one state at a time
            for (int st = 0; st < ns; ++st) {
                double2 mine = mk(0.0, 0.0);
#pragma unroll
                for (int u = 0; u < kHfStates; ++u)
                    if (u == st) mine = acc[u];
                red[threadIdx.x] = mine;
                __syncthreads();
                for (int stp = kHfThreads / 2; stp > 0; stp >>= 1) {
                    if (threadIdx.x < stp) red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + stp]);
                    __syncthreads();
                }
                if (threadIdx.x == 0) S[(static_cast<size_t>(st) * lat.nmesh + q) * na * na + a + na * b] = red[0];
                __syncthreads();
            }
        }
    }
}

// Shat[s][p][R] from S (adjoint of the lattice sum), for ns states.
// grid: (ceil(nR/256), npairs, ns)
__global__ void adjoint_fourier_kernel(LatticeDesc lat, const int* __restrict__ cells, int nR, int npairs,
                                       const double2* __restrict__ S, const double2* __restrict__ tw,
                                       double* __restrict__ shat) {
    const int R = blockIdx.x * blockDim.x + threadIdx.x;
    const int p = blockIdx.y;
    const int s = blockIdx.z;
    if (R >= nR) return;
    int a = 0, rem = p;
    while (rem >= lat.natoms - a) {
        rem -= lat.natoms - a;
        ++a;
    }
    const int b = a + rem;
    const int na = lat.natoms;
    const int n = lat.mesh_n;
    const int two_n = 2 * n;
    double sum = 0.0;
    for (int q = 0; q < lat.nmesh; ++q) {
        long long ph = 0;
        int rem2 = q;
        for (int j = 0; j < lat.ndim; ++j) {
            const int cj = rem2 % n;
            rem2 /= n;
            ph += static_cast<long long>(2 * cj - n + (n & 1)) * cells[3 * R + j];
        }
        int idx = static_cast<int>(ph % two_n);
        if (idx < 0) idx += two_n;
        const double2 w = tw[idx];  // exp(i q.R)
        const double2* Sq = S + (static_cast<size_t>(s) * lat.nmesh + q) * na * na;
        if (a < b) {
            const double2 sab = Sq[a + na * b], sba = Sq[b + na * a];
            // Re[S_ab e^{iqR} + S_ba e^{-iqR}]
            sum += (sab.x * w.x - sab.y * w.y) + (sba.x * w.x + sba.y * w.y);
        } else {
            const double2 saa = Sq[a + na * a];
            sum += saa.x * w.x + saa.y * w.y;  // Re[S_aa e^{-iqR}]
        }
    }
    shat[(static_cast<size_t>(s) * npairs + p) * nR + R] = sum;
}

// Exchange rows: fg[(s*N + i)*2*na + a] = f_a(i), [.. + na + a] = g_a(i) for state s.
// grid: (ceil(N/256), nstates)
__global__ void exchange_rows_kernel(LatticeDesc lat, int nk, int nv, int nc, const double2* __restrict__ evk,
                                     const double2* __restrict__ evkq, const double2* __restrict__ e1,
                                     const double2* __restrict__ psi, int64_t N, double2* __restrict__ fg) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int s = blockIdx.y;
    if (i >= N) return;
    const int na = lat.natoms;
    const int nb = nv + nc, ncv = nc * nv;
    const int k = static_cast<int>(i / ncv), cv = static_cast<int>(i % ncv);
    const int c = cv / nv, v = cv % nv;
    const double2 p = psi[i + static_cast<int64_t>(s) * N];
    const double2* vk = evk + (static_cast<size_t>(k) * nb + v) * lat.norb;
    const double2* ck = evkq + (static_cast<size_t>(k) * nb + nv + c) * lat.norb;
    double2* out = fg + (static_cast<size_t>(s) * N + i) * 2 * na;
    for (int a = 0; a < na; ++a) {
        double2 f = mk(0.0, 0.0);
        cfma_conj(f, p, e1[(static_cast<size_t>(k) * na + a) * ncv + cv]);
        double2 r2 = mk(0.0, 0.0);
        for (int al = lat.orb_begin[a]; al < lat.orb_begin[a + 1]; ++al) cfma_conj(r2, vk[al], ck[al]);
        out[a] = f;
        out[na + a] = cmul(r2, p);
    }
}

// Sum over the workgroup's 256 threads, the same in every thread.
__device__ inline double group_sum(double x, double* red) {
    x = wave_sum(x);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// W[s][a + na b] = 2 P_ab + G_ab, P_ab = sum_{j < i} f_a(j) g_b(i), G_ab = sum_i f_a(i) g_b(i): the
// exchange sums along the upper triangle. A thread has a run of rows; the runs' sums of f are
// scanned in LDS, which gives each its prefix. grid (states, na), block 256. Bound by the latency of a thread's
// loads: N = 5184, 3 atoms, 8 states: 20 us (on the host these sums, the contractions below and their
// read-backs took 2.4 of the 2.8 ms of a call).
__global__ __launch_bounds__(256) void exchange_sums_kernel(int na, int64_t N, const double2* __restrict__ fg,
                                                            double2* __restrict__ W) {
    __shared__ double2 s_run[256];
    __shared__ double red[4];
    const int st = blockIdx.x, a = blockIdx.y, t = threadIdx.x;
    const int64_t run = (N + 255) / 256, i0 = min(N, t * run), i1 = min(N, i0 + run);
    const double2* row = fg + static_cast<size_t>(st) * N * 2 * na;
    double2 total = mk(0.0, 0.0);
#pragma unroll 4
    for (int64_t i = i0; i < i1; ++i) total = cadd(total, row[i * 2 * na + a]);
    s_run[t] = total;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
        const double2 v = t >= d ? s_run[t - d] : mk(0.0, 0.0);
        __syncthreads();
        s_run[t] = cadd(s_run[t], v);
        __syncthreads();
    }
    const double2 before = t > 0 ? s_run[t - 1] : mk(0.0, 0.0);
    for (int b = 0; b < na; ++b) {
        double2 F = before, P = mk(0.0, 0.0), G = mk(0.0, 0.0);
#pragma unroll 4
        for (int64_t i = i0; i < i1; ++i) {
            const double2 f = row[i * 2 * na + a], g = row[i * 2 * na + na + b];
            cfma(P, F, g);
            cfma(G, f, g);
            F = cadd(F, f);
        }
        const double re = group_sum(2.0 * P.x + G.x, red), im = group_sum(2.0 * P.y + G.y, red);
        if (t == 0) W[static_cast<size_t>(st) * na * na + a + na * b] = mk(re, im);
    }
}

// Contractions of the derivative tables: out[s] = sum_e dv[e] Shat[s][e] (workgroup per state), and after them
// per pair sum_R dvx_p(R) e^{iQ R} as two values. block 256
__global__ __launch_bounds__(256) void gradient_sums_kernel(LatticeDesc lat, int nstates, int npairs, int nR,
                                                            const double* __restrict__ dv,
                                                            const double* __restrict__ dvx,
                                                            const double* __restrict__ shat,
                                                            const int* __restrict__ cells, double qx, double qy,
                                                            double qz, double* __restrict__ out) {
    __shared__ double red[4];
    if (static_cast<int>(blockIdx.x) < nstates) {
        const int64_t n = static_cast<int64_t>(npairs) * nR;
        const double* sh = shat + blockIdx.x * n;
        double sum = 0.0;
#pragma unroll 4
        for (int64_t e = threadIdx.x; e < n; e += 256) sum += dv[e] * sh[e];
        sum = group_sum(sum, red);
        if (threadIdx.x == 0) out[blockIdx.x] = sum;
        return;
    }
    const int p = blockIdx.x - nstates;
    double mr = 0.0, mi = 0.0;
    for (int R = threadIdx.x; R < nR; R += 256) {
        double v[3] = {0.0, 0.0, 0.0};
        for (int j = 0; j < lat.ndim; ++j)
            for (int x = 0; x < 3; ++x) v[x] += static_cast<double>(cells[3 * R + j]) * lat.bravais[3 * j + x];
        double si, co;
        sincos(qx * v[0] + qy * v[1] + qz * v[2], &si, &co);
        const double d = dvx[static_cast<int64_t>(p) * nR + R];
        mr += d * co;
        mi += d * si;
    }
    mr = group_sum(mr, red);
    mi = group_sum(mi, red);
    if (threadIdx.x == 0) {
        out[nstates + 2 * p] = mr;
        out[nstates + 2 * p + 1] = mi;
    }
}

}  // namespace

void hf_gradients(Context& c, int nstates, const double2* d_vec, int nparams, const int* params, double* grad_out) {
    if (!c.prepared) throw Error(XATU_ERR_LOGIC, "operator not prepared (call xatu_build_bse)");
    const int na = c.lat.natoms;
    const int npairs = na * (na + 1) / 2;
    const int nR = c.nR;
    const double T = static_cast<double>(c.inter.total_cells);
    hipStream_t s = c.stream;

    const bool direct = c.lat.ndim == 2 && conv_rows_available(c);
    DevBuf<int> d_kmap;
    DevBuf<double2> S;
    if (!direct) {
        // pair-density adjoint of kHfStates states at a time; k -> mesh-offset map
        const int n = c.lat.mesh_n;
        std::vector<int> kmap(c.lat.nmesh, -1);
        for (int k = 0; k < c.nk; ++k) {
            int lin = 0, mul = 1;
            for (int j = 0; j < c.lat.ndim; ++j) {
                int o = c.h_koff[k * c.lat.ndim + j] % n;
                if (o < 0) o += n;
                lin += o * mul;
                mul *= n;
            }
            kmap[lin] = k;
        }
        d_kmap.alloc(kmap.size());
        XATU_HIP(hipMemcpyAsync(d_kmap.p, kmap.data(), kmap.size() * sizeof(int), hipMemcpyHostToDevice, s));
        S.alloc(static_cast<size_t>(kHfStates) * c.lat.nmesh * na * na);
        XATU_HIP(hipStreamSynchronize(s));  // the map goes
    }

    // the lattice adjoint Shat of every state
    DevBuf<double> shat;
    shat.alloc(static_cast<size_t>(nstates) * npairs * nR);
    const int step = direct ? kHfRowStates : kHfStates;
    for (int s0 = 0; s0 < nstates; s0 += step) {
        const int ns = std::min(step, nstates - s0);
        if (direct) {
            // the cells' adjoint is the power spectrum of the transforms: no sums over q
            conv_cell_density(c, d_vec + static_cast<int64_t>(s0) * c.N, ns,
                              shat.p + static_cast<size_t>(s0) * npairs * nR);
            continue;
        }
        if (c.lat.ndim <= 2) {
            // autocorrelation on the mesh with FFTs: O(norb^2 M log M) instead of O(nk^2) pairs
            conv_pair_density(c, d_vec + static_cast<int64_t>(s0) * c.N, ns, S.p);
        } else {
            hipLaunchKernelGGL(pair_adjoint_kernel, dim3(c.lat.nmesh), dim3(kHfThreads), 0, s, c.lat, c.nk, c.nv,
                               c.nc, c.d_evec_k.p, c.d_evec_kq.p, c.d_kcoord.p, d_kmap.p, d_vec, c.N, s0, ns, S.p);
        }
        hipLaunchKernelGGL(adjoint_fourier_kernel, dim3((nR + 255) / 256, npairs, ns), dim3(256), 0, s, c.lat,
                           c.d_cells.p, nR, npairs, S.p, c.d_twiddle.p,
                           shat.p + static_cast<size_t>(s0) * npairs * nR);
        XATU_HIP(hipGetLastError());
    }
    const bool exchange = c.inter.exchange;
    DevBuf<double2> fg, Wx;
    if (exchange) {
        fg.alloc(static_cast<size_t>(nstates) * c.N * 2 * na);
        Wx.alloc(static_cast<size_t>(nstates) * na * na);
        hipLaunchKernelGGL(exchange_rows_kernel, dim3((c.N + 255) / 256, nstates), dim3(256), 0, s, c.lat, c.nk, c.nv,
                           c.nc, c.d_evec_k.p, c.d_evec_kq.p, c.d_e1.p, d_vec, c.N, fg.p);
        hipLaunchKernelGGL(exchange_sums_kernel, dim3(nstates, na), dim3(256), 0, s, na, c.N, fg.p, Wx.p);
        XATU_HIP(hipGetLastError());
    }
    // quadrature rule of the dV/dr0 evaluation
    static const std::vector<double> h_gl = [] {
        std::vector<double> r(2 * kGlNodes);
        gauss_legendre_rule(r.data());
        return r;
    }();
    // derivative tables of one parameter (direct, exchange), their contractions for all parameters
    const size_t ntab = static_cast<size_t>(npairs) * nR, nout = static_cast<size_t>(nstates) + 2 * npairs;
    DevBuf<double> work;
    work.alloc(h_gl.size() + 2 * ntab + nout * nparams);
    double *gl = work.p, *dv = gl + h_gl.size(), *dvx = dv + ntab, *out = dvx + ntab;
    XATU_HIP(hipMemcpyAsync(gl, h_gl.data(), h_gl.size() * sizeof(double), hipMemcpyHostToDevice, s));
    for (int ip = 0; ip < nparams; ++ip) {
        const int which = (params[ip] == XATU_PARAM_R0) ? 0 : 1;
        hipLaunchKernelGGL(dpotential_table_kernel, dim3((nR + 255) / 256, npairs), dim3(256), 0, s, c.lat, c.pot_d,
                           c.d_cells.p, nR, npairs, which, gl, dv);
        if (exchange)
            hipLaunchKernelGGL(dpotential_table_kernel, dim3((nR + 255) / 256, npairs), dim3(256), 0, s, c.lat,
                               c.pot_x, c.d_cells.p, nR, npairs, which, gl, dvx);
        hipLaunchKernelGGL(gradient_sums_kernel, dim3(nstates + (exchange ? npairs : 0)), dim3(256), 0, s, c.lat, nstates,
                           npairs, nR, dv, dvx, shat.p, c.d_cells.p, c.inter.Q[0], c.inter.Q[1], c.inter.Q[2],
                           out + nout * ip);
        XATU_HIP(hipGetLastError());
    }
    std::vector<double> h_out(nout * nparams);
    std::vector<double2> h_W(static_cast<size_t>(nstates) * na * na);
    XATU_HIP(hipMemcpyAsync(h_out.data(), out, h_out.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    if (exchange) XATU_HIP(hipMemcpyAsync(h_W.data(), Wx.p, Wx.bytes(), hipMemcpyDeviceToHost, s));
    XATU_HIP(hipStreamSynchronize(s));
    for (int ip = 0; ip < nparams; ++ip)
        for (int st = 0; st < nstates; ++st) {
            // direct: psi^H dD psi = (1/T) sum_p sum_R dV_p(R) Shat_p(R)
            const double dd = h_out[nout * ip + st] / T;
            // exchange: Re sum_ab dMQ_ab W_ab, with dMQ_ab = (1/T) sum_R dV_p(R) e^{iQR} (a < b),
            // dMQ_ba and dMQ_aa with e^{-iQR} (lower triangle and diagonal by conjugation)
            double dx = 0.0;
            if (exchange) {
                const double2* W = h_W.data() + static_cast<size_t>(st) * na * na;
                const double* m = h_out.data() + nout * ip + nstates;
                for (int a = 0; a < na; ++a)
                    for (int b = a; b < na; ++b, m += 2) {
                        if (a < b) {
                            const double2 wab = W[a + na * b], wba = W[b + na * a];
                            dx += (m[0] * wab.x - m[1] * wab.y) + (m[0] * wba.x + m[1] * wba.y);
                        } else {
                            const double2 waa = W[a + na * a];
                            dx += m[0] * waa.x + m[1] * waa.y;
                        }
                    }
                dx /= T;
            }
            grad_out[static_cast<size_t>(ip) * nstates + st] = -(dd - dx);
        }
}

}  // namespace xatu_dev
