// Streaming and small kernels of the chi0 -> Ec path (gfx950).
#include "kernels.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <tuple>

#include "gemm.h"

namespace lra {

// ------------------------------------------------------------------------------------
// G build helpers
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void scale_bands_kernel(const double *__restrict__ wre,
                                                          const double *__restrict__ wim,
                                                          const double *__restrict__ eps,
                                                          const double *__restrict__ wg, double *__restrict__ Zs,
                                                          int nk, int nbands, int nbasis, int lo0, int hi0, int lo1,
                                                          int hi1, TauList taus, double efermi, int nspin,
                                                          int nbands_g) {
    const int k = blockIdx.y, sg = blockIdx.z & 1, b0 = sg ? lo1 : lo0, b1 = sg ? hi1 : hi0;
    const long long per_k = (long long)(b1 - b0) * nbasis;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= per_k) return;
    const double tau = sg ? -taus.t[blockIdx.z >> 1] : taus.t[blockIdx.z >> 1];
    const int b = b0 + (int)(idx / nbasis);
    const int j = (int)(idx % nbasis);
    const double e = eps[(long long)k * nbands + b];
    const double g = wg[(long long)k * nbands + b];
    double w;
    if (tau > 0) {
        w = 1.0 / nk - g / 2 * nspin;
        if (w < 0) w = 0;
    } else {
        w = g * 0.5 * nspin;
    }
    double sc = -tau * (e - efermi);
    if (sc > 0) sc = 0;
    double sb = exp(sc) * w;
    if (nbands_g >= 0 && b >= nbands_g) sb = 0;
    const long long src = ((long long)k * nbands + b) * nbasis + j;
    double *z = Zs + ((long long)blockIdx.z * nk + k) * 2 * nbands * nbasis;
    z[(2ll * b) * nbasis + j] = sb * wre[src];
    z[(2ll * b + 1) * nbasis + j] = sb * wim[src];
}

void launch_scale_bands(const double *wre, const double *wim, const double *eps, const double *wg, double *Zs, int nk,
                        int nbands, int nbasis, const int b0[2], const int b1[2], const TauList &taus, double efermi,
                        int nspin, int nbands_g, hipStream_t s) {
    const long long per_k = (long long)std::max(b1[0] - b0[0], b1[1] - b0[1]) * nbasis;
    if (per_k <= 0 || taus.n <= 0) return;
    hipLaunchKernelGGL(scale_bands_kernel, dim3(ceil_div(per_k, 256), nk, 2 * taus.n), dim3(256), 0, s, wre, wim, eps,
                       wg, Zs, nk, nbands, nbasis, b0[0], b1[0], b0[1], b1[1], taus, efermi, nspin, nbands_g);
    HIP_CHECK(hipGetLastError());
}

// k -> R: a thread holds one (row, column) of kK2rCells cells, so that M is read once per group of
// cells and a small basis (17 functions on 27 k) still spreads over the device.  With one thread for
// all cells that case took 0.2 ms per tau point and sign on two workgroups.
constexpr int kK2rCells = 4;
template <class T>
__global__ __launch_bounds__(256) void k2r_kernel(const double *__restrict__ M, const double *__restrict__ cs,
                                                  const double *__restrict__ sn, const int *__restrict__ gcol,
                                                  T *__restrict__ G, int nk, int nR, int nbasis, TauList taus) {
    const long long nn = (long long)nbasis * nbasis;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nn) return;
    const int r0 = blockIdx.y * kK2rCells, z = blockIdx.z >> 1, sg = blockIdx.z & 1;
    // by the time itself, not by sg: a grid may hold tau = 0, where neither G changes sign
    const bool neg = sg ? taus.t[z] > 0 : taus.t[z] < 0;
    M += (long long)blockIdx.z * nk * 2 * nn;
    G += (long long)z * nR * 2 * nn;
    const int row = (int)(idx / nbasis), col = (int)(idx % nbasis);
    const long long dst = (long long)row * 2 * nbasis + gcol[sg * nbasis + col];
    double acc[kK2rCells];
#pragma unroll
    for (int i = 0; i < kK2rCells; ++i) acc[i] = 0;
    for (int k = 0; k < nk; ++k) {
        const double re = M[k * 2 * nn + idx], im = M[k * 2 * nn + nn + idx];
#pragma unroll
        for (int i = 0; i < kK2rCells; ++i) {
            const int r = min(r0 + i, nR - 1);
            acc[i] += cs[r * nk + k] * re + sn[r * nk + k] * im;
        }
    }
#pragma unroll
    for (int i = 0; i < kK2rCells; ++i)
        if (r0 + i < nR) G[(long long)(r0 + i) * 2 * nn + dst] = static_cast<T>(neg ? -acc[i] : acc[i]);
}

template <class T>
void launch_k2r(const double *Mstack, const double *cs, const double *sn, const int *gcol, T *Gpm, int nk, int nR,
                int nbasis, const TauList &taus, hipStream_t s) {
    const long long nn = (long long)nbasis * nbasis;
    hipLaunchKernelGGL((k2r_kernel<T>), dim3(ceil_div(nn, 256), ceil_div(nR, kK2rCells), 2 * taus.n), dim3(256), 0, s,
                       Mstack, cs, sn, gcol, Gpm, nk, nR, nbasis, taus);
    HIP_CHECK(hipGetLastError());
}
template void launch_k2r<double>(const double *, const double *, const double *, const int *, double *, int, int,
                                 int, const TauList &, hipStream_t);
template void launch_k2r<float>(const double *, const double *, const double *, const int *, float *, int, int,
                                int, const TauList &, hipStream_t);

template <class T>
__global__ void gather_cols_kernel(const T *__restrict__ src, long long src_ld, T *__restrict__ dst,
                                   const GatherJob *__restrict__ jobs, const long long *__restrict__ colsrc,
                                   int nrows, long long zs, long long zd) {
    const GatherJob J = jobs[blockIdx.y];
    src += blockIdx.z * zs;
    dst += blockIdx.z * zd;
    const long long n = (long long)nrows * J.ncol;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const int row = (int)(idx / J.ncol), c = (int)(idx % J.ncol);
        dst[J.dst_off + idx] = src[colsrc[J.col_off + c] + row * src_ld];
    }
}

template <class T>
void launch_gather_cols(const T *src, long long src_ld, T *dst, const GatherJob *jobs, int njobs,
                        const long long *colsrc, int nrows, int maxcol, hipStream_t s, int nz, long long zs,
                        long long zd) {
    if (njobs == 0) return;
    const long long n = (long long)nrows * maxcol;
    const int bx = std::min(ceil_div(n, 256), 2048);
    hipLaunchKernelGGL((gather_cols_kernel<T>), dim3(bx, njobs, nz), dim3(256), 0, s, src, src_ld, dst, jobs, colsrc,
                       nrows, zs, zd);
    HIP_CHECK(hipGetLastError());
}
template void launch_gather_cols<double>(const double *, long long, double *, const GatherJob *, int,
                                         const long long *, int, int, hipStream_t, int, long long, long long);
template void launch_gather_cols<float>(const float *, long long, float *, const GatherJob *, int,
                                        const long long *, int, int, hipStream_t, int, long long, long long);

// ------------------------------------------------------------------------------------
// chi0 (R, tau) -> dense chi0 (q, omega)
// ------------------------------------------------------------------------------------
// chi0(q, omega) element (row, col) and its Hermitian mirror in one of the dense layouts
template <class TD>
__device__ __forceinline__ void put_dense(TD *__restrict__ D, long long n, long long row, long long col, double re,
                                          double im, bool mirror, int lay) {
    D[row * n + col] = static_cast<TD>(re);
    if (mirror) D[col * n + row] = static_cast<TD>(re);
    if (lay == kPlanar) {
        D[(n + row) * n + col] = static_cast<TD>(im);
        if (mirror) D[(n + col) * n + row] = static_cast<TD>(-im);
    }
}

// NW accumulators per thread (a multiple of 8 covering the chunk): one pass over chi0(R, tau) per
// chunk of up to kChi0AssembleMaxW frequencies
template <class TS, class TD, int NW>
__global__ void chi0_assemble_kernel(const TS *__restrict__ chi0s, long long E_tot, int ntau,
                                     const PairDesc *__restrict__ pairs, int npairs, long long nelem,
                                     const long long *__restrict__ eoff, int nR, const double *__restrict__ gp,
                                     int nw, TD *__restrict__ dense, long long dstride, int n, int lay) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nelem) return;
    int lo = 0, hi = npairs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pairs[mid].e0 <= idx) lo = mid; else hi = mid - 1;
    }
    const PairDesc P = pairs[lo];
    const long long e = idx - P.e0;
    const int mu = (int)(e / P.naJ), nu = (int)(e % P.naJ);
    double re[NW], im[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) { re[w] = 0; im[w] = 0; }
    for (int r = 0; r < nR; ++r) {
        const long long off = eoff[(long long)lo * nR + r];
        if (off < 0) continue;
        for (int t = 0; t < ntau; ++t) {
            const double v = static_cast<double>(chi0s[(long long)t * E_tot + off + e]);
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w < nw) {
                    const double *g = gp + (((long long)w * nR + r) * ntau + t) * 2;
                    re[w] += g[0] * v;
                    im[w] += g[1] * v;
                }
            }
        }
    }
    const long long row = P.rowI + mu, col = P.colJ + nu;
    const bool mirror = P.I != P.J;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        if (w >= nw) break;
        put_dense(dense + w * dstride, n, row, col, re[w], im[w], mirror, lay);
    }
}

template <class TS, class TD>
void launch_chi0_assemble(const TS *chi0s, long long E_tot, int ntau, const PairDesc *pairs, int npairs,
                          long long n_pair_elems, const long long *eoff, int nR, const double *gam_ph, int nw,
                          TD *dense, long long dense_stride, int n, DenseLayout lay, hipStream_t s) {
    if (nw < 1 || nw > kChi0AssembleMaxW) LRA_THROW("omega chunk too large");
    hipLaunchKernelGGL((chi0_assemble_kernel<TS, TD, kChi0AssembleMaxW>), dim3(ceil_div(n_pair_elems, 256)), dim3(256),
                       0, s, chi0s, E_tot, ntau, pairs, npairs, n_pair_elems, eoff, nR, gam_ph, nw, dense, dense_stride,
                       n, (int)lay);
    HIP_CHECK(hipGetLastError());
}
template void launch_chi0_assemble<double, double>(const double *, long long, int, const PairDesc *, int, long long,
                                                   const long long *, int, const double *, int, double *, long long,
                                                   int, DenseLayout, hipStream_t);
template void launch_chi0_assemble<float, float>(const float *, long long, int, const PairDesc *, int, long long,
                                                 const long long *, int, const double *, int, float *, long long,
                                                 int, DenseLayout, hipStream_t);
template void launch_chi0_assemble<float, double>(const float *, long long, int, const PairDesc *, int, long long,
                                                  const long long *, int, const double *, int, double *, long long,
                                                  int, DenseLayout, hipStream_t);
template void launch_chi0_assemble<double, float>(const double *, long long, int, const PairDesc *, int, long long,
                                                  const long long *, int, const double *, int, float *, long long,
                                                  int, DenseLayout, hipStream_t);

// chiw[w][i] = sum_t coef[w][t] chi0s[t][i] for every element i of the chi0(R, tau) store: the
// cosine tau -> omega transform, done once for all q.  Coefficients in LDS; a thread owns one element
// and re-reads its ntau values once per group of 8 frequencies.  Where the elements alone are under 1024
// workgroups the groups go over the grid (a molecule: 17 us of load latency in one thread's two groups).
// A kernel takes its table as TAB (the ArgTable itself, or nothing) and a __restrict__ pointer: without
// that word a table in memory is read again by every lane after each store (16 atoms, 64 k: the R -> q sums
// 98 ms an evaluation, 44 to 50 with scalar loads).
struct NoArgTable {};
__device__ __forceinline__ double table_at(const ArgTable &t, const double *, int i) { return t.v[i]; }
__device__ __forceinline__ double table_at(const NoArgTable &, const double *p, int i) { return p[i]; }
// the table of a launch to the launch itself
template <class F> void with_table(const std::vector<double> &v, DevBuf &buf, hipStream_t s, F f) {
    if (v.size() <= (size_t)kArgTable) {
        ArgTable t;
        std::copy(v.begin(), v.end(), t.v);
        f(t, static_cast<const double *>(nullptr));
        return;
    }
    buf.reserve(v.size() * sizeof(double));
    HIP_CHECK(hipMemcpyAsync(buf.get(), v.data(), v.size() * sizeof(double), hipMemcpyHostToDevice, s));
    f(NoArgTable(), static_cast<const double *>(buf.as<double>()));
    HIP_CHECK(hipStreamSynchronize(s));  // the next table may go to the same buffer
}

template <class TS, class TAB>
__global__ __launch_bounds__(256) void tau_to_omega_kernel(const TS *__restrict__ chi0s, long long E_tot, int ntau,
                                                           const TAB tab, const double *__restrict__ coef, int nw, int wper,
                                                           double *__restrict__ chiw) {
    __shared__ double c[kTauOmegaMax * kTauOmegaMax];
    const int wb = blockIdx.y * wper, we = min(nw, wb + wper);
    for (int k = wb * ntau + threadIdx.x; k < we * ntau; k += blockDim.x) c[k] = table_at(tab, coef, k);
    __syncthreads();
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < E_tot;
         i += (long long)gridDim.x * blockDim.x) {
        for (int w0 = wb; w0 < we; w0 += 8) {
            double acc[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) acc[w] = 0.0;
            for (int t = 0; t < ntau; ++t) {
                const double v = static_cast<double>(chi0s[(long long)t * E_tot + i]);
#pragma unroll
                for (int w = 0; w < 8; ++w)
                    if (w0 + w < we) acc[w] += c[(w0 + w) * ntau + t] * v;
            }
#pragma unroll
            for (int w = 0; w < 8; ++w)
                if (w0 + w < we) chiw[(long long)(w0 + w) * E_tot + i] = acc[w];
        }
    }
}

template <class TS>
static void tau_to_omega(const TS *chi0s, long long E_tot, int ntau, const std::vector<double> &coef, DevBuf &buf, int nw,
                         double *chiw, hipStream_t s) {
    if (ntau > kTauOmegaMax || nw > kTauOmegaMax) LRA_THROW("tau -> omega: grid too large");
    const int bx = (int)std::min<long long>(ceil_div(E_tot, 256), 8192);
    const int wper = bx >= 1024 ? nw : 8;
    with_table(coef, buf, s, [&](auto table, const double *p) {
        hipLaunchKernelGGL((tau_to_omega_kernel<TS, decltype(table)>), dim3(bx, ceil_div(nw, wper)), dim3(256), 0, s, chi0s,
                           E_tot, ntau, table, p, nw, wper, chiw);
        HIP_CHECK(hipGetLastError());
    });
}
void launch_tau_to_omega(const double *chi0s, long long E_tot, int ntau, const std::vector<double> &coef, DevBuf &buf, int nw,
                         double *chiw, hipStream_t s) {
    tau_to_omega(chi0s, E_tot, ntau, coef, buf, nw, chiw, s);
}
void launch_tau_to_omega(const float *chi0s, long long E_tot, int ntau, const std::vector<double> &coef, DevBuf &buf, int nw,
                         double *chiw, hipStream_t s) {
    tau_to_omega(chi0s, E_tot, ntau, coef, buf, nw, chiw, s);
}

// chiw[w][i] (+)= coef[w][t] slice[i] for one tau slice t (the first slice overwrites): the same
// sums as tau_to_omega_kernel, accumulated slice by slice in the same order of t
template <class TS>
__global__ __launch_bounds__(256) void tau_accumulate_kernel(const TS *__restrict__ slice, long long E_tot, int t,
                                                             int ntau, const double *__restrict__ coef, int nw,
                                                             double *__restrict__ chiw) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < E_tot;
         i += (long long)gridDim.x * blockDim.x) {
        const double v = static_cast<double>(slice[i]);
        for (int w = 0; w < nw; ++w) {
            double *d = chiw + (long long)w * E_tot + i;
            const double base = t == 0 ? 0.0 : *d;
            *d = base + coef[w * ntau + t] * v;
        }
    }
}

template <class TS>
void launch_tau_accumulate(const TS *slice, long long E_tot, int t, int ntau, const double *coef, int nw, double *chiw,
                           hipStream_t s) {
    const int bx = (int)std::min<long long>(ceil_div(E_tot, 256), 16384);
    hipLaunchKernelGGL(tau_accumulate_kernel<TS>, dim3(bx), dim3(256), 0, s, slice, E_tot, t, ntau, coef, nw, chiw);
    HIP_CHECK(hipGetLastError());
}
template void launch_tau_accumulate<double>(const double *, long long, int, int, const double *, int, double *,
                                            hipStream_t);
template void launch_tau_accumulate<float>(const float *, long long, int, int, const double *, int, double *,
                                           hipStream_t);

// dense chi0(q, omega) of nw frequencies from chi0(R, omega) for up to NQ q points at once: per pair
// element, sum_r (cos_r + i sin_r) chiw[w][eoff[p][r] + e] with the phases ph[q][r] as (cos, sin); each
// chiw value read feeds every q of the launch.  A thread does wper frequencies, one when the elements
// alone are under 1024 workgroups: with all 16 in the loop the 2-atom cell (120 functions, 43
// workgroups) took 168 us where its bytes take 15; with one each the 64-atom cell takes 6.2 ms, not 4.7.
// q point qi writes its nw matrices at dense + qi * qstride.
template <class TD, int NQ, int WU, class TAB>
__global__ __launch_bounds__(256) void chi0_rq_kernel(const double *__restrict__ chiw, long long E_tot,
                                                      const PairDesc *__restrict__ pairs, int npairs, long long nelem,
                                                      const long long *__restrict__ eoff, int nR,
                                                      const TAB tab, const double *__restrict__ ph, int nq, int nw, int wper,
                                                      TD *__restrict__ dense, long long dstride, long long qstride,
                                                      int n, int lay) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nelem) return;
    int lo = 0, hi = npairs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pairs[mid].e0 <= idx) lo = mid; else hi = mid - 1;
    }
    const PairDesc P = pairs[lo];
    const long long e = idx - P.e0;
    const int mu = (int)(e / P.naJ), nu = (int)(e % P.naJ);
    const int we = min(nw, (int)(blockIdx.y + 1) * wper);
    for (int w0 = blockIdx.y * wper; w0 < we; w0 += WU) {
        double re[WU][NQ], im[WU][NQ];
#pragma unroll
        for (int u = 0; u < WU; ++u)
#pragma unroll
            for (int q = 0; q < NQ; ++q) re[u][q] = im[u][q] = 0.0;
        const double *cw = chiw + (long long)w0 * E_tot + e;
        for (int r = 0; r < nR; ++r) {
            const long long off = eoff[(long long)lo * nR + r];
            if (off < 0) continue;
            double v[WU];
#pragma unroll
            for (int u = 0; u < WU; ++u) v[u] = cw[off + (w0 + u < we ? u * E_tot : 0)];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (q < nq) {
                    const double c = table_at(tab, ph, 2 * (q * nR + r)), d = table_at(tab, ph, 2 * (q * nR + r) + 1);
#pragma unroll
                    for (int u = 0; u < WU; ++u) {
                        re[u][q] += c * v[u];
                        im[u][q] += d * v[u];
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < WU; ++u)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (q >= nq || w0 + u >= we) break;
                put_dense(dense + q * qstride + (w0 + u) * dstride, n, P.rowI + mu, P.colJ + nu, re[u][q], im[u][q],
                          P.I != P.J, lay);
            }
    }
}

template <class TD>
void launch_chi0_rq_multi(const double *chiw, long long E_tot, const PairDesc *pairs, int npairs,
                          long long n_pair_elems, const long long *eoff, int nR, const std::vector<double> &ph,
                          DevBuf &buf, int nq, int nw, TD *dense, long long dense_stride, long long q_stride, int n,
                          DenseLayout lay, hipStream_t s) {
    if (nq < 1 || nq > kChi0RqMaxQ) LRA_THROW("chi0_rq_multi: 1 to kChi0RqMaxQ q points per launch");
    const int bx = ceil_div(n_pair_elems, 256), wper = bx >= 1024 ? nw : 1;
    with_table(ph, buf, s, [&](auto table, const double *p) {
        using TAB = decltype(table);
        const auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(bx, ceil_div(nw, wper)), dim3(256), 0, s, chiw, E_tot, pairs, npairs,
                               n_pair_elems, eoff, nR, table, p, nq, nw, wper, dense, dense_stride, q_stride, n, (int)lay);
        };
        // one q: four frequencies at a time, whose loads are in flight together (128 atoms: 20.6 -> 19.0 ms)
        if (nq > 1) go(chi0_rq_kernel<TD, kChi0RqMaxQ, 1, TAB>);
        else if (wper > 1) go(chi0_rq_kernel<TD, 1, 4, TAB>);
        else go(chi0_rq_kernel<TD, 1, 1, TAB>);
        HIP_CHECK(hipGetLastError());
    });
}
template void launch_chi0_rq_multi<double>(const double *, long long, const PairDesc *, int, long long,
                                           const long long *, int, const std::vector<double> &, DevBuf &, int, int,
                                           double *, long long, long long, int, DenseLayout, hipStream_t);
template void launch_chi0_rq_multi<float>(const double *, long long, const PairDesc *, int, long long,
                                           const long long *, int, const std::vector<double> &, DevBuf &, int, int,
                                           float *, long long, long long, int, DenseLayout, hipStream_t);

// ------------------------------------------------------------------------------------
// dense helpers
// ------------------------------------------------------------------------------------
// (Re, Im) planes <-> the real embedding [[Re, -Im], [Im, Re]]
__global__ void planes_to_embedded_kernel(const double *__restrict__ M, double *__restrict__ E, int n) {
    const long long nn = (long long)n * n, idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nn) return;
    const long long i = idx / n, j = idx % n, ld = 2 * n;
    const double re = M[idx], im = M[nn + idx];
    E[i * ld + j] = E[(n + i) * ld + n + j] = re;
    E[(n + i) * ld + j] = im;
    E[i * ld + n + j] = -im;
}
void launch_planes_to_embedded(const double *M, double *E, int n, hipStream_t s) {
    hipLaunchKernelGGL(planes_to_embedded_kernel, dim3(ceil_div((long long)n * n, 256)), dim3(256), 0, s, M, E, n);
    HIP_CHECK(hipGetLastError());
}
__global__ void embedded_to_planes_kernel(const double *__restrict__ E, double *__restrict__ M, int n) {
    const long long nn = (long long)n * n, idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nn) return;
    const long long i = idx / n, j = idx % n, ld = 2 * n;
    M[idx] = E[i * ld + j];
    M[nn + idx] = E[(n + i) * ld + j];
}
void launch_embedded_to_planes(const double *E, double *M, int n, hipStream_t s) {
    hipLaunchKernelGGL(embedded_to_planes_kernel, dim3(ceil_div((long long)n * n, 256)), dim3(256), 0, s, E, M, n);
    HIP_CHECK(hipGetLastError());
}

// zero above the diagonal; the diagonal too on odd planes (blockIdx.y counts matrices, .z planes im apart)
__global__ void zero_upper_kernel(double *A, int n, int lda, long long stride, long long im) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n * n) return;
    const int i = (int)(idx / n), j = (int)(idx % n);
    if (j > i || (j == i && blockIdx.z)) A[blockIdx.y * stride + blockIdx.z * im + (long long)i * lda + j] = 0.0;
}

template <class TS, class TD>
__global__ void convert_kernel(const TS *__restrict__ src, TD *__restrict__ dst, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        dst[i] = static_cast<TD>(src[i]);
}
template <class TS, class TD> void launch_convert(const TS *src, TD *dst, long long n, hipStream_t s) {
    const int bx = std::min(ceil_div(n, 256), 65536);
    hipLaunchKernelGGL((convert_kernel<TS, TD>), dim3(bx), dim3(256), 0, s, src, dst, n);
    HIP_CHECK(hipGetLastError());
}
template void launch_convert<double, float>(const double *, float *, long long, hipStream_t);

__global__ void copy_lower_f2d_kernel(const float *__restrict__ src, double *__restrict__ dst, int n, long long stride) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n * n) return;
    const int i = (int)(idx / n), j = (int)(idx % n);
    const long long o = blockIdx.y * stride + idx;
    if (j <= i) dst[o] = static_cast<double>(src[o]);
}
void launch_copy_lower_f2d(const float *src, double *dst, int n, long long nmat, long long stride, hipStream_t s) {
    for (long long m0 = 0; m0 < nmat; m0 += 32768) {
        hipLaunchKernelGGL(copy_lower_f2d_kernel, dim3(ceil_div((long long)n * n, 256), (unsigned)std::min(32768LL, nmat - m0)),
                           dim3(256), 0, s, src + m0 * stride, dst + m0 * stride, n, stride);
        HIP_CHECK(hipGetLastError());
    }
}

__global__ __launch_bounds__(256) void v_scatter_kernel(const double2 *__restrict__ blk, const VBlock *__restrict__ desc,
                                                        double *V, long long n, int lay, int drop_imag, int q0,
                                                        long long stride) {
    const VBlock b = desc[blockIdx.x];
    V += (b.q - q0) * stride;
    const int tot = b.na * b.nb;
    for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < tot; e += gridDim.y * blockDim.x) {
        const int mu = e / b.nb, nu = e % b.nb;
        double2 v = blk[b.off + e];
        if (drop_imag) v.y = 0.0;
        put_dense(V, n, b.r0 + mu, b.c0 + nu, v.x, v.y, !b.diag, lay);
    }
}

void launch_v_scatter(const double *blk, const VBlock *d, int nblk, double *V, int n, DenseLayout lay, int drop_imag,
                      int q0, long long stride, hipStream_t s) {
    if (nblk == 0) return;
    // a molecule has a handful of blocks of up to 10^4 elements: several workgroups each
    const int split = nblk >= 2048 ? 1 : nblk >= 256 ? 4 : 16;
    hipLaunchKernelGGL(v_scatter_kernel, dim3(nblk, split), dim3(256), 0, s, reinterpret_cast<const double2 *>(blk), d, V,
                       (long long)n, (int)lay, drop_imag, q0, stride);
    HIP_CHECK(hipGetLastError());
}

__global__ __launch_bounds__(256) void add_signs_trace_kernel(double *A, int n, long long stride,
                                                              const double *__restrict__ signs, int per, double *acc) {
    __shared__ double red[256];
    const long long u = blockIdx.x;
    double *M = A + u * stride;
    const double *S = signs + (u / per) * n;
    double v = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double m = M[(long long)i * n + i] + S[i];
        M[(long long)i * n + i] = m;
        v += S[i] * m;
    }
    red[threadIdx.x] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) acc[2 * u] += red[0];
}
void launch_add_signs_trace(double *A, int n, long long nmat, long long stride, const double *signs, int per, double *acc,
                            hipStream_t s) {
    if (nmat <= 0) return;
    hipLaunchKernelGGL(add_signs_trace_kernel, dim3((unsigned)nmat), dim3(256), 0, s, A, n, stride, signs, per, acc);
    HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// Blocked Cholesky with log-determinant
// ------------------------------------------------------------------------------------
// A double of another lane (lane is wave-uniform).
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(u & 0xffffffffu), lane));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), lane));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

typedef double v4d __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4d mfma16(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int chol_nb(bool cplx) { return cplx ? 32 : 64; }  // columns of a diagonal block
// per matrix: Linv, then Linv with row c times the pivot sign of c, each in planes
constexpr long long chol_work(bool cplx) { return 2LL * (cplx ? 2 : 1) * chol_nb(cplx) * chol_nb(cplx); }

// Factor the nb x nb diagonal block at (j0, j0) of matrix blockIdx.x as L S L^H with S = diag(+-1) (a
// Cholesky factorisation that tolerates negative pivots), write L11 back, write L11^{-1} and
// S L11^{-1} (row-major) and the pivot signs, and accumulate sum log|d_j| = ln |det| of the block.  A
// zero or NaN pivot sets *flag.
//
// One workgroup per matrix, the block in LDS, 64 real or 32 complex columns in panels of 16.  A panel
// is factored by one wave: lane t holds its 16 entries of row t (complex: lanes t and t + 32 the real
// and imaginary parts), takes the pivot and the other rows' entries by readlane.  The four waves then
// update the rest with MFMA.  The inverse goes from the 16 x 16 diagonal blocks, a wave each, outwards:
// X_ij = -X_ii sum_k L_ik X_kj with the sum's accumulators as the next MFMA's operand.  (With all 64
// columns in one wave's registers, every pivot step updates 64 columns lane by lane: 62 us a block.)
template <bool CPLX>
__global__ __launch_bounds__(256) void potrf_block_kernel(double *A0, long long strideA, long long im, int lda, int j0,
                                                          int nb, double *work, double *logdet0, long long ld_stride,
                                                          int *flag, double *signs, long long sstride) {
    constexpr int NB = chol_nb(CPLX), PL = CPLX ? 2 : 1, PN = NB / 16, NX = PN * (PN + 1) / 2;
    __shared__ double L[PL][NB][NB + 1];
    __shared__ double X[PL][NX][16][17];
    __shared__ double sg[NB], dinv[NB];  // pivot signs, 1 / L_jj
    double *A = A0 + strideA * blockIdx.x;
    double *Linv = work + chol_work(CPLX) * blockIdx.x, *SLinv = Linv + (long long)PL * NB * NB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, kq = lane >> 4;
    for (int e = tid; e < PL * NB * NB; e += 256) {
        const int h = e / (NB * NB), r = (e / NB) % NB, q = e % NB;
        L[h][r][q] = (r < nb && q <= r) ? A[h * im + (long long)(j0 + r) * lda + j0 + q] : (r == q && h == 0 ? 1.0 : 0.0);
    }
    __syncthreads();
    const int t = lane % NB, half = lane / NB;  // row and plane of a panel lane
    double my_r = 1.0;
    bool bad = false;
    for (int p = 0; p < PN; ++p) {
        if (wave == 0) {
            double a[16], own = 1.0;
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = L[half][t][16 * p + k];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int jj = 16 * p + j;
                double d = readlane_f64(a[j], jj);
                if (!(fabs(d) > 0.0)) { bad = true; d = 1.0; }
                const double s = d > 0 ? 1.0 : -1.0, q = fabs(d);
                // 1 / sqrt(q) from the hardware's approximation by one step of third order: short, where
                // sqrt and a division are a chain of 300 cycles in each of the columns.  sqrt(q) itself is only
                // written, once per panel
                double y = __builtin_amdgcn_rsq(q);
                const double e = fma(-(q * y), y, 1.0);
                y = q < INFINITY ? fma(y * e, fma(0.375, e, 0.5), y) : 0.0;
                // L_tj = a_tj / (s r), so that A = L S L^H also for a negative pivot
                const double l = t > jj ? a[j] * (s * y) : 0.0;
                if (t == jj) { own = q; if (!half) { sg[t] = s; dinv[t] = y; } }
                if (t > jj) a[j] = l;
                const double f1 = s * l;
                if constexpr (CPLX) {
                    // a_tk -= s L_tj conj(L_kj): real lanes lr lr' + li li', imaginary lanes li lr' - lr li'
                    const double lp = __shfl_xor(l, 32, 64), f2 = half ? -s * lp : s * lp;
#pragma unroll
                    for (int k = j + 1; k < 16; ++k)
                        a[k] -= f1 * readlane_f64(a[j], 16 * p + k) + f2 * readlane_f64(a[j], 32 + 16 * p + k);
                } else {
#pragma unroll
                    for (int k = j + 1; k < 16; ++k) a[k] -= f1 * readlane_f64(a[j], 16 * p + k);
                }
            }
            const double r = sqrt(own);
            if (t >= 16 * p) {
                const int dk = t - 16 * p;
                if (half == 0 && dk < 16) my_r = r;
#pragma unroll
                for (int k = 0; k < 16; ++k) L[half][t][16 * p + k] = k == dk ? (half ? 0.0 : r) : a[k];
            }
        }
        __syncthreads();
        // tiles right of the panel: L_ij -= L_ip S L_jp^H
        int n = 0;
        for (int i = p + 1; i < PN; ++i)
            for (int j = p + 1; j <= i; ++j)
                for (int h = 0; h < PL; ++h, ++n) {
                    if ((n & 3) != wave) continue;
                    v4d acc;
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[r] = L[h][16 * i + 4 * r + kq][16 * j + c];
#pragma unroll
                    for (int st = 0; st < 4; ++st) {
                        const int k = 16 * p + 4 * st + kq;
                        const double s = sg[k];
                        if constexpr (!CPLX) {
                            acc = mfma16(-s * L[0][16 * i + c][k], L[0][16 * j + c][k], acc);
                        } else {
                            const double ar = L[0][16 * i + c][k], ai = L[PL - 1][16 * i + c][k];
                            acc = mfma16(-s * (h ? ai : ar), L[0][16 * j + c][k], acc);
                            acc = mfma16(h ? s * ar : -s * ai, L[PL - 1][16 * j + c][k], acc);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) L[h][16 * i + 4 * r + kq][16 * j + c] = acc[r];
                }
        __syncthreads();
    }
    for (int e = tid; e < PL * NB * NB; e += 256) {
        const int h = e / (NB * NB), r = (e / NB) % NB, q = e % NB;
        if (r < nb && q <= r) A[h * im + (long long)(j0 + r) * lda + j0 + q] = L[h][r][q];
    }
    // inverses of the diagonal blocks: lane c (complex: c and c + 16) holds column c
    if (wave < PN) {
        const int hx = CPLX ? kq & 1 : 0, b = 16 * wave;
        double x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = (r == c && hx == 0) ? 1.0 : 0.0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] *= dinv[b + r];
            double xp = 0;
            if constexpr (CPLX) {
                xp = __shfl_xor(x[r], 16, 64);
                if (!hx) xp = -xp;
            }
#pragma unroll
            for (int q = r + 1; q < 16; ++q) {
                x[q] -= L[0][b + q][b + r] * x[r];
                if constexpr (CPLX) x[q] -= L[PL - 1][b + q][b + r] * xp;
            }
        }
        if (kq < PL)
#pragma unroll
            for (int r = 0; r < 16; ++r) X[kq][wave * (wave + 3) / 2][r][c] = x[r];
    }
    __syncthreads();
    for (int dist = 1; dist < PN; ++dist) {
        const int i = dist + wave, j = wave;
        if (i < PN) {
            v4d tr = {0, 0, 0, 0}, ti = {0, 0, 0, 0};
            for (int k = j; k < i; ++k) {
                const int xb = k * (k + 1) / 2 + j;
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    const int q = 4 * st + kq;
                    const double lr = L[0][16 * i + c][16 * k + q], xr = X[0][xb][q][c];
                    tr = mfma16(lr, xr, tr);
                    if constexpr (CPLX) {
                        const double li = L[PL - 1][16 * i + c][16 * k + q], xi = X[PL - 1][xb][q][c];
                        tr = mfma16(-li, xi, tr);
                        ti = mfma16(lr, xi, ti);
                        ti = mfma16(li, xr, ti);
                    }
                }
            }
            v4d yr = {0, 0, 0, 0}, yi = {0, 0, 0, 0};
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const double xr = -X[0][i * (i + 3) / 2][c][4 * st + kq];
                yr = mfma16(xr, tr[st], yr);
                if constexpr (CPLX) {
                    const double xi = -X[PL - 1][i * (i + 3) / 2][c][4 * st + kq];
                    yr = mfma16(-xi, ti[st], yr);
                    yi = mfma16(xr, ti[st], yi);
                    yi = mfma16(xi, tr[st], yi);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                X[0][i * (i + 1) / 2 + j][4 * r + kq][c] = yr[r];
                if constexpr (CPLX) X[PL - 1][i * (i + 1) / 2 + j][4 * r + kq][c] = yi[r];
            }
        }
        __syncthreads();
    }
    for (int e = tid; e < PL * NB * NB; e += 256) {
        const int h = e / (NB * NB), r = (e / NB) % NB, q = e % NB, bi = r / 16, bj = q / 16;
        const double v = (q <= r && r < nb) ? X[h][bi * (bi + 1) / 2 + bj][r % 16][q % 16] : 0.0;
        Linv[e] = v;
        SLinv[e] = sg[r] * v;
    }
    if (signs != nullptr && tid < nb) signs[sstride * blockIdx.x + j0 + tid] = sg[tid];
    if (wave == 0) {
        double v = (half == 0 && t < nb) ? 2.0 * log(my_r) : 0.0;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) {
            logdet0[ld_stride * blockIdx.x] += v;
            if (bad) *flag = 1;
        }
    }
}

// m x nb blocks of nmat matrices (blockIdx.y) and their planes (.z)
__global__ void copy_panel_kernel(const double *__restrict__ src, int lds, long long sstride, long long splane,
                                  double *__restrict__ dst, int ldd, long long dstride, long long dplane, int m, int nb) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)m * nb) return;
    const long long r = idx / nb, q = idx % nb;
    dst[blockIdx.y * dstride + blockIdx.z * dplane + r * ldd + q] = src[blockIdx.y * sstride + blockIdx.z * splane + r * lds + q];
}

struct CholPlan {
    std::vector<int> j0s, nbs;
    std::vector<GemmBatch> trsm, inpanel;  // per step of one diagonal block
    std::vector<GemmBatch> mid;            // per step: the middle panel's update of the outer panel's other columns
    std::vector<GemmBatch> trail;          // per step: the trailing update after an outer panel
};

static std::map<std::tuple<int, int, int, long long, hipStream_t, int, long long>, CholPlan> &chol_plans() {
    static std::map<std::tuple<int, int, int, long long, hipStream_t, int, long long>, CholPlan> p;
    return p;
}

// Right-looking blocked L S L^H factorisation in three levels.  Steps of one diagonal block (64 real or 32
// complex columns, by potrf_block_kernel; Q = A21 L11^-H and Q S by one GEMM launch) update only the rest
// of their middle panel (512 real or 256 complex columns); after each middle panel one GEMM updates the
// remaining columns of its outer panel; after each outer panel one lower-triangular GEMM updates the
// trailing matrix (2048 real or 1024 complex columns for n >= 4096 / 2048, else the middle level is the
// outer one).  Few, deep trailing updates read and write the trailing matrix four times less often.  All of
// them on 64x64 tiles: 128x128 ones waste half of every diagonal tile and run FP64 at 42 TF/s, not 50 (16
// atoms and 8 k, n = 960: 7.5 -> 4.2 ms of trailing updates; n = 5760: 24.8 -> 21.0).  Q and Q S of the
// outer panel's columns are kept in wide buffers per matrix (pitch = outer panel width, indexed by global
// row).
//
// A Hermitian matrix is factored as such, from its two planes, each product as two real segments:
// 4/3 n^3 real multiply-adds, where the real embedding [[Re, -Im], [Im, Re]] (2n x 2n) needs 8/3 n^3.
void cholesky_logdet_batched(double *A, long long strideA, int nbatch, int n, int lda, double *logdet,
                             long long ld_stride, int *flag, bool keep_L, CholWork &w, hipStream_t s, int ncols,
                             double *signs, long long sstride, long long im) {
    const bool cplx = im != 0;
    const int nf = (ncols > 0 && ncols < n) ? ncols : n;
    const int NB = chol_nb(cplx), PW = 8 * NB, PO = n >= 64 * NB ? 4 * PW : PW, PL = cplx ? 2 : 1;
    const long long wstride = chol_work(cplx), wplane = (long long)NB * NB;
    const long long qplane = (long long)n * PO, qs_off = PL * qplane, pstride = 2 * qs_off;  // Q planes, then Q S planes
    w.linv.reserve(sizeof(double) * wstride * nbatch);
    w.panel.reserve(sizeof(double) * pstride * nbatch);
    auto key = std::make_tuple(n, lda, nbatch, strideA, s, nf, im);
    auto &plans = chol_plans();
    auto it = plans.find(key);
    if (it == plans.end()) {
        CholPlan cp;
        // C (+)= A B^H: one real problem, or its real and imaginary parts as two segments each
        auto add = [&](GemmBatch &b, int M, int N, int K, long long ao, long long ap, int la, long long bo, long long bp,
                       int lb, long long co, long long cpl, int lc) {
            GemmProb p = make_prob(M, N, K, ao, la, bo, lb, co, lc);
            if (cplx) { p.sgn2 = 1; p.a_off2 = ao + ap; p.b_off2 = bo + bp; }
            b.add(p);
            if (!cplx) return;
            p = make_prob(M, N, K, ao + ap, la, bo, lb, co + cpl, lc);
            p.sgn2 = -1;
            p.a_off2 = ao;
            p.b_off2 = bo + bp;
            b.add(p);
        };
        for (int o0 = 0; o0 < nf; o0 += PO) {
            const int oend = std::min(o0 + PO, nf);
            for (int p0 = o0; p0 < oend; p0 += PW) {
                const int pend = std::min(p0 + PW, oend);
                for (int j0 = p0; j0 < pend; j0 += NB) {
                    const int nb = std::min(NB, pend - j0);
                    const int m = n - j0 - nb;
                    const int wcols = pend - j0 - nb;  // middle panel columns right of this step
                    cp.j0s.push_back(j0);
                    cp.nbs.push_back(nb);
                    GemmBatch tr, ip, md, tl;
                    if (m > 0) {
                        tr.trans_b = true;
                        ip.trans_b = true;
                        for (int b = 0; b < nbatch; ++b) {
                            const long long wq = pstride * b + (long long)(j0 + nb) * PO + (j0 - o0);
                            const long long a21 = strideA * b + (long long)(j0 + nb) * lda + j0;
                            // Q = A21 Linv^H and Q S (A21: m x nb at (j0+nb, j0)) into the wide buffers
                            add(tr, m, nb, nb, a21, im, lda, wstride * b, wplane, NB, wq, qplane, PO);
                            add(tr, m, nb, nb, a21, im, lda, wstride * b + PL * wplane, wplane, NB, wq + qs_off, qplane, PO);
                            // A[j0+nb:, j0+nb:pend] -= (Q S) Q[0:wcols]^H
                            if (wcols > 0)
                                add(ip, m, wcols, nb, wq + qs_off, qplane, PO, wq, qplane, PO,
                                    strideA * b + (long long)(j0 + nb) * lda + (j0 + nb), im, lda);
                        }
                        tr.finalize(T64x64, s);
                        if (wcols > 0) ip.finalize(T64x64, s);
                    }
                    if (j0 + nb == pend && pend < oend) {
                        // the middle panel's update of the outer panel: A[pend:, pend:oend] -= (Q S) Q^H
                        // over its pend - p0 columns (rectangular; the upper part of the diagonal
                        // block is not read)
                        md.trans_b = true;
                        for (int b = 0; b < nbatch; ++b) {
                            const long long wq = pstride * b + (long long)pend * PO + (p0 - o0);
                            add(md, n - pend, oend - pend, pend - p0, wq + qs_off, qplane, PO, wq, qplane, PO,
                                strideA * b + (long long)pend * lda + pend, im, lda);
                        }
                        md.finalize(T64x64, s);
                    }
                    const int mt = n - oend;
                    if (j0 + nb == oend && mt > 0) {
                        // trailing update of the outer panel: A22 -= (Q S) Q^H over its oend - o0 columns
                        tl.trans_b = true;
                        tl.lower_only = true;
                        for (int b = 0; b < nbatch; ++b) {
                            const long long wq = pstride * b + (long long)oend * PO;
                            add(tl, mt, mt, oend - o0, wq + qs_off, qplane, PO, wq, qplane, PO,
                                strideA * b + (long long)oend * lda + oend, im, lda);
                        }
                        tl.finalize(T64x64, s);
                    }
                    cp.trsm.push_back(std::move(tr));
                    cp.inpanel.push_back(std::move(ip));
                    cp.mid.push_back(std::move(md));
                    cp.trail.push_back(std::move(tl));
                }
            }
        }
        it = plans.emplace(key, std::move(cp)).first;
    }
    CholPlan &cp = it->second;
    double *work = w.linv.as<double>();
    double *panel = w.panel.as<double>();
    for (size_t b = 0; b < cp.j0s.size(); ++b) {
        const int j0 = cp.j0s[b], nb = cp.nbs[b];
        const int o0 = (j0 / PO) * PO;
        if (cplx)
            hipLaunchKernelGGL(potrf_block_kernel<true>, dim3(nbatch), dim3(256), 0, s, A, strideA, im, lda, j0, nb, work,
                               logdet, ld_stride, flag, signs, sstride);
        else
            hipLaunchKernelGGL(potrf_block_kernel<false>, dim3(nbatch), dim3(256), 0, s, A, strideA, im, lda, j0, nb, work,
                               logdet, ld_stride, flag, signs, sstride);
        HIP_CHECK(hipGetLastError());
        const int m = n - j0 - nb;
        if (m > 0) {
            gemm_run(Prec::F64, cp.trsm[b], A, work, panel, 1.0, 0.0, s);
            if (keep_L) {
                const double *qs = panel + qs_off + (long long)(j0 + nb) * PO + (j0 - o0);
                hipLaunchKernelGGL(copy_panel_kernel, dim3(ceil_div((long long)m * nb, 256), nbatch, PL), dim3(256), 0, s,
                                   qs, PO, pstride, qplane, A + (long long)(j0 + nb) * lda + j0, lda, strideA, im, m, nb);
                HIP_CHECK(hipGetLastError());
            }
            gemm_run(Prec::F64, cp.inpanel[b], panel, panel, A, -1.0, 1.0, s);
        }
        gemm_run(Prec::F64, cp.mid[b], panel, panel, A, -1.0, 1.0, s);
        gemm_run(Prec::F64, cp.trail[b], panel, panel, A, -1.0, 1.0, s);
    }
    if (keep_L) {
        hipLaunchKernelGGL(zero_upper_kernel, dim3(ceil_div((long long)n * n, 256), nbatch, PL), dim3(256), 0, s, A, n, lda,
                           strideA, im);
        HIP_CHECK(hipGetLastError());
    }
}

}  // namespace lra
