// G0W0 on one GPU: W(q, i omega) -> W(R, i tau) and the correlation self-energy.
//
// Screened interaction (compute_Wc_freq_q_blacs, src/core/epsilon.cpp:1763-2321):
//   Wc = v^{1/2} [(1 - v^{1/2} chi0 v^{1/2})^{-1} - 1] v^{1/2}  =  L M^{-1} L^H - v,
// with v = L L^H (Cholesky) and M = 1 - L^H chi0 L, exact when the truncated Coulomb
// equals the bare one.  L M^{-1} L^H - v is read off as minus the Schur complement of
// the augmented matrix [[M, L^H], [L, v]] after eliminating its first block column with
// the signed blocked Cholesky; with k points all matrices are held as real and imaginary planes.
// All frequencies of as many q as memory allows go through every step together.
// W(R, tau) = Re sum_w gamma_f2t(tau, w) (1/N_k) sum_q e^{-i 2 pi q.R} Wc(q, w)
// (CT_FT_Wc_freq_q, epsilon.cpp:2490-2666) is accumulated on the device.  With an IBZ
// mapping only the irreducible q are formed; the others must be their time-reversal partners
// (FT_Wc_freq_q, epsilon.cpp:2430-2452, takes W(-q) = conj W(q)), whose real parts of
// e^{-i 2 pi q.R} W(q) are equal, so each irreducible q is weighted by its star size.
// A Coulomb matrix with a negative pivot, a positive sqrt_coulomb_threshold or a head
// replacement at q = 0 takes the square roots from an eigen-decomposition instead
// (power_hemat, src/math/matrix_m.h:916-970, eigenvalues below the threshold dropped); then
// W = S_c eps^{-1} S_c - S_c S_c, the Schur complement of [[eps, S_c], [S_c, S_c S_c]].
//
// Self-energy (RI::GW::cal_Sigmas, thirdparty/LibRI/include/RI/physics/GW.hpp:102-122,
// called from G0W0::build_spacetime, src/core/gw.cpp:217-875), per tau and spin, both signs at once:
//   U_J(S)[(X,x)][j][nu] = sum_{(L,Rb) in N(J)} G_XL(S+Rb) C^J(L,Rb)           (GEMM per (J,S,sign))
//   CW_IJ(R)[c][i][nu] = sum_mu C^I[(c,i)][mu] W_IJ(R)(mu,nu), c = (n,k) in N(I)  (GEMM per (I,J,R))
//   label a0b0_a2b2: Sigma_IJ(R)(i,j) = sum_(c,nu) CW_IJ(R)[c][i][nu] U_J(R-Ra_c)[c][j][nu]
//   label a0b0_a1b2: Sigma_KJ(R-Ra)(k,j) += sum_(i,nu) CW_IJ(R)[c][i][nu] U_J(R)[(I,i)][j][nu]
//   label a0b0_a1b1: Y_I[(S,L,l)][i][mu] = sum_{J,R,j} G_IJ(R)(i,j) CW_JI(-R)[(L,S-R,l)][j][mu]
//                    Sigma_KL(S-Ra)(k,l) += sum_(i,mu) C^I[c][i][mu] Y_I[(S,L,l)][i][mu]
//   label a0b0_a2b1: the transpose of a0b0_a1b2, Sigma_XY(R) += [a1b2]_YX(-R)^T.
// CW holds neither sign nor spin and serves three labels (the third by W_IJ(R) = W_JI(-R)^T), where W
// against U and against G C^J would be two products of its size per sign: 1 + 2 * 5/4.6 of its flops
// a tau point, not 2 + 2 * 2 (n_aux = 4.6 n_ao).  It takes the room that T = W U would.
// Y's outputs are indexed by a cell difference: they go through an extended (2p-1)^3 cell grid with
// atomic accumulation and are folded back to the BvK cell afterwards.  Sigma(R, i w) =
// sum_tau 0.5 (S+ + S-) gamma_c + i 0.5 (S+ - S-) gamma_s (gw.cpp:681-797).
#include "gw.h"

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>

#include "dielec.h"
#include "gw_kernels.h"

namespace lra {

namespace {
double now_s() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
}  // namespace

// ------------------------------------------------------------------------------------------
// plan
// ------------------------------------------------------------------------------------------
void GwEngine::plan(const Dataset &ds, std::shared_ptr<RpaEngine> r) {
    rpa = std::move(r);
    const RpaEngine &R0 = *rpa;
    prec = R0.prec;
    ts = R0.ts;
    natom = R0.natom;
    NAO = R0.NAO;
    NABF = R0.NABF;
    nR = R0.nR;
    nk = R0.nk;
    nspin = R0.nspin;
    ntau = R0.planned_ntau;
    LD = (long long)nR * NAO;
    const auto &nb = R0.nb;
    const auto &na = R0.na;
    const auto &ao = R0.ao;
    const auto &abf = R0.abf;
    const auto &cells = R0.cells;
    const hipStream_t st = R0.stream;
    // ---- extended cell grid ----
    const int *p = R0.period;
    for (int a = 0; a < 3; ++a) E[a] = 2 * p[a] - 1;
    NE = E[0] * E[1] * E[2];
    c0 = linr(p[0] - 1, p[1] - 1, p[2] - 1);
    std::vector<int> fold(NE), neg(nR);
    for (int x = 0; x < E[0]; ++x)
        for (int y = 0; y < E[1]; ++y)
            for (int z = 0; z < E[2]; ++z)
                fold[(x * E[1] + y) * E[2] + z] = R0.fold_index(x - (p[0] - 1), y - (p[1] - 1), z - (p[2] - 1));
    for (int rr = 0; rr < nR; ++rr) neg[rr] = R0.fold_index(-cells[rr][0], -cells[rr][1], -cells[rr][2]);
    d_fold = upload(fold, st);
    d_neg = upload(neg, st);
    std::vector<long long> ext_cols(LD);
    for (int rr = 0; rr < nR; ++rr)
        for (int c = 0; c < NAO; ++c)
            ext_cols[(size_t)rr * NAO + c] =
                (linr(cells[rr][0], cells[rr][1], cells[rr][2]) + c0) * NAO * (long long)NAO + c;

    reclaim_if_low();
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));

    // ---- U_J(S) for all J, S and signs (resident) and the gathered G panels by chunks of J ----
    u_off.assign((size_t)natom * nR + 1, 0);
    for (int J = 0; J < natom; ++J)
        for (int S = 0; S < nR; ++S)
            u_off[(size_t)J * nR + S + 1] = u_off[(size_t)J * nR + S] + (long long)NAO * nb[J] * na[J];
    u_elems = u_off[(size_t)natom * nR];
    y_off.assign(natom + 1, 0);
    for (int I = 0; I < natom; ++I) y_off[I + 1] = y_off[I] + (long long)na[I] * nb[I] * LD;
    y_elems = y_off[natom];
    const double ghat_budget = std::min(24e9, 0.08 * (double)free_b), wrt = 8.0 * ntau * nR * (double)NABF * NABF;
    double cw_least = 0;  // CW of one atom
    for (int x = 0; x < natom; ++x) cw_least = std::max(cw_least, (double)ts * nR * R0.lsum[x] * nb[x] * NABF);
    signs = 2.0 * ts * (u_elems + y_elems) + ghat_budget + wrt + std::max(4e9, cw_least) > 0.85 * (double)free_b ? 1 : 2;
    if (const char *e = std::getenv("LIBRPA_AMD_SIGMA_SIGNS")) signs = std::atoi(e) == 1 ? 1 : signs;
    const long long gpm_r = (long long)NAO * 2 * NAO;
    max_ghat = 0;
    for (int only = signs == 2 ? -1 : 0; only < (signs == 2 ? 0 : 2); ++only) {
        int j = 0;
        while (j < natom) {
            UChunk c;
            c.sg = only;
            const int j0 = j;
            for (; j < natom; ++j) {
                const long long g1 = (long long)nR * signs * NAO * R0.lsum[j];
                if (j > j0 && (double)(c.ghat_elems + g1) * ts > ghat_budget) break;
                const long long ls = R0.lsum[j];
                for (int S = 0; S < nR; ++S)
                    for (int sg = 0; sg < 2; ++sg) {
                        if (only >= 0 && sg != only) continue;
                        GatherJob gj;
                        gj.dst_off = c.ghat_elems;
                        gj.ncol = (int)ls;
                        gj.col_off = (int)c.colsrc.size();
                        for (const auto &n : R0.nbrs[j]) {
                            const auto &R2 = cells[n.r];
                            const auto &Sv = cells[S];
                            const int rr = R0.fold_index(Sv[0] + R2[0], Sv[1] + R2[1], Sv[2] + R2[2]);
                            for (int l = 0; l < nb[n.K]; ++l)
                                c.colsrc.push_back(rr * gpm_r + 2 * ao[n.K] + (long long)sg * nb[n.K] + l);
                        }
                        c.max_gcol = std::max(c.max_gcol, gj.ncol);
                        c.jobs.push_back(gj);
                        // K = 0 (an atom without Cs) writes zeros
                        c.ub.add(make_prob(NAO, nb[j] * na[j], (int)ls, c.ghat_elems, (int)ls, R0.cwb_off[j],
                                           nb[j] * na[j], (only < 0 ? sg * u_elems : 0) + u_off[(size_t)j * nR + S], nb[j] * na[j]));
                        c.ghat_elems += (long long)NAO * ls;
                    }
            }
            c.d_jobs = upload(c.jobs, st);
            c.d_colsrc = upload(c.colsrc, st);
            // default tiles: the autotuner's choices on the 64-atom, 8-k cell (FP64)
            c.ub.finalize(prec == Prec::F64 ? T128x64w8 : big_tile(prec), st);
            flops_sigma += c.ub.flops;
            max_ghat = std::max(max_ghat, c.ghat_elems);
            uchunks.push_back(std::move(c));
        }
    }

    // ---- the contraction of Y ----
    a3 = GemmBatch();
    a3.atomic = true;
    a3.trans_b = true;
    a3.coltab = ext_cols;
    for (int I = 0; I < natom; ++I) {
        if (R0.lsum[I] == 0) continue;
        GemmProb q = make_prob((int)R0.lsum[I], (int)LD, na[I] * nb[I], 0, 0, y_off[I], na[I] * nb[I], 0, 0);
        q.rt_off = (int)(a3.rowtab.size() / 2);
        q.ct_off = 0;
        for (size_t n = 0; n < R0.nbrs[I].size(); ++n) {
            const int K = R0.nbrs[I][n].K;
            const auto &Ra = cells[R0.nbrs[I][n].r];
            const long long lr = linr(Ra[0], Ra[1], Ra[2]);
            for (int k = 0; k < nb[K]; ++k) {
                a3.rowtab.push_back(R0.cfin_off[I] + (R0.loff[I][n] + k) * nb[I] * na[I]);
                a3.rowtab.push_back((ao[K] + k) * NAO - lr * NAO * (long long)NAO);
            }
        }
        a3.add(q);
    }
    a3.finalize(big_tile(prec), st);
    flops_sigma += 2 * a3.flops;

    // ---- CW by chunks of atoms, and the passes over it ----
    const double per_sign = (double)ts * (u_elems + max_ghat + y_elems + (2.0 * nR + NE) * NAO * (double)NAO);
    double cw_total = 0, fl = 0;
    std::vector<long long> cw_x(natom);  // CW of atom x in its chunk: [R][J][c][i][nu]
    {
        double budget = std::max(4e9, std::min(96e9, 0.6 * (double)free_b - signs * per_sign - wrt));
        if (const char *cb = std::getenv("LIBRPA_AMD_CHUNK_BYTES"))
            if (std::atof(cb) > 0) budget = std::min(budget, std::atof(cb));
        int x = 0;
        while (x < natom) {
            XChunk c;
            c.x0 = x;
            for (; x < natom; ++x) {
                const long long t = (long long)nR * R0.lsum[x] * nb[x] * NABF;
                if (x > c.x0 && (double)(c.cw_elems + t) * ts > budget) break;
                cw_x[x] = c.cw_elems;
                c.cw_elems += t;
            }
            c.x1 = x;
            cw_total += (double)c.cw_elems;
            max_cw = std::max(max_cw, c.cw_elems);
            xchunks.push_back(std::move(c));
        }
    }
    std::vector<long long> seg_i(natom + 1, 0);  // segment table: atom, cell
    for (int I = 0; I < natom; ++I) seg_i[I + 1] = seg_i[I] + nR * R0.lsum[I];
    auto pack = [&](std::map<std::pair<int, int>, std::vector<SigTask>> &m, std::vector<Tasks> &out) {
        for (auto &kv : m) {
            Tasks t;
            t.a = kv.first.first;
            t.b = kv.first.second;
            t.n = (int)kv.second.size();
            t.d = upload(kv.second, st);
            HIP_CHECK(hipStreamSynchronize(st));
            out.push_back(std::move(t));
        }
    };
    for (auto &c : xchunks) {
        std::vector<SigBlk> blks;
        for (int I = c.x0; I < c.x1; ++I) {
            const long long lb = R0.lsum[I] * nb[I];
            if (lb == 0) continue;
            for (int rr = 0; rr < nR; ++rr)
                for (int J = 0; J < natom; ++J) {
                    const long long at = cw_x[I] + (rr * (long long)NABF + abf[J]) * lb;
                    c.cwb.add(make_prob((int)lb, na[J], na[I], R0.cfin_off[I], na[I],
                                        (long long)rr * NABF * NABF + abf[I] * NABF + abf[J], NABF, at, na[J]));
                    blks.push_back({at, u_off[(size_t)J * nR], nb[I], nb[J], na[J], (int)R0.lsum[I], (int)ao[I],
                                    (int)ao[J], rr, (int)(seg_i[I] + rr * R0.lsum[I])});
                    fl += 8.0 * R0.lsum[I] * nb[I] * na[J] * nb[J] + 4.0 * nb[I] * na[I] * nb[J] * R0.lsum[J];
                }
        }
        c.cwb.finalize(prec == Prec::F64 ? T128x64w8 : T128x64, st);
        c.d_blks = upload(blks, st);
        fl += c.cwb.flops / nspin;
        HIP_CHECK(hipStreamSynchronize(st));
    }
    flops_sigma = (flops_sigma + fl) * nspin * ntau;
    // tau points per pass, as in the chi0 build: up to about 120 GFLOP, and 12 GB
    nbatch = 1;
    if (signs == 2 && uchunks.size() == 1 && xchunks.size() == 1)
        nbatch = (int)std::max(1.0, std::min({(double)R0.nbatch, std::ceil(1.2e11 / std::max(1.0, flops_sigma / ntau)),
                                              std::min(12e9, 0.1 * (double)free_b) / (ts * cw_total + signs * per_sign)}));
    nbatch = ceil_div(ntau, ceil_div(ntau, nbatch));
    for (auto &c : xchunks) {
        std::map<std::pair<int, int>, std::vector<SigTask>> td, tb;
        int b = 0;
        const double nblk = (double)(c.x1 - c.x0) * natom * nR * nbatch;
        for (int I = c.x0; I < c.x1; ++I) {
            const int l = (int)R0.lsum[I];
            if (l * nb[I] == 0) continue;  // (as where the blocks that tasks count were made)
            // 2048 workgroups, each with at least 16 segments
            const int parts = std::max(1, std::min(ceil_div(l, 16), (int)std::ceil(2048.0 / nblk)));
            for (int rr = 0; rr < nR; ++rr)
                for (int J = 0; J < natom; ++J, ++b) {
                    const int fi = nb[I] > 16 ? 2 : 1, fj = nb[J] > 16 ? 2 : 1, fc = l > 64 ? 2 : 1;
                    for (int j0 = 0; j0 < nb[J]; j0 += 16 * fj) {
                        for (int i0 = 0; i0 < nb[I]; i0 += 16 * fi)
                            for (int q = 0; q < parts; ++q)
                                td[{fi, fj}].push_back({b, i0, j0, (int)((long long)l * q / parts),
                                                        (int)((long long)l * (q + 1) / parts)});
                        for (int t0 = 0; t0 < l; t0 += 64 * fc) tb[{fc, fj}].push_back({b, 0, j0, t0, l});
                    }
                }
        }
        pack(td, c.d);
        pack(tb, c.b);
    }
    // entries (J, R) of every (S, L): J's neighbours L in the cell S - R
    {
        std::vector<SigYEnt> ents;
        std::vector<int> e0((size_t)nR * natom + 1, 0);
        std::vector<std::vector<int>> nbr_at(natom, std::vector<int>((size_t)natom * nR, -1));
        for (int J = 0; J < natom; ++J)
            for (size_t n = 0; n < R0.nbrs[J].size(); ++n)
                nbr_at[J][(size_t)R0.nbrs[J][n].K * nR + R0.nbrs[J][n].r] = (int)n;
        for (int S = 0; S < nR; ++S)
            for (int L = 0; L < natom; ++L) {
                for (int J = 0; J < natom; ++J)
                    for (int rr = 0; rr < nR && nb[J] > 0; ++rr) {
                        const int r2 = R0.fold_index(cells[S][0] - cells[rr][0], cells[S][1] - cells[rr][1],
                                                     cells[S][2] - cells[rr][2]);
                        const int n = nbr_at[J][(size_t)L * nR + r2];
                        if (n < 0) continue;
                        const long long lb = R0.lsum[J] * nb[J];
                        ents.push_back({rr * gpm_r + 2 * ao[J], cw_x[J] + neg[rr] * (long long)NABF * lb, (int)lb,
                                        (int)(R0.loff[J][n] * nb[J]), nb[J], J});
                    }
                e0[(size_t)S * natom + L + 1] = (int)ents.size();
            }
        std::map<int, std::vector<SigYTask>> ty;
        for (int S = 0; S < nR; ++S)
            for (int L = 0; L < natom; ++L)
                for (int I = 0; I < natom; ++I) {
                    const int fi = nb[I] > 16 ? 2 : 1;
                    for (int l0 = 0; l0 < nb[L]; l0 += 4)
                        for (int mu0 = 0; mu0 < na[I]; mu0 += 64)
                            for (int i0 = 0; i0 < nb[I]; i0 += 16 * fi)
                                ty[fi].push_back({y_off[I] + ((long long)S * NAO + ao[L]) * nb[I] * na[I],
                                                  e0[(size_t)S * natom + L], e0[(size_t)S * natom + L + 1], nb[I], na[I],
                                                  (int)ao[I], (int)abf[I], l0, nb[L], mu0, i0});
                }
        for (auto &kv : ty) {
            Tasks t;
            t.a = kv.first;
            t.n = (int)kv.second.size();
            t.d = upload(kv.second, st);
            HIP_CHECK(hipStreamSynchronize(st));
            ytasks.push_back(std::move(t));
        }
        d_yent = upload(ents, st);
        HIP_CHECK(hipStreamSynchronize(st));
    }
}

// ------------------------------------------------------------------------------------------
// W(q, omega) -> W(R, tau)
// ------------------------------------------------------------------------------------------
namespace {
// C = A B of nmat matrices, real or of two planes each, nn elements apart; the operands of matrix m at
// a[m], b[m] (offsets), the results compact
GemmBatch square_batch(int n, bool herm, const std::vector<long long> &a, const std::vector<long long> &b, hipStream_t st) {
    GemmBatch out;
    const long long plane = (long long)n * n, nn = plane * (herm ? 2 : 1);
    for (size_t m = 0; m < a.size(); ++m)
        for (int h = 0; h < (herm ? 2 : 1); ++h) {
            GemmProb p = make_prob(n, n, n, a[m], n, b[m] + h * plane, n, (long long)m * nn + h * plane, n);
            if (herm) {
                p.sgn2 = h ? 1 : -1;
                p.a_off2 = a[m] + plane;
                p.b_off2 = b[m] + (1 - h) * plane;
            }
            out.add(p);
        }
    // a single small matrix on few workgroups is bound by one tile's K loop: smaller tiles
    out.finalize((double)n * n * out.probs.size() < 64.0 * 64 * 512 ? T32x64 : T64x64, st);
    return out;
}

// Principal square roots of the Hermitian positive-definite matrices A + sel[m] nn (in place) by the
// coupled Newton-Schulz iteration Y <- Y T, Z <- T Z, T = (3 I - Z Y) / 2 from Y = A / c, Z = I with
// c = ||A||_F >= lambda_max; Y -> (A / c)^{1/2}.  Equals the eigen-decomposition root of
// power_hemat (src/math/matrix_m.h:916-970) for positive-definite input.  Runs to convergence, all
// matrices together; the host looks at the changes of every fourth iteration's batch only.
// work: at least 5 matrices per root, or memory is allocated.
void ns_sqrt(double *A, int n, bool herm, const std::vector<int> &sel, double *work, size_t work_elems, hipStream_t st) {
    if (sel.empty()) return;
    const int nm = (int)sel.size(), pl = herm ? 2 : 1;
    const size_t nn = (size_t)n * n * pl, all = nn * 8 * nm;
    constexpr int kMax = 200, kLook = 4;
    DevBuf own, dpart(32 * 8 * (size_t)nm), dscale(8 * (size_t)nm), dchg(sizeof(unsigned long long) * 2 * nm * kMax);
    if (work_elems < 5 * nn * nm) {
        own.alloc(5 * all);
        work = own.as<double>();
    }
    double *dY = work, *dZ = dY + nn * nm, *dP = dZ + nn * nm, *dYn = dP + nn * nm, *dZn = dYn + nn * nm;
    DevBuf dsel = upload(sel, st);
    std::vector<long long> at(nm);
    for (int m = 0; m < nm; ++m) at[m] = (long long)m * (long long)nn;
    GemmBatch b = square_batch(n, herm, at, at, st);
    HIP_CHECK(hipMemsetAsync(dchg.get(), 0, dchg.bytes(), st));
    launch_ns_init(A, dsel.as<int>(), nm, n, pl, dpart.as<double>(), dY, dZ,
                   dscale.as<double>(), st);
    std::vector<double> c(nm), h(2 * (size_t)nm * kLook), prev(nm, 1e300);
    std::vector<int> stall(nm, 0);
    std::vector<char> done(nm, 0);
    HIP_CHECK(hipMemcpyAsync(c.data(), dscale.get(), 8 * (size_t)nm, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    for (double x : c)
        if (!(x > 0) || !std::isfinite(x)) LRA_THROW("Coulomb matrix is zero or not finite");
    bool all_done = false;
    for (int k0 = 0; k0 < kMax && !all_done; k0 += kLook) {
        for (int k = k0; k < k0 + kLook; ++k) {
            gemm_run(Prec::F64, b, dZ, dY, dP, 1.0, 0.0, st);
            launch_ns_step(dP, nm, n, pl, st);
            gemm_run(Prec::F64, b, dY, dP, dYn, 1.0, 0.0, st);
            gemm_run(Prec::F64, b, dP, dZ, dZn, 1.0, 0.0, st);
            launch_ns_change(dYn, dY, nm, n, pl, dchg.as<unsigned long long>() + 2 * (size_t)nm * k, st);
            std::swap(dY, dYn);
            std::swap(dZ, dZn);
        }
        HIP_CHECK(hipMemcpyAsync(h.data(), dchg.as<unsigned long long>() + 2 * (size_t)nm * k0, 8 * h.size(),
                                 hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        all_done = true;
        for (int m = 0; m < nm; ++m) {
            for (int k = 0; k < kLook && !done[m]; ++k) {
                const double rel = h[2 * ((size_t)k * nm + m)] / std::max(h[2 * ((size_t)k * nm + m) + 1], 1e-300);
                if (!std::isfinite(rel)) LRA_THROW("square root of the Coulomb matrix did not converge (not positive definite?)");
                // quadratic phase ends at rounding level: stop once the update no longer shrinks
                if (rel < 1e-13 && (rel >= prev[m] || ++stall[m] >= 3)) done[m] = 1;
                prev[m] = rel;
            }
            all_done = all_done && done[m];
        }
    }
    if (!all_done) LRA_THROW("square root of the Coulomb matrix did not converge");
    launch_ns_finish(dY, dscale.as<double>(), dsel.as<int>(), nm, n, pl, A, st);
    HIP_CHECK(hipStreamSynchronize(st));
}

// Filtered square root of the symmetric n x n matrix A (in place): A <- sum_{lam_j >= thr, lam_j > 0}
// lam_j^{1/2} u_j u_j^T from its eigen-decomposition (power_hemat, src/math/matrix_m.h:916-970;
// the real embedding of a Hermitian matrix has every eigenvalue twice and the embedded root).
// The eigen-decomposition is rocSOLVER's syevd, once per q; the root is one GEMM B^T B with the
// eigenvectors scaled by lam^{1/4}.  top (optional, length n / halves): the eigenvector of the
// largest eigenvalue, taken from one diagonal half of an embedded matrix when halves = 2.
// Returns the largest and second largest eigenvalue.
std::pair<double, double> eig_sqrt(double *A, int n, double thr, double *top, int halves, hipStream_t st) {
    static rocblas_handle handle = nullptr;
    if (!handle && rocblas_create_handle(&handle) != rocblas_status_success)
        LRA_THROW("rocblas_create_handle failed");
    if (rocblas_set_stream(handle, st) != rocblas_status_success) LRA_THROW("rocblas_set_stream failed");
    const size_t nn = (size_t)n * n;
    DevBuf dU(nn * 8), dW((size_t)n * 8), dE((size_t)n * 8), dinfo(8), df((size_t)n * 8);
    HIP_CHECK(hipMemcpyAsync(dU.get(), A, nn * 8, hipMemcpyDeviceToDevice, st));
    // column-major eigenvectors of a symmetric matrix: row j of the row-major view is u_j
    if (rocsolver_dsyevd(handle, rocblas_evect_original, rocblas_fill_lower, n, dU.as<double>(), n, dW.as<double>(),
                         dE.as<double>(), reinterpret_cast<rocblas_int *>(dinfo.get())) != rocblas_status_success)
        LRA_THROW("rocsolver_dsyevd failed");
    std::vector<double> lam(n);
    int info = 0;
    HIP_CHECK(hipMemcpyAsync(lam.data(), dW.get(), (size_t)n * 8, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipMemcpyAsync(&info, dinfo.get(), sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    if (info != 0) LRA_THROW("eigen-decomposition of the Coulomb matrix did not converge");
    if (top) {
        std::vector<double> u(n);
        HIP_CHECK(hipMemcpyAsync(u.data(), dU.as<double>() + (size_t)(n - 1) * n, (size_t)n * 8, hipMemcpyDeviceToHost,
                                 st));
        HIP_CHECK(hipStreamSynchronize(st));
        const int h = n / halves;
        int best = 0;
        double bn = -1;
        for (int c = 0; c < halves; ++c) {
            double s2 = 0;
            for (int i = 0; i < h; ++i) s2 += u[(size_t)c * h + i] * u[(size_t)c * h + i];
            if (s2 > bn) { bn = s2; best = c; }
        }
        std::vector<double> t(u.begin() + (size_t)best * h, u.begin() + (size_t)(best + 1) * h);
        const double nr = std::sqrt(bn);
        for (double &x : t) x /= nr;
        HIP_CHECK(hipMemcpyAsync(top, t.data(), (size_t)h * 8, hipMemcpyHostToDevice, st));
        HIP_CHECK(hipStreamSynchronize(st));
    }
    std::vector<double> f(n);
    for (int j = 0; j < n; ++j) f[j] = (lam[j] >= thr && lam[j] > 0) ? std::pow(lam[j], 0.25) : 0.0;
    HIP_CHECK(hipMemcpyAsync(df.get(), f.data(), (size_t)n * 8, hipMemcpyHostToDevice, st));
    launch_scale_rows(dU.as<double>(), n, df.as<double>(), st);
    GemmBatch b;
    b.trans_a = true;
    b.add(make_prob(n, n, n, 0, n, 0, n, 0, n));
    b.finalize(T64x64, st);
    gemm_run(Prec::F64, b, dU.get(), dU.get(), A, 1.0, 0.0, st);
    HIP_CHECK(hipStreamSynchronize(st));
    // largest distinct eigenvalues (an embedded matrix repeats each one)
    const double l0 = lam[n - 1], l1 = lam[std::max(0, n - 1 - halves)];
    return {l0, l1};
}

// the blocks of the k points qs
void stage_coulomb(const RpaEngine &R0, const std::map<std::tuple<int, int, int>, std::vector<cplx>> &store,
                   const std::vector<int> &qs, CoulombStage &out, hipStream_t st) {
    std::vector<VBlock> desc;
    std::vector<cplx> vals;
    out.first.assign(1, 0);
    out.vmax.assign(qs.size(), 0.0);
    out.imax.assign(qs.size(), 0.0);
    for (size_t i = 0; i < qs.size(); ++i) {
        for (auto it = store.lower_bound({qs[i], 0, 0}); it != store.end() && std::get<0>(it->first) == qs[i]; ++it) {
            const int I = std::get<1>(it->first), J = std::get<2>(it->first);
            if (I > J) continue;
            if (it->second.size() != (size_t)R0.na[I] * R0.na[J]) LRA_THROW("Coulomb block of the wrong size");
            for (const cplx &v : it->second) {
                out.vmax[i] = std::max(out.vmax[i], std::norm(v));
                out.imax[i] = std::max(out.imax[i], std::fabs(v.imag()));
            }
            desc.push_back({(long long)vals.size(), (int)R0.abf[I], (int)R0.abf[J], R0.na[I], R0.na[J], I == J ? 1 : 0, (int)i});
            vals.insert(vals.end(), it->second.begin(), it->second.end());
        }
        out.vmax[i] = std::sqrt(out.vmax[i]);
        out.first.push_back((int)desc.size());
    }
    out.blk = upload(vals, st);
    out.desc = upload(desc, st);
    HIP_CHECK(hipStreamSynchronize(st));
}

// dense matrices of qs[i0, i0 + cnt) into V, stride elements apart
void dense_coulomb(const CoulombStage &cs, int i0, int cnt, int n, DenseLayout lay, bool real_part, double *V,
                   long long stride, hipStream_t st) {
    HIP_CHECK(hipMemsetAsync(V, 0, sizeof(double) * (size_t)stride * cnt, st));
    launch_v_scatter(cs.blk.as<double>(), cs.desc.as<VBlock>() + cs.first[i0], cs.first[i0 + cnt] - cs.first[i0], V, n,
                     lay, real_part ? 1 : 0, i0, stride, st);
}
}  // namespace

namespace {
// at_least: what a later phase will take of the same buffer
template <class F> void carve(DevBuf &buf, F layout, size_t at_least = 0) {
    Carve count{nullptr};
    layout(count);
    buf.reserve(std::max(count.at, at_least));
    Carve c{buf.as<char>()};
    layout(c);
}
}  // namespace

double GwEngine::keep_bytes() {
    const char *e = std::getenv("LIBRPA_AMD_KEEP_BYTES");
    return e ? std::atof(e) : 12e9;
}

void GwEngine::sigma_layout(Carve &c, SigmaWork &w) const {
    const size_t nel = (size_t)nR * NAO * NAO, next = (size_t)NE * NAO * NAO;
    w.U = c.take<char>(signs * (size_t)u_elems * nbatch * ts);
    w.Ghat = c.take<char>((size_t)max_ghat * nbatch * ts);
    w.CW = c.take<char>(((size_t)max_cw * nbatch + kChi0Pad) * ts);
    w.Y = c.take<char>(signs * (size_t)y_elems * nbatch * ts);
    w.sigma = c.take<char>(2 * (size_t)nbatch * (2 * nel + next) * ts);
    w.Wlow = prec != Prec::F64 ? c.take<char>((size_t)nbatch * nR * NABF * NABF * ts) : nullptr;
}

void GwEngine::build_w(const Dataset &ds, const TFGrid &g, Result &out) {
    auto &prof = profiler();
    const double t0 = now_s();
    RpaEngine &R0 = *rpa;
    const hipStream_t st = R0.stream;
    const int n = NABF;
    const int nw = g.n;
    if (R0.ntau_done != g.n) LRA_THROW("chi0 must be built on the same grid before W");
    if (R0.host_staged) LRA_THROW("G0W0 needs the device-resident chi0 store (too large for this device)");
    out.Wrt.alloc(sizeof(double) * (size_t)g.n * nR * n * n);
    HIP_CHECK(hipMemsetAsync(out.Wrt.get(), 0, out.Wrt.bytes(), st));
    // no truncated Coulomb: v_c^{1/2} = 0 and W = 0 (epsilon.cpp:1862-1879)
    out.w_zero = ds.vq_cut.empty();
    if (out.w_zero) { HIP_CHECK(hipStreamSynchronize(st)); t_w = now_s() - t0; return; }
    // irreducible q and their star sizes; a reducible q must be the time-reversal partner of its
    // irreducible q (the assumption of FT_Wc_freq_q, epsilon.cpp:2430-2452)
    std::vector<int> mult(nk, 0);
    for (int k = 0; k < nk; ++k) {
        const int r = ds.ibz_map.empty() ? k : ds.ibz_map[k];
        if (r < 0 || r >= nk || (!ds.ibz_map.empty() && ds.ibz_map[r] != r))
            LRA_THROW("IBZ mapping: k point " + std::to_string(k) + " maps to a point that is not irreducible");
        if (r != k) {
            bool partner = true;
            for (int d = 0; d < 3; ++d) {
                const double sum = ds.kfrac[(size_t)k * 3 + d] + ds.kfrac[(size_t)r * 3 + d];
                partner = partner && std::fabs(sum - std::round(sum)) < 1e-8;
            }
            if (!partner)
                LRA_THROW("G0W0 with an IBZ mapping needs every reducible q to be -q of its irreducible q (k point " +
                          std::to_string(k) + ")");
        }
        mult[r]++;
    }
    const bool herm = nk > 1;
    const DenseLayout lay = herm ? kPlanar : kReal;
    const int N = 2 * n, pl = herm ? 2 : 1;
    const long long plane = (long long)n * n, nn = plane * pl, im = herm ? 4 * plane : 0, NN = 4 * plane * pl;
    std::vector<int> qs;
    for (int k = 0; k < nk; ++k)
        if (mult[k] > 0) qs.push_back(k);
    const int nq = (int)qs.size();
    // the Coulomb inputs go to the device once per plan and list of q (the engine goes with the inputs).
    // v_c = v lets W = L M^{-1} L^T - v use the Cholesky factor of v; otherwise the square roots
    // of v and v_c are formed and W = v_c^{1/2} eps^{-1} v_c^{1/2} - v_c
    if (v_qs != qs) {
        v_qs.clear();
        same_cut = ds.vq_cut.size() == ds.vq.size();
        for (const auto &kv : ds.vq) {
            auto it = ds.vq_cut.find(kv.first);
            same_cut = same_cut && it != ds.vq_cut.end() && it->second.size() == kv.second.size();
            for (size_t i = 0; same_cut && i < kv.second.size(); ++i)
                same_cut = it->second[i] == kv.second[i] ||
                           std::abs(it->second[i] - kv.second[i]) <= 1e-12 * (1.0 + std::abs(kv.second[i]));
        }
        stage_coulomb(R0, ds.vq, qs, vst, st);
        if (!same_cut) stage_coulomb(R0, ds.vq_cut, qs, vcst, st);
        v_qs = qs;
    }
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    free_b += work.bytes();
    // chi0(R, omega) once for all q when it fits in a quarter of the free memory
    if (!R0.chiw_ok && R0.form_chiw(g, 0.25 * (double)free_b, st)) {
        HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
        free_b += work.bytes();
    }
    // all frequencies of several q per pass (q is the inner loop of every launch), or some of one q
    const double per_w = 8.0 * ((double)NN + 2.0 * nn) + 16.0 * pl * N * (N >= (herm ? 2048 : 4096) ? (herm ? 1024 : 2048) : (herm ? 256 : 512));
    const double per_q = 8.0 * 14 * nn;
    const double budget = std::min(160e9, 0.7 * (double)free_b) - per_q;
    const auto cap = [](const char *name, int v) {
        const char *e = std::getenv(name);
        return e ? std::max(1, std::min(v, std::atoi(e))) : v;
    };
    const int WCH = cap("LIBRPA_AMD_W_FREQS", std::max(1, std::min(nw, (int)(budget / per_w))));
    const int QG = WCH < nw ? 1 : cap("LIBRPA_AMD_W_QGROUP", std::max(1, std::min(nq, (int)((budget + per_q) / (nw * per_w + per_q)))));
    const int UCH = QG > 1 ? QG * nw : WCH;
    // F: v and then its factor (Cholesky, or square root); C: v_c and then its root; V0: v_c, or S_c S_c
    // when a root is filtered
    double *F, *C, *V0, *D, *X, *A, *acc, *Sg, *ld, *U0, *Q, *dph, *dcoef;
    int *flag;
    const auto layout = [&](Carve &c) {
        F = c.take<double>(2 * nn * QG);
        C = F + nn * QG;
        V0 = c.take<double>(nn * QG);
        D = c.take<double>(nn * UCH);
        X = c.take<double>(nn * UCH);
        A = c.take<double>(NN * UCH);
        acc = c.take<double>(UCH);
        Sg = c.take<double>((size_t)n * QG);
        ld = c.take<double>(QG);
        U0 = c.take<double>(n);
        Q = c.take<double>(WCH);
        dph = c.take<double>(2 * (size_t)nR * QG);
        dcoef = c.take<double>((size_t)UCH * g.n);
        flag = c.take<int>(2);
    };
    SigmaWork later;
    Carve count{nullptr};
    sigma_layout(count, later);
    carve(work, layout, count.at);
    DevBuf dE;
    std::vector<double> hsg;
    HIP_CHECK(hipMemsetAsync(acc, 0, 8 * (size_t)UCH, st));
    HIP_CHECK(hipMemsetAsync(flag, 0, 2 * sizeof(int), st));
    CholWork &cw = R0.ec_cw;
    // L S L^H of cnt matrices in place; which of them have a zero or negative pivot: v^{1/2} must then come
    // from the eigen-decomposition with the negative eigenvalues dropped (power_hemat, matrix_m.h:916-970).
    // A zero pivot raises the flag of the whole batch, whose matrices are then looked at one by one.
    auto factor = [&](double *M, int cnt, std::vector<char> &neg) {
        neg.assign(cnt, 0);
        // (X is free until chi0's products)
        if (cnt > 1) HIP_CHECK(hipMemcpyAsync(X, M, nn * 8 * cnt, hipMemcpyDeviceToDevice, st));
        auto run = [&](int m0, int m1) {
            HIP_CHECK(hipMemsetAsync(ld, 0, 8 * (size_t)QG, st));
            HIP_CHECK(hipMemsetAsync(flag + 1, 0, sizeof(int), st));
            cholesky_logdet_batched(M + m0 * nn, nn, m1 - m0, n, n, ld, 1, flag + 1, true, cw, st,
                                    -1, Sg, n, herm ? plane : 0);
            hsg.resize((size_t)n * (m1 - m0));
            int zf = 0;
            HIP_CHECK(hipMemcpyAsync(hsg.data(), Sg, 8 * hsg.size(), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipMemcpyAsync(&zf, flag + 1, sizeof(int), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipStreamSynchronize(st));
            for (int m = m0; m < m1; ++m)
                for (int i = 0; i < n; ++i)
                    if (!(hsg[(size_t)(m - m0) * n + i] > 0)) neg[m] = 1;
            return zf != 0;
        };
        if (!run(0, cnt)) return;
        if (cnt == 1) { neg[0] = 1; return; }
        HIP_CHECK(hipMemcpyAsync(M, X, nn * 8 * cnt, hipMemcpyDeviceToDevice, st));
        for (int m = 0; m < cnt; ++m) {
            neg[m] = 0;
            if (run(m, m + 1)) neg[m] = 1;
        }
    };
    // head replacement at q = 0: eps_mac per frequency and the leading eigenvector of Re v(0)
    DevBuf dHead;
    if (!head.empty()) {
        if ((int)head.size() != nw) LRA_THROW("dielectric function: one value per frequency of the grid is needed");
        dHead = upload(head, st);
    }
    // filtered root of one matrix, through the real embedding when there are k points
    auto eig_root = [&](double *M, double *top) {
        if (!herm) return eig_sqrt(M, n, sqrt_threshold, top, 1, st);
        dE.reserve(4 * plane * 8);
        launch_planes_to_embedded(M, dE.as<double>(), n, st);
        const auto r = eig_sqrt(dE.as<double>(), 2 * n, sqrt_threshold, top, 2, st);
        launch_embedded_to_planes(dE.as<double>(), M, n, st);
        HIP_CHECK(hipStreamSynchronize(st));
        return r;
    };
    std::map<std::tuple<int, int, bool>, std::pair<GemmBatch, GemmBatch>> batches;
    auto get_batches = [&](int qg, int cnt, bool tri) -> std::pair<GemmBatch, GemmBatch> & {
        auto it = batches.find({qg, cnt, tri});
        if (it != batches.end()) return it->second;
        auto &pr = batches[{qg, cnt, tri}];
        GemmBatch &bx = pr.first, &bm = pr.second;
        bm.trans_a = true;
        bm.lower_only = true;
        for (int qi = 0; qi < qg; ++qi)
            for (int w = 0; w < cnt; ++w)
                for (int h = 0; h < pl; ++h) {
                    // plane h of X = D F and of F^H X
                    const long long u = ((long long)qi * cnt + w), l = qi * nn;
                    GemmProb px = make_prob(n, n, n, u * nn, n, l + h * plane, n, u * nn + h * plane, n);
                    px.kmode = tri ? 1 : 0;  // triangular Cholesky factor, or the full square root
                    GemmProb pm = make_prob(n, n, n, l, n, u * nn + h * plane, n, u * NN + h * im, N);
                    pm.kmode = tri ? 2 : 0;
                    if (herm) {
                        px.sgn2 = h ? 1 : -1;
                        px.a_off2 = u * nn + plane;
                        px.b_off2 = l + (1 - h) * plane;
                        pm.sgn2 = h ? -1 : 1;
                        pm.a_off2 = l + plane;
                        pm.b_off2 = u * nn + (1 - h) * plane;
                    }
                    bx.add(px);
                    bm.add(pm);
                }
        bx.finalize(T64x64, st);
        bm.finalize(T64x64, st);
        return pr;
    };
    const auto &cells = R0.cells;
    for (int iq0 = 0; iq0 < nq; iq0 += QG) {
        const int qg = std::min(QG, nq - iq0);
        if (verbose) { fprintf(stderr, "[librpa-mi355x] W: q %d / %d (%.1f s)\n", qs[iq0] + 1, nk, now_s() - t0); fflush(stderr); }
        std::vector<const double *> kfs(qg);
        int gamma = -1;  // position of q = 0 in the pass
        for (int i = 0; i < qg; ++i) {
            kfs[i] = &ds.kfrac[(size_t)qs[iq0 + i] * 3];
            if (std::fabs(kfs[i][0]) < 1e-12 && std::fabs(kfs[i][1]) < 1e-12 && std::fabs(kfs[i][2]) < 1e-12) gamma = i;
        }
        const bool head_here = gamma >= 0 && !head.empty();
        // v^{1/2} from Re v at q = 0 (power_hemat_blacs_real, epsilon.cpp:2019-2024)
        if (gamma >= 0 && same_cut && vst.imax[iq0 + gamma] > 1e-12 * std::max(vst.vmax[iq0 + gamma], 1e-300))
            LRA_THROW("W at q = 0 with v_c = v needs a real Coulomb matrix (Im v(0) != 0)");
        auto fill_v = [&](double *dst) {
            dense_coulomb(vst, iq0, qg, n, lay, false, dst, nn, st);
            if (gamma >= 0) dense_coulomb(vst, iq0 + gamma, 1, n, lay, true, dst + gamma * nn, nn, st);
        };
        std::vector<char> neg(qg, 0), negc(qg, 0);
        bool tri = same_cut && sqrt_threshold <= 0;  // every factor of the pass is a Cholesky factor
        if (tri) {
            // v_c = v with v = L S L^T, S = I: the Cholesky identity
            prof.begin("gw_w_chol_v", st);
            fill_v(V0);
            HIP_CHECK(hipMemcpyAsync(F, V0, nn * 8 * qg, hipMemcpyDeviceToDevice, st));
            factor(F, qg, neg);
            prof.end("gw_w_chol_v", st, (herm ? 4.0 : 1.0) * qg * n * (double)n * n / 3.0);
        }
        std::vector<char> chol(qg, 0);
        for (int i = 0; i < qg; ++i) {
            chol[i] = same_cut && sqrt_threshold <= 0 && !neg[i] && !(head_here && i == gamma);
            tri = tri && chol[i];
        }
        if (tri || (same_cut && std::count(chol.begin(), chol.end(), 1) > 0))
            HIP_CHECK(hipMemcpyAsync(C, F, nn * 8 * qg, hipMemcpyDeviceToDevice, st));
        if (!tri) {
            // F <- S = v^{1/2}; C <- S_c = v_c^{1/2} (complex v_c kept, as the reference does);
            // V0 <- v_c, or S_c S_c when a root is filtered
            prof.begin("gw_w_sqrt_v", st);
            std::vector<char> eig(qg, 0), eigc(qg, 0);
            if (!same_cut) {
                for (int i = 0; i < qg; ++i)
                    if (!herm && vcst.imax[iq0 + i] > 1e-12 * std::max(vcst.vmax[iq0 + i], 1e-300))
                        LRA_THROW("a complex truncated Coulomb matrix at Gamma-only sampling is outside this build");
                fill_v(F);
                dense_coulomb(vcst, iq0, qg, n, lay, false, C, nn, st);
                HIP_CHECK(hipMemcpyAsync(V0, C, nn * 8 * qg, hipMemcpyDeviceToDevice, st));
                if (sqrt_threshold <= 0) {
                    // (D is free until chi0 is assembled)
                    HIP_CHECK(hipMemcpyAsync(D, F, nn * 8 * qg, hipMemcpyDeviceToDevice, st));
                    factor(D, qg, neg);
                    HIP_CHECK(hipMemcpyAsync(D, C, nn * 8 * qg, hipMemcpyDeviceToDevice, st));
                    factor(D, qg, negc);
                }
            } else if (sqrt_threshold > 0) {
                fill_v(V0);
            }
            std::vector<int> sel;  // roots by iteration: F of i at i, C of i at QG + i
            for (int i = 0; i < qg; ++i) {
                if (chol[i]) continue;
                if (same_cut) HIP_CHECK(hipMemcpyAsync(F + i * nn, V0 + i * nn, nn * 8, hipMemcpyDeviceToDevice, st));
                const bool head_q = head_here && i == gamma;
                // (with v_c = v a pivot that is not positive is the reason to be here, or the threshold, or the head)
                eig[i] = same_cut || sqrt_threshold > 0 || head_q || neg[i];
                eigc[i] = !same_cut && (sqrt_threshold > 0 || negc[i]);
                if (!eig[i]) sel.push_back(i);
                if (!same_cut && !eigc[i]) sel.push_back(QG + i);
            }
            ns_sqrt(F, n, herm, sel, A, (size_t)NN * UCH, st);
            std::vector<long long> sq;
            std::vector<int> which;
            for (int i = 0; i < qg; ++i) {
                if (chol[i]) continue;
                const bool head_q = head_here && i == gamma;
                if (eig[i]) {
                    const auto top2 = eig_root(F + i * nn, head_q ? U0 : nullptr);
                    if (head_q && !(top2.first - top2.second > 1e-8 * std::fabs(top2.first)))
                        LRA_THROW("head of the dielectric matrix: the largest eigenvalue of v(0) is degenerate");
                }
                if (same_cut) HIP_CHECK(hipMemcpyAsync(C + i * nn, F + i * nn, nn * 8, hipMemcpyDeviceToDevice, st));
                else if (eigc[i]) eig_root(C + i * nn, nullptr);
                if (eig[i] || eigc[i]) {
                    GemmBatch b = square_batch(n, herm, {i * nn}, {i * nn}, st);
                    gemm_run(Prec::F64, b, C, C, V0 + i * nn, 1.0, 0.0, st);
                    HIP_CHECK(hipStreamSynchronize(st));  // b's problem list is freed here
                }
            }
            prof.end("gw_w_sqrt_v", st);
        }
        std::vector<double> ph((size_t)qg * nR * 2);
        for (int i = 0; i < qg; ++i)
            for (int rr = 0; rr < nR; ++rr) {
                const double ang = 2 * M_PI * (kfs[i][0] * cells[rr][0] + kfs[i][1] * cells[rr][1] + kfs[i][2] * cells[rr][2]);
                ph[((size_t)i * nR + rr) * 2] = std::cos(ang);
                ph[((size_t)i * nR + rr) * 2 + 1] = std::sin(ang);
            }
        HIP_CHECK(hipMemcpyAsync(dph, ph.data(), 8 * ph.size(), hipMemcpyHostToDevice, st));
        const int cstep = qg > 1 ? nw : WCH;
        for (int w0 = 0; w0 < nw; w0 += cstep) {
            const int cnt = std::min(cstep, nw - w0), nu = qg * cnt;
            prof.begin("gw_w_chi0q", st);
            R0.assemble_dense_q(g, kfs, w0, cnt, D, true, nn, lay, st);
            prof.end("gw_w_chi0q", st);
            auto &bb = get_batches(qg, cnt, tri);
            prof.begin("gw_w_gemm", st);
            gemm_run(Prec::F64, bb.first, D, F, X, 1.0, 0.0, st);
            launch_fill_aug(A, NN, im, qg, cnt, n, C, V0, st);
            gemm_run(Prec::F64, bb.second, F, X, A, -1.0, 1.0, st);
            if (head_here) {
                // eps += (eps_mac - u^T eps u) u u^T, u the leading eigenvector of Re v(0): the
                // head overwrite of epsilon.cpp:2106-2181 in the eigenbasis of v (real at q = 0)
                double *A0 = A + (long long)gamma * cnt * NN;
                HIP_CHECK(hipMemsetAsync(Q, 0, sizeof(double) * cnt, st));
                launch_head_quad(A0, NN, N, n, cnt, U0, Q, st);
                launch_head_update(A0, NN, N, n, cnt, U0, dHead.as<double>() + w0, Q, st);
            }
            prof.end("gw_w_gemm", st, bb.first.flops + bb.second.flops);
            prof.begin("gw_w_schur", st);
            cholesky_logdet_batched(A, NN, nu, N, N, acc, 1, flag, false, cw, st, n,
                                    nullptr, 0, im);
            prof.end("gw_w_schur", st, (herm ? 4.0 : 1.0) * nu * (7.0 / 3.0) * n * (double)n * n);
            // W(R, tau) += sum_(q, w) f2t(tau, w) / N_k (cos Re W + sin Im W)
            prof.begin("gw_w_accum", st);
            std::vector<double> coef((size_t)nu * g.n);
            for (int i = 0; i < qg; ++i)
                for (int w = 0; w < cnt; ++w)
                    for (int t = 0; t < g.n; ++t)
                        coef[((size_t)i * cnt + w) * g.n + t] = g.cos_f2t[(size_t)t * g.n + w0 + w] * mult[qs[iq0 + i]] / nk;
            HIP_CHECK(hipMemcpyAsync(dcoef, coef.data(), 8 * coef.size(), hipMemcpyHostToDevice, st));
            launch_w_accum(A, NN, im, qg, cnt, n, dcoef, g.n, dph, nR,
                           out.Wrt.as<double>(), st);
            HIP_CHECK(hipStreamSynchronize(st));
            prof.end("gw_w_accum", st, 0, 8.0 * nu * (double)nn * ceil_div(g.n, 4) + 16.0 * g.n * nR * (double)n * n);
        }
    }
    int hflag = 0;
    HIP_CHECK(hipMemcpyAsync(&hflag, flag, sizeof(hflag), hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    if (hflag) LRA_THROW("1 - v^1/2 chi0 v^1/2 is singular or not finite at some (q, omega)");
    const double n3 = (herm ? 4.0 : 1.0) * n * (double)n * n;
    flops_w = nq * (n3 / 3.0 + nw * (n3 + n3 / 3.0 + (7.0 / 3.0) * n3));
    t_w = now_s() - t0;
}

// ------------------------------------------------------------------------------------------
// Sigma(R, i omega)
// ------------------------------------------------------------------------------------------
void GwEngine::build_sigma(const Dataset &ds, const TFGrid &g, Result &out) {
    auto &prof = profiler();
    const double t0 = now_s();
    RpaEngine &R0 = *rpa;
    const hipStream_t st = R0.stream;
    const int nw = g.n;
    const long long nel = (long long)nR * NAO * NAO;
    out.Sre.alloc(sizeof(double) * (size_t)nspin * nw * nel);
    out.Sim.alloc(sizeof(double) * (size_t)nspin * nw * nel);
    HIP_CHECK(hipMemsetAsync(out.Sre.get(), 0, out.Sre.bytes(), st));
    HIP_CHECK(hipMemsetAsync(out.Sim.get(), 0, out.Sim.bytes(), st));
    if (out.w_zero) { HIP_CHECK(hipStreamSynchronize(st)); t_sigma = now_s() - t0; return; }
    const size_t next = (size_t)NE * NAO * NAO, sig_elems = 2 * (size_t)nbatch * (2 * nel + next);
    SigmaWork w;
    carve(work, [&](Carve &c) { sigma_layout(c, w); });
    char *const U = w.U, *const Ghat = w.Ghat, *const CW = w.CW, *const Y = w.Y, *const sigma = w.sigma, *const Wlow = w.Wlow;
    R0.prepare_gf(ds.mf, -1);  // all bands (get_gf_cplx_imagtimes_Rs, meanfield.cpp:309-365)
    const long long nn_abf = (long long)NABF * NABF, zg = (long long)nR * NAO * 2 * NAO;
    DevBuf dcw = upload(g.cos_t2f, st), dsw = upload(g.sin_t2f, st);
    // LIBRPA_AMD_TUNE_SIGMA=1 times the U and CW batches' candidate tiles on the first pass (the
    // trials cost about as much as they save in one G0W0 run, so the defaults are used otherwise)
    const char *tsg = std::getenv("LIBRPA_AMD_TUNE_SIGMA");
    const bool tune_sigma = R0.autotune && tsg && std::atoi(tsg) != 0;
    auto passes = [&](auto tag) {
        using T = decltype(tag);
        const T *G = R0.d_Gpm.as<T>();
        T *const tU = reinterpret_cast<T *>(U), *const tCW = reinterpret_cast<T *>(CW), *const tY = reinterpret_cast<T *>(Y);
        for (int it = 0, nz = 1; it < g.n; it += nz) {
            // tau points [it, it + nz) in one pass
            nz = std::min(nbatch, g.n - it);
            const void *Wf = out.Wrt.as<double>() + (size_t)it * nR * nn_abf;
            if (prec != Prec::F64) {
                launch_convert<double, float>(out.Wrt.as<double>() + (size_t)it * nR * nn_abf, reinterpret_cast<float *>(Wlow),
                                              (long long)nz * nR * nn_abf, st);
                Wf = Wlow;
            }
            if (verbose) {
                HIP_CHECK(hipStreamSynchronize(st));
                fprintf(stderr, "[librpa-mi355x] Sigma_c: tau %d / %d (%.1f s)\n", it + 1, g.n, now_s() - t0);
                fflush(stderr);
            }
            for (int s = 0; s < nspin; ++s) {
                R0.build_gf(ds.mf, &g.tau[it], nz, s);
                T *sig = reinterpret_cast<T *>(sigma), *s2 = sig + 2 * (size_t)nbatch * nel, *ext = s2 + 2 * (size_t)nbatch * nel;
                HIP_CHECK(hipMemsetAsync(sigma, 0, sig_elems * ts, st));
                for (int sg0 = 0; sg0 < 2; sg0 += signs) {
                    // U_J(S) for all J, S
                    for (auto &c : uchunks) {
                        if (c.sg >= 0 && c.sg != sg0) continue;
                        prof.begin("gw_gather", st);
                        launch_gather_cols<T>(G, 2LL * NAO, reinterpret_cast<T *>(Ghat), c.d_jobs.template as<GatherJob>(), (int)c.jobs.size(),
                                              c.d_colsrc.template as<long long>(), NAO, c.max_gcol, st, nz, zg, c.ghat_elems);
                        prof.end("gw_gather", st, 0, 2.0 * nz * c.ghat_elems * ts);
                        prof.begin("gw_U", st);
                        c.ub.nz = nz;
                        c.ub.za = c.ghat_elems;
                        c.ub.zc = signs * u_elems;
                        if (tune_sigma && !c.ub.tuned)
                            c.ub.tune(prec, Ghat, R0.d_CWb.get(), U, 1.0, 0.0, st);
                        gemm_run(prec, c.ub, Ghat, R0.d_CWb.get(), U, 1.0, 0.0, st);
                        prof.end("gw_U", st, nz * c.ub.flops);
                    }
                    for (auto &c : xchunks) {
                        if ((s == 0 && sg0 == 0) || xchunks.size() > 1) {
                            prof.begin("gw_CW", st);
                            c.cwb.nz = nz;
                            c.cwb.zb = nR * nn_abf;
                            c.cwb.zc = c.cw_elems;
                            if (tune_sigma && !c.cwb.tuned)
                                c.cwb.tune(prec, R0.d_Cfin.get(), Wf, CW, 1.0, 0.0, st);
                            gemm_run(prec, c.cwb, R0.d_Cfin.get(), Wf, CW, 1.0, 0.0, st);
                            prof.end("gw_CW", st, nz * c.cwb.flops);
                        }
                        const SigBlk *blks = c.d_blks.template as<SigBlk>();
                        const Chi0Seg *segs = R0.d_segs.as<Chi0Seg>();
                        prof.begin("gw_D", st);
                        for (auto &t : c.d)
                            launch_sigma_d<T>(t.d.template as<SigTask>(), t.n, t.a, t.b, blks, segs, tCW, c.cw_elems,
                                              tU, u_elems, sig + sg0 * nel, nel, NAO, nz, signs, st);
                        prof.end("gw_D", st);
                        prof.begin("gw_B", st);
                        for (auto &t : c.b)
                            launch_sigma_b<T>(t.d.template as<SigTask>(), t.n, t.a, t.b, blks, segs, tCW, c.cw_elems,
                                              tU, u_elems, s2 + sg0 * nel, nel, NAO, nz, signs, st);
                        prof.end("gw_B", st);
                        prof.begin("gw_Y", st);
                        for (auto &t : ytasks)
                            launch_sigma_y<T>(t.d.template as<SigYTask>(), t.n, t.a, d_yent.as<SigYEnt>(), tCW, c.cw_elems,
                                              G, zg, tY, y_elems, NAO, c.x0, c.x1, c.x0 == 0, nz, signs, sg0, st);
                        prof.end("gw_Y", st);
                    }
                    prof.begin("gw_A3", st);
                    a3.nz = signs * nz;
                    a3.zb = y_elems;
                    a3.zc = (2 / signs) * (long long)next;
                    gemm_run(prec, a3, R0.d_Cfin.get(), Y, ext + sg0 * next, 1.0, 1.0, st);
                    prof.end("gw_A3", st, signs * nz * a3.flops);
                }
                prof.begin("gw_fold", st);
                launch_sigma_fold<T>(sig, s2, ext, d_fold.as<int>(), d_neg.as<int>(), NE, nR, NAO, nz, st);
                launch_sigma_freq<T>(sig, nel, dcw.as<double>(), dsw.as<double>(), nw, g.n, it, nz,
                                     out.Sre.as<double>() + (size_t)s * nw * nel, out.Sim.as<double>() + (size_t)s * nw * nel,
                                     st);
                prof.end("gw_fold", st);
            }
        }
    };
    if (prec == Prec::F64) passes(double());
    else passes(float());
    HIP_CHECK(hipStreamSynchronize(st));
    t_sigma = now_s() - t0;
}

void GwEngine::w_block(int it, int I, int J, int r, double *out) const {
    const RpaEngine &R0 = *rpa;
    const size_t nn = (size_t)NABF * NABF;
    std::vector<double> row(R0.na[J]);
    for (int mu = 0; mu < R0.na[I]; ++mu) {
        const size_t off = ((size_t)it * nR + r) * nn + (size_t)(R0.abf[I] + mu) * NABF + R0.abf[J];
        HIP_CHECK(hipMemcpy(out + (size_t)mu * R0.na[J], res->Wrt.as<double>() + off, sizeof(double) * R0.na[J],
                            hipMemcpyDeviceToHost));
    }
}

void GwEngine::sigma_block(int spin, int iw, int I, int J, int r, double *re, double *im) const {
    const RpaEngine &R0 = *rpa;
    const long long nel = (long long)nR * NAO * NAO;
    for (int i = 0; i < R0.nb[I]; ++i) {
        const size_t off = ((size_t)spin * ntau + iw) * nel + (size_t)r * NAO * NAO + (size_t)(R0.ao[I] + i) * NAO +
                           R0.ao[J];
        HIP_CHECK(hipMemcpy(re + (size_t)i * R0.nb[J], res->Sre.as<double>() + off, sizeof(double) * R0.nb[J],
                            hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(im + (size_t)i * R0.nb[J], res->Sim.as<double>() + off, sizeof(double) * R0.nb[J],
                            hipMemcpyDeviceToHost));
    }
}

// Sigma_KS(k, i w)_nn = sum_ab conj(U_na) Sigma(k)_ab U_nb with Sigma(k) = sum_R e^{i 2 pi k.R'} Sigma(R)
// and R' the image of R nearest to the atom pair (build_sigc_matrix_KS_blacs, gw.cpp:992-1040).
std::vector<std::vector<cplx>> GwEngine::ks_diag(const Dataset &ds, int spin, int ik,
                                                  const std::vector<int> &states) {
    const RpaEngine &R0 = *rpa;
    const hipStream_t st = R0.stream;
    const int nw = ntau;
    const double *kf = &ds.kfrac[(size_t)ik * 3];
    const bool frac = ds.frac.size() == 3 * (size_t)natom && ds.lat_set;
    std::vector<double> ph((size_t)natom * natom * nR * 2);
    for (int I = 0; I < natom; ++I)
        for (int J = 0; J < natom; ++J)
            for (int rr = 0; rr < nR; ++rr) {
                int Rb[3] = {R0.cells[rr][0], R0.cells[rr][1], R0.cells[rr][2]};
                if (frac) {
                    double best = 1e300;
                    int bc[3] = {Rb[0], Rb[1], Rb[2]};
                    for (int a = -1; a < 2; ++a)
                        for (int b = -1; b < 2; ++b)
                            for (int c = -1; c < 2; ++c) {
                                const int Rc[3] = {a * R0.period[0] + Rb[0], b * R0.period[1] + Rb[1],
                                                   c * R0.period[2] + Rb[2]};
                                double d2 = 0;
                                for (int x = 0; x < 3; ++x) {
                                    double v = 0;
                                    for (int y = 0; y < 3; ++y)
                                        v += (ds.frac[3 * I + y] - ds.frac[3 * J + y] - Rc[y]) * ds.latvec[3 * y + x];
                                    d2 += v * v;
                                }
                                if (d2 < best) { best = d2; bc[0] = Rc[0]; bc[1] = Rc[1]; bc[2] = Rc[2]; }
                            }
                    Rb[0] = bc[0]; Rb[1] = bc[1]; Rb[2] = bc[2];
                }
                const double ang = 2 * M_PI * (kf[0] * Rb[0] + kf[1] * Rb[1] + kf[2] * Rb[2]);
                ph[(((size_t)I * natom + J) * nR + rr) * 2] = std::cos(ang);
                ph[(((size_t)I * natom + J) * nR + rr) * 2 + 1] = std::sin(ang);
            }
    // one upload and one download per 16 states, in buffers that stay
    std::lock_guard<std::mutex> lk(ks_mu);
    const auto &Uk = ds.mf.wfc[(size_t)spin * nk + ik];
    std::vector<std::vector<cplx>> out(states.size(), std::vector<cplx>(nw));
    const long long nel = (long long)nR * NAO * NAO;
    for (size_t s0 = 0; s0 < states.size(); s0 += 16) {
        const int ns = (int)std::min<size_t>(16, states.size() - s0);
        std::vector<double> in(ph);
        in.resize(ph.size() + (size_t)ns * NAO * 2 + NAO);
        double *U = in.data() + ph.size();
        for (int a = 0; a < ns; ++a)
            for (int b = 0; b < NAO; ++b) {
                const cplx u = Uk[(size_t)states[s0 + a] * NAO + b];
                U[((size_t)a * NAO + b) * 2] = u.real();
                U[((size_t)a * NAO + b) * 2 + 1] = u.imag();
            }
        int *atom_of = reinterpret_cast<int *>(U + (size_t)ns * NAO * 2);
        for (int I = 0; I < natom; ++I)
            for (int i = 0; i < R0.nb[I]; ++i) atom_of[R0.ao[I] + i] = I;
        std::vector<double> Y((size_t)nw * NAO * ns * 2);
        ks_in.reserve(8 * in.size());
        ks_out.reserve(8 * Y.size());
        const double *dph = ks_in.as<double>(), *dU = dph + ph.size();
        HIP_CHECK(hipMemcpyAsync(ks_in.get(), in.data(), 8 * in.size(), hipMemcpyHostToDevice, st));
        launch_sigma_ks_rows(res->Sre.as<double>() + (size_t)spin * nw * nel, res->Sim.as<double>() + (size_t)spin * nw * nel,
                             nw, nR, NAO, reinterpret_cast<const int *>(dU + (size_t)ns * NAO * 2), natom, dph, dU, ns,
                             ks_out.as<double>(), st);
        HIP_CHECK(hipMemcpyAsync(Y.data(), ks_out.get(), Y.size() * 8, hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        for (int a = 0; a < ns; ++a)
            for (int w = 0; w < nw; ++w) {
                cplx acc(0, 0);
                for (int x = 0; x < NAO; ++x) {
                    const cplx y(Y[(((size_t)w * NAO + x) * ns + a) * 2], Y[(((size_t)w * NAO + x) * ns + a) * 2 + 1]);
                    acc += std::conj(Uk[(size_t)states[s0 + a] * NAO + x]) * y;
                }
                out[s0 + a][w] = acc;
            }
    }
    return out;
}

// ------------------------------------------------------------------------------------------
// analytic continuation and QP equation (host)
// ------------------------------------------------------------------------------------------
PadeAC::PadeAC(int n_pars, const std::vector<cplx> &xs, const std::vector<cplx> &data) {
    const int nd = (int)data.size();
    std::vector<cplx> px, pd;
    if (n_pars < 0) n_pars = nd;
    if (nd <= n_pars) {
        n_pars = nd;
        px = xs;
        pd = data;
    } else {
        // n_pars - 1 evenly spaced nodes, then the last datum. LibRPA sizes its node list to
        // n_pars and fills only the first n_pars - 1, so that datum sits at the node 0
        // (src/core/analycont.cpp:35-45); the same node keeps the continuation identical.
        const int step = nd / (n_pars - 1);
        for (int i = 0; i < n_pars - 1; ++i) { px.push_back(xs[(size_t)i * step]); pd.push_back(data[(size_t)i * step]); }
        px.push_back(cplx(0.0, 0.0));
        pd.push_back(data[nd - 1]);
    }
    n = n_pars;
    x = px;
    // reciprocal differences, g(i, p) for i >= p
    std::vector<cplx> gm((size_t)n * n);
    for (int i = 0; i < n; ++i) gm[(size_t)i * n] = pd[i];
    for (int p = 1; p < n; ++p)
        for (int i = p; i < n; ++i)
            gm[(size_t)i * n + p] = (gm[(size_t)(p - 1) * n + p - 1] - gm[(size_t)i * n + p - 1]) /
                                    ((x[i] - x[p - 1]) * gm[(size_t)i * n + p - 1]);
    y.resize(n);
    for (int p = 0; p < n; ++p) y[p] = gm[(size_t)p * n + p];
}

cplx PadeAC::operator()(cplx z) const {
    cplx t(1.0, 0.0);
    for (int p = n - 1; p > 0; --p) t = 1.0 + y[p] * (z - x[p - 1]) / t;
    return y[0] / t;
}

int qpe_solve(const PadeAC &p, double e_mf, double e_fermi, double vxc, double sigx, double &e_qp, cplx &sigc,
              double diff_init, double thres, int n_iter_max) {
    const double escale = 0.1;
    int n_iter = 0;
    double e_last = e_mf, e_this;
    double diff = diff_init;
    cplx s_this, s_last;
    while (n_iter++ < n_iter_max) {
        e_this = e_last + escale * diff;
        s_this = p(cplx(e_this - e_fermi, 0.0));
        diff = e_mf - vxc + sigx + s_this.real() - e_this;
        e_last = e_mf - vxc + sigx + s_this.real();
        s_last = s_this;
        if (std::fabs(diff) < thres || n_iter == n_iter_max - 1) break;
    }
    sigc = s_last;
    e_qp = e_last;
    return n_iter > n_iter_max - 1 ? 1 : 0;
}

// ------------------------------------------------------------------------------------------
// API drivers
// ------------------------------------------------------------------------------------------
void gw_build_sigma(Dataset &d, const LibrpaOptions &o) {
    if (o.use_shrink_abfs == LIBRPA_SWITCH_ON) LRA_THROW("ABF shrinking is outside this build's path");
    if (o.sqrt_coulomb_threshold < 0) LRA_THROW("sqrt_coulomb_threshold must not be negative");
    lra_prepare_grid(d, o);
    // head of the dielectric matrix from the macroscopic dielectric function
    // (librpa_get_g0w0_sigc_kgrid path, src/api/compute_g0w0.cpp:102-118), on the grid's
    // frequencies as interpolate_dielec_func (src/core/dielecmodel.cpp:65-104) puts it:
    // 0 as given, 1 cubic spline, 2 Havriliak-Negami fit
    std::vector<double> head;
    if (o.replace_w_head == LIBRPA_SWITCH_ON && !d.dielect_omega.empty())
        head = interpolate_dielec(o.option_dielect_func, d.dielect_omega, d.dielect_val, d.grid.omega);
    auto eng = d.rpa;
    if (!eng || eng->prec != d.chi0_prec || eng->mixed != d.chi0_mixed || eng->planned_ntau != d.grid.n) {
        // the new plan sizes itself by the free memory: what the old engines hold beside the results that
        // the getters read goes back first (the results stay, should the new build fail)
        if (eng) {
            KeptMemory::InUse use(*eng);
            eng->release_stores();
        }
        if (d.gw) {
            KeptMemory::InUse use(*d.gw);
            d.gw->work.release();
        }
        if (d.gw && d.gw->rpa != eng) {
            KeptMemory::InUse use(*d.gw->rpa);
            d.gw->rpa->release_stores();
        }
        d.rpa.reset();
        eng = std::make_shared<RpaEngine>();
        eng->mixed = d.chi0_mixed;
        KeptMemory::InUse planning(*eng);
        eng->plan(d, d.chi0_prec, d.ec_prec, d.grid.n);
        d.rpa = eng;
    }
    // the plan and the work memory stay with the inputs they were made for
    auto gw = d.gw;
    if (!gw || gw->rpa != eng) gw = std::make_shared<GwEngine>();
    KeptMemory::InUse use_eng(*eng), use_gw(*gw);
    // what is large goes back however the build ends
    struct Trim {
        GwEngine &gw;
        RpaEngine &eng;
        ~Trim() {
            const double keep = GwEngine::keep_bytes();
            if ((double)gw.work.bytes() > keep) gw.work.release();
            if (eng.work_bytes() > keep) eng.release_work();
            if (eng.ec_bytes() > keep) eng.release_ec();
        }
    } trim{*gw, *eng};
    eng->build_chi0(d, d.grid, o.n_bands_chi0);
    // chi0(R, tau) stays; large chi0 work buffers and those of an earlier Ec evaluation are rebuilt on demand
    if (eng->work_bytes() > GwEngine::keep_bytes()) eng->release_work();
    if (eng->ec_bytes() > GwEngine::keep_bytes()) eng->release_ec();
    gw->verbose = o.output_level >= LIBRPA_VERBOSE_DEBUG;
    gw->head = head;
    gw->sqrt_threshold = o.sqrt_coulomb_threshold;
    if (gw->rpa != eng) gw->plan(d, eng);
    auto res = std::make_shared<GwEngine::Result>();
    gw->build_w(d, d.grid, *res);
    gw->build_sigma(d, d.grid, *res);
    gw->res = res;
    d.gw = gw;
}

void gw_sigc_kgrid(Dataset &d, const LibrpaOptions &o, int n_spins, int n_kpts_this, const int *iks_this,
                   int i_state_low, int i_state_high, const double *vxc, const double *vexx, double *sigc_re,
                   double *sigc_im) {
    const auto &mf = d.mf;
    i_state_low = std::max(0, i_state_low);
    i_state_high = std::min(mf.nbands, i_state_high);
    if (n_spins != mf.nspin) LRA_THROW("parsed nspins is not consistent with the SCF starting point");
    if (i_state_high <= i_state_low) return;
    const int nst = i_state_high - i_state_low;
    if (!d.gw) gw_build_sigma(d, o);
    GwEngine &g = *d.gw;
    std::vector<cplx> xs;
    for (int w = 0; w < d.grid.n; ++w) xs.push_back(cplx(0.0, d.grid.omega[w]));
    std::vector<int> states;
    for (int i = i_state_low; i < i_state_high; ++i) states.push_back(i);
    for (int isp = 0; isp < n_spins; ++isp) {
        const int start_isp = isp * n_kpts_this * nst;
        for (int kk = 0; kk < n_kpts_this; ++kk) {
            const int start_k = start_isp + kk * nst;
            const int ik = iks_this[kk];
            if (ik < 0 || ik >= mf.nk) LRA_THROW("k index out of range");
            auto vals = g.ks_diag(d, isp, ik, states);
            for (int i = 0; i < nst; ++i) {
                const double eks = mf.eps[((size_t)isp * mf.nk + ik) * mf.nbands + states[i]];
                sigc_re[start_k + i] = std::nan("");
                sigc_im[start_k + i] = std::nan("");
                PadeAC pade(o.n_params_anacon, xs, vals[i]);
                double eqp;
                cplx sc;
                if (qpe_solve(pade, eks, mf.efermi, vxc[start_k + i], vexx[start_k + i], eqp, sc) == 0) {
                    sigc_re[start_k + i] = sc.real();
                    sigc_im[start_k + i] = sc.imag();
                }
            }
        }
    }
}

}  // namespace lra
