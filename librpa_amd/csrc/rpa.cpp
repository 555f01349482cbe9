// Space-time chi0 builder and RPA correlation energy on one GPU.
//
// Per imaginary time tau (LibRPA build_chi0_q_space_time_LibRI_routing,
// src/core/chi0.cpp:1014-1164) the device pipeline is
//   1. G(R, +-tau): per k, M_k = U^T diag(s) conj(U) as one real GEMM on the
//      stacked [Re; Im] eigenvectors, then the k -> R sum keeping the real part
//      (build_gf_Rt_libri_serial, chi0.cpp:303-426).  G(+tau) and G(-tau) are
//      stored side by side per atom column block: Gpm[R][row][2*ao(J) + s*nb(J) + j].
//   2. W(K, J, S)[k, (j, nu)] = sum_{(L,R2) in N(J)} G(S+R2)_KL C^J(L,R2): one GEMM
//      per (J, S, sign) on a gathered G panel, written as W[(K, k)][(s, j)][nu].
//   3. chi0s(I,J,R) = sum_(K,R1,k) C^I [G_IJ W(K,J,R-R1)] + W(I,-R)^T W(J,R), one launch per tile
//      class (chi0.hip): the bracket is formed in registers and never stored.
// The four terms of LibRI's labels a1b1_a2b2 and a1b2_a2b1 called with
// (G+, G-) and (G-, G+) (thirdparty/LibRI/include/RI/physics/RPA.hpp:104-138)
// are the four (sign, term) products of step 3.
//
// chi0s(R, tau) of every tau stays resident; the tau -> omega cosine transform
// and the R -> q sum (chi_libri_ft_ct, chi0.cpp:507-596) are fused into the
// assembly of dense Hermitian chi0(q, omega) matrices, and Ec
// (compute_RPA_correlation_blacs_2d{,_gamma_only}, src/core/epsilon.cpp:43-558)
// uses ln |det(1 - V chi0)| = ln |det(S - L^T chi0 L)| with V = L S L^T (S = diag(+-1), the
// pivot signs; S = I for a positive-definite V).
#include "rpa.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <thread>

namespace lra {

namespace {
inline int bvk_mod(int v, int n) { return (((v % n) + 3 * n / 2) % n) - n / 2; }
double now_s() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
}  // namespace

namespace {
struct KeptList {
    std::mutex mu;
    std::set<KeptMemory *> all;
};
// (never destroyed: handles may outlive the statics of this file)
KeptList &kept() {
    static KeptList *l = new KeptList;
    return *l;
}
}  // namespace

KeptMemory::KeptMemory() {
    std::lock_guard<std::mutex> lk(kept().mu);
    kept().all.insert(this);
}

KeptMemory::~KeptMemory() {
    std::lock_guard<std::mutex> lk(kept().mu);
    kept().all.erase(this);
}

void KeptMemory::hold() {
    while (held.exchange(true)) std::this_thread::yield();  // (a reclaim in another thread)
}

void reclaim_kept_memory() {
    std::lock_guard<std::mutex> lk(kept().mu);
    for (KeptMemory *k : kept().all) {
        if (k->held.exchange(true)) continue;
        k->give_back();
        k->held = false;
    }
}

void reclaim_if_low() {
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    if (free_b < total_b / 2) reclaim_kept_memory();
}

int RpaEngine::cell_index(int x, int y, int z) const {
    const int x0 = -(period[0] / 2), y0 = -(period[1] / 2), z0 = -(period[2] / 2);
    return ((x - x0) * period[1] + (y - y0)) * period[2] + (z - z0);
}

int RpaEngine::fold_index(int x, int y, int z) const {
    return cell_index(bvk_mod(x, period[0]), bvk_mod(y, period[1]), bvk_mod(z, period[2]));
}

void RpaEngine::plan(const Dataset &ds, Prec p, Prec pe, int ntau) {
    prec = p;
    ec_prec = pe;
    planned_ntau = ntau;
    ts = (prec == Prec::F64) ? 8 : 4;
    // parts of each contraction (LIBRPA_AMD_SPLITK; default: by load; 1 = one plain write)
    int splitk = 0;
    if (const char *e = std::getenv("LIBRPA_AMD_SPLITK")) splitk = std::max(1, std::atoi(e));
    const auto &mf = ds.mf;
    natom = (int)ds.nb_wfc.size();
    if (natom == 0 || ds.nb_aux.size() != (size_t)natom) LRA_THROW("atomic basis sizes not set");
    nb.assign(ds.nb_wfc.begin(), ds.nb_wfc.end());
    na.assign(ds.nb_aux.begin(), ds.nb_aux.end());
    ao.assign(natom + 1, 0);
    abf.assign(natom + 1, 0);
    for (int a = 0; a < natom; ++a) { ao[a + 1] = ao[a] + nb[a]; abf[a + 1] = abf[a] + na[a]; }
    NAO = (int)ao[natom];
    NABF = (int)abf[natom];
    if (NAO != mf.nbasis) LRA_THROW("sum of atomic basis sizes != nbasis of the mean-field input");
    nk = mf.nk;
    nspin = mf.nspin;
    nbands = mf.nbands;
    if (mf.nspinor != 1) LRA_THROW("spinor (SOC) input is outside this build's path");
    for (int a = 0; a < 3; ++a) period[a] = ds.period[a] > 0 ? ds.period[a] : 1;
    if (period[0] * period[1] * period[2] != nk) LRA_THROW("k mesh size does not match the number of k points");
    cells.clear();
    for (int x = -(period[0] / 2); x <= (period[0] - 1) / 2; ++x)
        for (int y = -(period[1] / 2); y <= (period[1] - 1) / 2; ++y)
            for (int z = -(period[2] / 2); z <= (period[2] - 1) / 2; ++z) cells.push_back({x, y, z});
    nR = (int)cells.size();

    // ---- fold Cs to the BvK cell (RI_Tools::cal_period) ----
    std::map<std::tuple<int, int, int>, std::vector<double>> folded;  // (I, K, r) -> API layout
    for (const auto &kv : ds.cs) {
        const int I = std::get<0>(kv.first), K = std::get<1>(kv.first);
        const int r = fold_index(std::get<2>(kv.first), std::get<3>(kv.first), std::get<4>(kv.first));
        auto &dst = folded[{I, K, r}];
        if (dst.empty()) dst = kv.second;
        else for (size_t i = 0; i < dst.size(); ++i) dst[i] += kv.second[i];
    }
    n_cs_blocks = (long long)folded.size();
    nbrs.assign(natom, {});
    for (const auto &kv : folded) nbrs[std::get<0>(kv.first)].push_back({std::get<1>(kv.first), std::get<2>(kv.first)});
    koff.assign(natom, {});
    loff.assign(natom, {});
    ksum.assign(natom, 0);
    lsum.assign(natom, 0);
    cfin_off.assign(natom + 1, 0);
    cwb_off.assign(natom + 1, 0);
    for (int I = 0; I < natom; ++I) {
        long long k = 0, l = 0;
        for (const auto &n : nbrs[I]) {
            koff[I].push_back(k);
            loff[I].push_back(l);
            k += (long long)nb[n.K] * nb[I];
            l += nb[n.K];
        }
        ksum[I] = k;
        lsum[I] = l;
        cfin_off[I + 1] = cfin_off[I] + (long long)na[I] * ksum[I];
        cwb_off[I + 1] = cwb_off[I] + lsum[I] * nb[I] * na[I];
    }
    // packed Cs in the two GEMM layouts
    {
        std::vector<double> cfin(cfin_off[natom] + kChi0Pad), cwb(cwb_off[natom]);
        cnorm.assign(natom, 0.0);
        for (int I = 0; I < natom; ++I) {
            for (size_t n = 0; n < nbrs[I].size(); ++n) {
                const int K = nbrs[I][n].K;
                const auto &blk = folded.at({I, K, nbrs[I][n].r});
                double ss = 0;
                for (double v : blk) ss += v * v;
                cnorm[I] += std::sqrt(ss);
                const int ni = nb[I], nkk = nb[K], nm = na[I];
                for (int i = 0; i < ni; ++i)
                    for (int k = 0; k < nkk; ++k)
                        for (int mu = 0; mu < nm; ++mu) {
                            const double v = blk[((size_t)i * nkk + k) * nm + mu];
                            // Cfin_I stored transposed: [koff + k * nb(I) + i][mu]
                            cfin[cfin_off[I] + (size_t)(koff[I][n] + (size_t)k * ni + i) * nm + mu] = v;
                            // CWb_I[(loff + k)][i * na(I) + mu]   (I plays the role of J, K of L)
                            cwb[cwb_off[I] + (size_t)(loff[I][n] + k) * ni * nm + (size_t)i * nm + mu] = v;
                        }
            }
        }
        if (prec == Prec::F64) {
            d_Cfin = upload(cfin, stream);
            d_CWb = upload(cwb, stream);
            if (mixed) {
                std::vector<float> f1(cfin.begin(), cfin.end()), f2(cwb.begin(), cwb.end());
                d_Cfin32 = upload(f1, stream);
                d_CWb32 = upload(f2, stream);
                HIP_CHECK(hipStreamSynchronize(stream));
            }
        } else {
            std::vector<float> f1(cfin.begin(), cfin.end()), f2(cwb.begin(), cwb.end());
            d_Cfin = upload(f1, stream);
            d_CWb = upload(f2, stream);
            HIP_CHECK(hipStreamSynchronize(stream));
        }
    }

    // ---- outputs (I <= J, all cells), ordered by J ----
    outs.clear();
    E_tot = 0;
    for (int J = 0; J < natom; ++J)
        for (int I = 0; I <= J; ++I)
            for (int r = 0; r < nR; ++r) {
                outs.push_back({I, J, r, E_tot});
                E_tot += (long long)na[I] * na[J];
            }
    std::vector<int> out_index((size_t)natom * natom * nR, -1);
    for (size_t o = 0; o < outs.size(); ++o)
        out_index[((size_t)outs[o].I * natom + outs[o].J) * nR + outs[o].r] = (int)o;

    // ---- flop model (canonical count, per spin per tau) ----
    {
        double f = 0;
        for (int J = 0; J < natom; ++J) f += (double)nR * 2.0 * 2.0 * NAO * nb[J] * na[J] * lsum[J];
        for (const auto &o : outs)
            for (const auto &n : nbrs[o.I])
                f += 8.0 * nb[o.I] * nb[o.J] * nb[n.K] * na[o.J] + 2.0 * na[o.I] * nb[o.I] * nb[n.K] * na[o.J];
        flops_chi0_alg = f * ntau;
    }

    // ---- W(K, J, S) of every J stays resident: [(K, k)][(s', j)][nu] per (J, S) ----
    w_off.assign((size_t)natom * nR + 1, 0);
    for (int J = 0; J < natom; ++J)
        for (int S = 0; S < nR; ++S)
            w_off[(size_t)J * nR + S + 1] = w_off[(size_t)J * nR + S] + 2LL * nb[J] * NAO * na[J];
    // ---- chunking over J by memory budget (gathered G panels) ----
    reclaim_if_low();
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    // chi0(R, tau) of every tau beside the W slabs, or staged through pinned host memory
    const double w_bytes = (double)w_off.back() * ts, slice_bytes = (double)ts * E_tot;
    free_host_store();
    host_staged = w_bytes + slice_bytes * ntau + 24e9 > (double)free_b;
    if (const char *hs = std::getenv("LIBRPA_AMD_HOST_CHI0")) host_staged = host_staged || std::atoi(hs) != 0;
    double budget = host_staged ? std::min(48e9, 0.5 * ((double)free_b - w_bytes - slice_bytes - 16e9))
                                : std::min(48e9, 0.35 * (double)free_b - w_bytes);
    // LIBRPA_AMD_CHUNK_BYTES=<bytes> caps the chunk size (smaller chunks, same results)
    if (const char *cb = std::getenv("LIBRPA_AMD_CHUNK_BYTES")) {
        const double v = std::atof(cb);
        if (v > 0) budget = std::min(budget, v);
    }
    chunks.clear();
    {
        int j = 0;
        while (j < natom) {
            Chunk c;
            c.j_begin = j;
            long long g = 0;
            int jj = j;
            while (jj < natom) {
                const long long g1 = (long long)nR * 2 * NAO * lsum[jj];
                if (jj > j && (double)(g + g1) * ts > budget) break;
                g += g1;
                ++jj;
            }
            c.j_end = jj;
            c.ghat_elems = g;
            chunks.push_back(std::move(c));
            j = jj;
        }
    }

    const long long gpm_r = (long long)NAO * 2 * NAO;  // elements per cell of Gpm
    flops_chi0_exec = 0;
    ghat_max = 0;
    auto say = [&](const char *what, size_t a, size_t b) {
        if (!verbose) return;
        fprintf(stderr, "[librpa-mi355x] plan: %s %zu / %zu\n", what, a, b);
        fflush(stderr);
    };
    say("outputs (I <= J, R) and chunks", outs.size(), chunks.size());
    for (auto &c : chunks) {
        say("problem lists of chunk", (size_t)(&c - chunks.data()) + 1, chunks.size());
        // offsets inside the chunk buffers
        long long go = 0;
        for (int J = c.j_begin; J < c.j_end; ++J)
            for (int S = 0; S < nR; ++S)
                for (int sg = 0; sg < 2; ++sg) { c.ghat_off.push_back(go); go += (long long)NAO * lsum[J]; }
        auto ghat_at = [&](int J, int S, int sg) { return c.ghat_off[((size_t)(J - c.j_begin) * nR + S) * 2 + sg]; };
        auto w_at = [&](int J, int S) { return w_off[(size_t)J * nR + S]; };

        // gather jobs: Ghat(J,S,sg)[row][(n, l)] = G^sg(S + R2_n)[row][ao(L_n) + l]
        for (int J = c.j_begin; J < c.j_end; ++J)
            for (int S = 0; S < nR; ++S)
                for (int sg = 0; sg < 2; ++sg) {
                    GatherJob gj;
                    gj.dst_off = ghat_at(J, S, sg);
                    gj.ncol = (int)lsum[J];
                    gj.col_off = (int)c.colsrc.size();
                    for (const auto &n : nbrs[J]) {
                        const auto &R2 = cells[n.r];
                        const auto &Sv = cells[S];
                        const int rr = fold_index(Sv[0] + R2[0], Sv[1] + R2[1], Sv[2] + R2[2]);
                        for (int l = 0; l < nb[n.K]; ++l)
                            c.colsrc.push_back(rr * gpm_r + 2 * ao[n.K] + (long long)sg * nb[n.K] + l);
                    }
                    c.max_gcol = std::max(c.max_gcol, gj.ncol);
                    c.jobs.push_back(gj);
                }
        // W build: W[(K,k)][(s', j)][nu], s' = 1 holds W+ (from G+), s' = 0 holds W- (from G-)
        for (int J = c.j_begin; J < c.j_end; ++J)
            for (int S = 0; S < nR; ++S)
                for (int sg = 0; sg < 2; ++sg) {
                    const int sp = (sg == 0) ? 1 : 0;
                    GemmProb pr = make_prob(NAO, nb[J] * na[J], (int)lsum[J], ghat_at(J, S, sg), (int)lsum[J],
                                            cwb_off[J], nb[J] * na[J],
                                            w_at(J, S) + (long long)sp * nb[J] * na[J], 2 * nb[J] * na[J]);
                    c.wb.add(pr);  // K = 0 (an atom without Cs) writes zeros
                }
        c.wb.finalize(big_tile(prec), stream);
        c.d_jobs = upload(c.jobs, stream);
        c.d_colsrc = upload(c.colsrc, stream);
        flops_chi0_exec += c.wb.flops;
        ghat_max = std::max(ghat_max, c.ghat_elems);
    }
    // ---- the contraction: every output block (chi0.hip) ----
    {
        std::vector<Chi0Seg> segs;
        std::vector<int> segtab((size_t)natom * nR);
        for (int I = 0; I < natom; ++I)
            for (int r = 0; r < nR; ++r) {
                const size_t first = segs.size();
                segtab[(size_t)I * nR + r] = (int)first;
                int at = 0;
                for (const auto &n : nbrs[I]) {
                    const auto &R1 = cells[n.r];
                    const int S = fold_index(cells[r][0] - R1[0], cells[r][1] - R1[1], cells[r][2] - R1[2]);
                    for (int k = 0; k < nb[n.K]; ++k) segs.push_back({S, (int)ao[n.K] + k, at++, 0});
                }
                std::sort(segs.begin() + first, segs.end(), [](const Chi0Seg &a, const Chi0Seg &b) {
                    return std::make_pair(a.cell, a.row) < std::make_pair(b.cell, b.row);
                });
            }
        std::vector<Chi0Out> co(outs.size());
        out_flops.assign(outs.size(), 0.0);
        contract_flops = contract_bytes = 0;
        for (size_t o = 0; o < outs.size(); ++o) {
            const auto &O = outs[o];
            const auto &Rv = cells[O.r];
            const int mr = fold_index(-Rv[0], -Rv[1], -Rv[2]);
            Chi0Out &c = co[o];
            c.cfin = cfin_off[O.I];
            c.gpm = O.r * gpm_r + ao[O.I] * 2LL * NAO + 2 * ao[O.J];
            c.wseg = w_off[(size_t)O.J * nR];
            c.xa = w_off[(size_t)O.I * nR + mr] + ao[O.J] * 2 * nb[O.I] * na[O.I];
            c.xb = w_off[(size_t)O.J * nR + O.r] + ao[O.I] * 2 * nb[O.J] * na[O.J];
            c.eoff = O.eoff;
            c.I = O.I; c.J = O.J; c.r = O.r;
            c.ni = nb[O.I]; c.nj = nb[O.J]; c.ai = na[O.I]; c.aj = na[O.J];
            c.lsum = (int)lsum[O.I];
            c.segtab = segtab[(size_t)O.I * nR + O.r];
            // T, its contraction with C^I, and the direct term
            const double ni = c.ni, nj = c.nj, ai = c.ai, aj = c.aj;
            out_flops[o] = 4.0 * ni * nj * lsum[O.I] * aj + 2.0 * ai * ni * lsum[O.I] * aj + 4.0 * ai * aj * ni * nj;
            contract_flops += out_flops[o];
            contract_bytes += 2.0 * ts * ai * aj;
        }
        // what the contraction has to move: W and Cs read once, chi0s read and written
        contract_bytes += (double)ts * (w_off.back() + cfin_off[natom]);
        flops_chi0_exec += contract_flops;
        d_segs = upload(segs, stream);
        d_couts = upload(co, stream);
        // tau points per launch: one tau point of a small system leaves the device idle between its
        // launches, so several run as copies of one batch, up to about 120 GFLOP (2 ms), 8 GB and the
        // kTauMax that a kernel's arguments hold (an evenly spaced grid may have more points)
        double wflops = 0;
        for (const auto &c : chunks) wflops += c.wb.flops;
        const double per_tau = 8.0 * (2.0 * nk * (2.0 * nbands * NAO + 2.0 * NAO * NAO)) +
                               ts * ((double)nR * 2 * NAO * NAO + ghat_max + (double)w_off.back());
        nbatch = 1;
        if (!host_staged && chunks.size() == 1)
            nbatch = (int)std::max(1.0, std::min({(double)ntau, (double)kTauMax, std::ceil(1.2e11 / std::max(1.0, contract_flops + wflops)),
                                                  std::min(8e9, 0.1 * (double)free_b) / per_tau}));
        if (const char *e = std::getenv("LIBRPA_AMD_TAU_BATCH")) nbatch = std::max(1, std::min(nbatch, std::atoi(e)));
        nbatch = ceil_div(ntau, ceil_div(ntau, nbatch));
        ctasks[0].build(co, prec == Prec::F64, nbatch, splitk, stream);
        if (mixed) ctasks[1].build(co, false, nbatch, splitk, stream);
        d_skip.alloc(std::max<size_t>(1, outs.size()) * nbatch);
        HIP_CHECK(hipStreamSynchronize(stream));
    }
    flops_chi0_exec *= ntau;
    d_Ghat.alloc(ghat_max * nbatch * ts);
    d_W.alloc((size_t)(w_off.back() * nbatch + kChi0Pad) * ts);
    screen_plan(ds);

    // ---- G build data ----
    {
        std::vector<double> zz((size_t)nk * 2 * nbands * 2 * NAO), wre((size_t)nk * nbands * NAO),
            wim((size_t)nk * nbands * NAO);
        d_eps.alloc(sizeof(double) * (size_t)nspin * nk * nbands);
        d_wg.alloc(sizeof(double) * (size_t)nspin * nk * nbands);
        HIP_CHECK(hipMemcpyAsync(d_eps.get(), mf.eps.data(), d_eps.bytes(), hipMemcpyHostToDevice, stream));
        HIP_CHECK(hipMemcpyAsync(d_wg.get(), mf.wg.data(), d_wg.bytes(), hipMemcpyHostToDevice, stream));
        d_ZZ.alloc(sizeof(double) * zz.size() * nspin);
        d_wre.alloc(sizeof(double) * wre.size() * nspin);
        d_wim.alloc(sizeof(double) * wim.size() * nspin);
        for (int s = 0; s < nspin; ++s) {
            for (int k = 0; k < nk; ++k) {
                const auto &U = mf.wfc[(size_t)s * nk + k];
                if (U.size() != (size_t)nbands * NAO) LRA_THROW("eigenvectors missing for a k point");
                double *z = &zz[(size_t)k * 2 * nbands * 2 * NAO];
                for (int b = 0; b < nbands; ++b)
                    for (int j = 0; j < NAO; ++j) {
                        const double x = U[(size_t)b * NAO + j].real(), y = U[(size_t)b * NAO + j].imag();
                        z[(size_t)(2 * b) * 2 * NAO + j] = x;
                        z[(size_t)(2 * b) * 2 * NAO + NAO + j] = y;
                        z[(size_t)(2 * b + 1) * 2 * NAO + j] = y;
                        z[(size_t)(2 * b + 1) * 2 * NAO + NAO + j] = -x;
                        wre[((size_t)k * nbands + b) * NAO + j] = x;
                        wim[((size_t)k * nbands + b) * NAO + j] = y;
                    }
            }
            HIP_CHECK(hipMemcpy(d_ZZ.as<double>() + zz.size() * s, zz.data(), zz.size() * 8, hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(d_wre.as<double>() + wre.size() * s, wre.data(), wre.size() * 8, hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(d_wim.as<double>() + wim.size() * s, wim.data(), wim.size() * 8, hipMemcpyHostToDevice));
        }
        d_Zs.alloc(sizeof(double) * (size_t)nbatch * 2 * nk * 2 * nbands * NAO);
        d_Mst.alloc(sizeof(double) * (size_t)nbatch * 2 * nk * 2 * NAO * NAO);
        d_Gpm.alloc(ts * (size_t)nbatch * nR * NAO * 2 * NAO);
        std::vector<double> cs((size_t)nR * nk), sn((size_t)nR * nk);
        for (int r = 0; r < nR; ++r)
            for (int k = 0; k < nk; ++k) {
                const double *kf = &ds.kfrac[(size_t)k * 3];
                const double ang = 2 * M_PI * (kf[0] * cells[r][0] + kf[1] * cells[r][1] + kf[2] * cells[r][2]);
                cs[(size_t)r * nk + k] = std::cos(ang);
                sn[(size_t)r * nk + k] = std::sin(ang);
            }
        d_cs = upload(cs, stream);
        d_sn = upload(sn, stream);
        std::vector<int> gcol(2 * (size_t)NAO);
        for (int J = 0; J < natom; ++J)
            for (int j = 0; j < nb[J]; ++j)
                for (int sg = 0; sg < 2; ++sg) gcol[(size_t)sg * NAO + ao[J] + j] = (int)(2 * ao[J] + sg * nb[J] + j);
        d_gcol = upload(gcol, stream);
        HIP_CHECK(hipStreamSynchronize(stream));
    }

    // ---- chi0s store and transform descriptors ----
    d_chi0s.alloc(ts * (size_t)E_tot * (host_staged ? 1 : ntau));
    if (host_staged) {
        // pageable memory: a store this size can exceed what the host lets a process pin
        h_chi0s.assign(ntau, {});
        for (int t = 0; t < ntau; ++t) h_chi0s[t].resize(ts * (size_t)E_tot);
    }
    pairs.clear();
    pair_eoff.clear();
    n_pair_elems = 0;
    for (int I = 0; I < natom; ++I)
        for (int J = I; J < natom; ++J) {
            PairDesc pd;
            pd.I = I; pd.J = J; pd.naI = na[I]; pd.naJ = na[J];
            pd.rowI = (int)abf[I]; pd.colJ = (int)abf[J];
            pd.e0 = n_pair_elems;
            n_pair_elems += (long long)na[I] * na[J];
            pairs.push_back(pd);
            for (int r = 0; r < nR; ++r) {
                const int o = out_index[((size_t)I * natom + J) * nR + r];
                pair_eoff.push_back(o >= 0 ? outs[o].eoff : -1);
            }
        }
    d_pairs = upload(pairs, stream);
    d_pair_eoff = upload(pair_eoff, stream);
    HIP_CHECK(hipStreamSynchronize(stream));
}

void RpaEngine::prepare_gf(const MeanField &mf, int nbands_g) {
    // band ranges with non-zero weight for each sign
    bool same = !gb.empty();
    for (int sg = 0; sg < 2; ++sg) {
        int lo = nbands, hi = 0;
        for (int s = 0; s < nspin; ++s)
            for (int k = 0; k < nk; ++k)
                for (int b = 0; b < nbands; ++b) {
                    const double wgv = mf.wg[((size_t)s * nk + k) * nbands + b];
                    double w = (sg == 0) ? 1.0 / nk - wgv / 2 * nspin : wgv * 0.5 * nspin;
                    if (w < 0) w = 0;
                    if (nbands_g >= 0 && b >= nbands_g) w = 0;
                    if (w > 0) { lo = std::min(lo, b); hi = std::max(hi, b + 1); }
                }
        if (hi <= lo) { lo = 0; hi = 0; }
        same = same && band_lo[sg] == lo && band_hi[sg] == hi;
        band_lo[sg] = lo;
        band_hi[sg] = hi;
    }
    gf_nbands = nbands_g;
    if (same) return;
    // both signs in one batch; a sign without bands has K = 0 and gets zeros.  The signs take turns, and fewer
    // than 8 k points give 8 strips of rows each: every XCD works through one range of the tiles, and with all
    // of one sign before the other (K = 2 x the empty or the occupied bands, 12 : 1 on the 128-atom cell) half
    // of them ran out early (68 ms for 16 tau points, where two launches had taken 44).
    gb = GemmBatch();
    gb.trans_a = true;
    const long long zs_k = 2LL * nbands * NAO, mst_k = 2LL * NAO * NAO;
    const int strip = nk >= 8 ? 2 * NAO : std::max(64, ceil_div(2 * NAO, 8 * 64) * 64);
    for (int k = 0; k < nk; ++k)
        for (int m0 = 0; m0 < 2 * NAO; m0 += strip)
            for (int sg = 0; sg < 2; ++sg)
                gb.add(make_prob(std::min(strip, 2 * NAO - m0), NAO, 2 * (band_hi[sg] - band_lo[sg]),
                                 k * 2 * zs_k + 4LL * band_lo[sg] * NAO + m0, 2 * NAO,
                                 ((long long)sg * nk + k) * zs_k + 2LL * band_lo[sg] * NAO, NAO,
                                 ((long long)sg * nk + k) * mst_k + (long long)m0 * NAO, NAO));
    gb.zb = 2 * nk * zs_k;
    gb.zc = 2 * nk * mst_k;
    gb.finalize(T64x64, stream);
}

void RpaEngine::build_gf(const MeanField &mf, const double *taus, int nz, int s) {
    auto &prof = profiler();
    const size_t zz_s = (size_t)nk * 2 * nbands * 2 * NAO * s;
    const size_t w_s = (size_t)nk * nbands * NAO * s;
    const size_t e_s = (size_t)nk * nbands * s;
    const long long gpm_bytes = (long long)nz * nR * NAO * 2 * NAO * ts;
    if (nz > nbatch || nz > kTauMax) LRA_THROW("G build: more tau points than the buffers hold");
    TauList tl;
    tl.n = nz;
    for (int z = 0; z < nz; ++z) tl.t[z] = taus[z];
    prof.begin("gf_build", stream);
    launch_scale_bands(d_wre.as<double>() + w_s, d_wim.as<double>() + w_s, d_eps.as<double>() + e_s,
                       d_wg.as<double>() + e_s, d_Zs.as<double>(), nk, nbands, NAO, band_lo, band_hi, tl, mf.efermi,
                       nspin, gf_nbands, stream);
    gb.nz = nz;
    gemm_run(Prec::F64, gb, d_ZZ.as<double>() + zz_s, d_Zs.get(), d_Mst.get(), 1.0, 0.0, stream);
    if (cur == Prec::F64)
        launch_k2r<double>(d_Mst.as<double>(), d_cs.as<double>(), d_sn.as<double>(), d_gcol.as<int>(),
                           d_Gpm.as<double>(), nk, nR, NAO, tl, stream);
    else
        launch_k2r<float>(d_Mst.as<double>(), d_cs.as<double>(), d_sn.as<double>(), d_gcol.as<int>(), d_Gpm.as<float>(),
                          nk, nR, NAO, tl, stream);
    prof.end("gf_build", stream, nz * gb.flops, (double)gpm_bytes);
}

void RpaEngine::build_chi0(const Dataset &ds, const TFGrid &g, int nbands_g) {
    const auto &mf = ds.mf;
    auto &prof = profiler();
    const double t0 = now_s();
    const int ntau = g.n;
    chiw_ok = false;  // chi0(R, omega) of an earlier build is stale
    if (host_staged) d_chiw.release();  // its room goes back to G and W (reformed for Ec)
    prepare_gf(mf, nbands_g);
    d_Ghat.reserve(ghat_max * nbatch * ts);
    d_W.reserve((size_t)(w_off.back() * nbatch + kChi0Pad) * ts);
    if (mixed) {
        if (prec != Prec::F64) LRA_THROW("mixed chi0 precision needs the FP64 plan");
        if (const char *e = std::getenv("LIBRPA_AMD_MIXED_AMAX")) mixed_amax = std::atof(e);
    }
    cur = prec;
    // LIBRPA_AMD_AUTOTUNE=0 keeps the default tile shapes (no timing runs on first use)
    if (const char *at = std::getenv("LIBRPA_AMD_AUTOTUNE")) autotune = std::atoi(at) != 0;
    HIP_CHECK(hipMemsetAsync(d_chi0s.get(), 0, d_chi0s.bytes(), stream));
    if (screen_mode != 0 && nspin > 1) LRA_THROW("chi0 block screening needs nspin = 1");
    if (host_staged && collect) LRA_THROW("screening samples need the device-resident chi0 store (too large here)");
    if (screen_mode == 2) {
        if (screen_model.size() != (size_t)MLP_NMODEL) LRA_THROW("learned screening without a model");
        d_model = upload(screen_model, stream);
    }
    scr_blocks = scr_skipped = scr_flops = scr_flops_skipped = 0;
    if (collect) features.assign((size_t)ntau * MLP_NFEAT * outs.size(), 0.0f);
    bool tuned_chi0[2] = {false, false};  // [plan precision, FP32 of the mixed mode]
    n_lowp_tau = 0;
    // mixed precision: FP32 contractions for the tau points whose column of the cosine t->f matrix is
    // small (the transform amplifies chi0(R, tau) errors by that column's entries)
    std::vector<Prec> tau_prec(ntau, prec);
    for (int it = 0; mixed && it < ntau; ++it) {
        double amax = 0;
        for (int w = 0; w < g.n; ++w) amax = std::max(amax, std::fabs(g.cos_t2f[(size_t)w * g.n + it]));
        if (amax <= mixed_amax) tau_prec[it] = mixed_low;
    }
    const long long zg = (long long)nR * NAO * 2 * NAO, zw = w_off.back();
    for (int it = 0, nz = 1; it < ntau; it += nz) {
        // tau points [it, it + nz) of one precision in one pass
        cur = tau_prec[it];
        for (nz = 1; nz < nbatch && it + nz < ntau && tau_prec[it + nz] == cur; ++nz) {}
        const bool lowp = cur != prec;
        n_lowp_tau += lowp ? nz : 0;
        // low-precision tau points time under their own region names
        const char *lsuf = cur == Prec::BF16X3 ? "_bf16x3" : "_f32";
        auto rn = [lowp, lsuf](const char *r) { return lowp ? std::string(r) + lsuf : std::string(r); };
        const double bsc = lowp ? 4.0 / ts : 1.0;  // algorithmic bytes scale with the element size
        const void *CWb_p = lowp ? d_CWb32.get() : d_CWb.get();
        // the one slice of a host-staged store starts from zero at every tau
        if (host_staged) HIP_CHECK(hipMemsetAsync(d_chi0s.get(), 0, d_chi0s.bytes(), stream));
        if (mixed)
            for (auto &c : chunks) c.wb.use_tiles(cur, stream);
        for (int s = 0; s < nspin; ++s) {
            build_gf(mf, &g.tau[it], nz, s);
            if (s == 0 && (screen_mode != 0 || collect)) screen_taus(it, &g.tau[it], nz);
            // tiles are tuned per precision on the first tau point built at it
            const bool tune_now = autotune && s == 0 && !tuned_chi0[lowp];
            for (auto &c : chunks) {
                if (tune_now && verbose) {
                    fprintf(stderr, "[librpa-mi355x] chi0: tuning the W build of chunk %d / %zu\n",
                            (int)(&c - chunks.data()) + 1, chunks.size());
                    fflush(stderr);
                }
                prof.begin(rn("chi0_gather"), stream);
                if (cur == Prec::F64)
                    launch_gather_cols<double>(d_Gpm.as<double>(), 2LL * NAO, d_Ghat.as<double>(), c.d_jobs.as<GatherJob>(),
                                               (int)c.jobs.size(), c.d_colsrc.as<long long>(), NAO, c.max_gcol, stream, nz, zg,
                                               c.ghat_elems);
                else
                    launch_gather_cols<float>(d_Gpm.as<float>(), 2LL * NAO, d_Ghat.as<float>(), c.d_jobs.as<GatherJob>(),
                                              (int)c.jobs.size(), c.d_colsrc.as<long long>(), NAO, c.max_gcol, stream, nz, zg,
                                               c.ghat_elems);
                prof.end(rn("chi0_gather"), stream, 0, 2.0 * nz * c.ghat_elems * (lowp ? 4 : ts));
                c.wb.nz = nz;
                c.wb.za = c.ghat_elems;
                c.wb.zc = zw;
                if (tune_now && c.wb.cfg_by_prec[(int)cur] < 0) c.wb.tune(cur, d_Ghat.get(), CWb_p, d_W.get(), 1.0, 0.0, stream);
                prof.begin(rn("chi0_W"), stream);
                gemm_run(cur, c.wb, d_Ghat.get(), CWb_p, d_W.get(), 1.0, 0.0, stream);
                prof.end(rn("chi0_W"), stream, nz * c.wb.flops);
            }
            // the contraction; a BF16x3 tau point contracts in FP32 (the kernel is bound by its
            // operand reads there, and FP32 keeps more digits)
            const size_t coff = host_staged ? 0 : (size_t)it * E_tot;
            const unsigned char *skip = screen_mode != 0 ? d_skip.as<unsigned char>() : nullptr;
            const std::string region = cur == Prec::F64 || prec == Prec::F32 ? "chi0_contract" : "chi0_contract_f32";
            const int nout = (int)outs.size();
            prof.begin(region, stream);
            if (cur == Prec::F64)
                launch_chi0_contract<double, double>(ctasks[0], d_couts.as<Chi0Out>(), nout, d_segs.as<Chi0Seg>(),
                                                     d_Gpm.as<double>(), zg, d_W.as<double>(), zw, d_Cfin.as<double>(),
                                                     d_chi0s.as<double>() + coff, E_tot, NAO, nz, skip, stream);
            else if (lowp)
                launch_chi0_contract<float, double>(ctasks[1], d_couts.as<Chi0Out>(), nout, d_segs.as<Chi0Seg>(),
                                                    d_Gpm.as<float>(), zg, d_W.as<float>(), zw, d_Cfin32.as<float>(),
                                                    d_chi0s.as<double>() + coff, E_tot, NAO, nz, skip, stream);
            else
                launch_chi0_contract<float, float>(ctasks[0], d_couts.as<Chi0Out>(), nout, d_segs.as<Chi0Seg>(),
                                                   d_Gpm.as<float>(), zg, d_W.as<float>(), zw, d_Cfin.as<float>(),
                                                   d_chi0s.as<float>() + coff, E_tot, NAO, nz, skip, stream);
            prof.end(region, stream, nz * contract_flops, nz * contract_bytes * bsc);
        }
        tuned_chi0[lowp] = tuned_chi0[lowp] || autotune;
        if (verbose) {
            HIP_CHECK(hipStreamSynchronize(stream));
            fprintf(stderr, "[librpa-mi355x] chi0: tau %d / %d (%.1f s)\n", it + nz, ntau, now_s() - t0);
            fflush(stderr);
        }
        // a host-staged build keeps its slice in pageable host memory (stream order makes the next
        // tau's kernels wait for the copy)
        if (host_staged)
            HIP_CHECK(hipMemcpyAsync(h_chi0s[it].data(), d_chi0s.get(), ts * (size_t)E_tot, hipMemcpyDeviceToHost,
                                     stream));
    }
    cur = prec;  // later G builds (the self-energy's) run at the plan's precision
    HIP_CHECK(hipStreamSynchronize(stream));
    ntau_done = ntau;
    t_chi0 = now_s() - t0;
}

namespace {
// IBZ k list as in PeriodicBoundaryData::set_ibz_mapping (src/core/pbc.cpp:110-153)
void ibz_list(const Dataset &ds, int nk, std::vector<int> &ibz_k, std::vector<double> &w) {
    std::vector<int> map = ds.ibz_map;
    if ((int)map.size() != nk) { map.resize(nk); for (int k = 0; k < nk; ++k) map[k] = k; }
    std::map<int, int> pos;
    ibz_k.clear();
    w.clear();
    for (int k = 0; k < nk; ++k) {
        const int kb = map[k];
        auto it = pos.find(kb);
        if (it == pos.end()) { pos[kb] = (int)ibz_k.size(); ibz_k.push_back(kb); w.push_back(1.0 / nk); }
        else w[it->second] += 1.0 / nk;
    }
}
}  // namespace

RpaResult RpaEngine::ec(const Dataset &ds, const TFGrid &g) {
    auto &prof = profiler();
    const double t0 = now_s();
    RpaResult res;
    // a Hermitian matrix of a k point is its real and imaginary plane (n x n each), every product two
    // real segments: half the work and the bytes of the real embedding [[Re, -Im], [Im, Re]]
    const bool herm = nk > 1;
    const DenseLayout lay = herm ? kPlanar : kReal;
    const int n = NABF;
    const long long plane = (long long)n * n;
    const size_t nn = (size_t)plane * (herm ? 2 : 1);
    std::vector<int> ibz;
    std::vector<double> wq;
    ibz_list(ds, nk, ibz, wq);
    res.qcontrib.assign(ibz.size(), cplx(0, 0));
    const bool f64 = ec_prec == Prec::F64;
    const size_t es = f64 ? 8 : 4;
    const int nw = g.n;
    const int nq = (int)ibz.size();
    // chi0(R, omega) once for all q when it fits in a third of the free memory
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    if (!chiw_ok) {
        prof.begin("chi0_tau_to_omega", stream);
        if (host_staged) {
            // the chi0 work buffers make room for chi0(R, omega); build_chi0 reserves them again
            release_work();
            HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
            if (!form_chiw(g, 0.8 * (double)free_b, stream))
                LRA_THROW("chi0(R, omega) does not fit on the device beside the Ec buffers");
        } else {
            form_chiw(g, 0.33 * (double)free_b, stream);
        }
        prof.end("chi0_tau_to_omega", stream, 0, (double)E_tot * g.n * (ts * ceil_div(g.n, 8) + 8.0));
    }
    // all omega of a q are factorised together, as far as memory allows; small matrices (k-point
    // workloads) also take several q per pass, so that the GEMM, Cholesky and log-det launches hold
    // enough matrices to fill the device
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    // the Ec buffers kept from an earlier call count as free here (they are reused or regrown)
    const double held = ec_bytes();
    const double panel_w = 16.0 * n * (n >= (herm ? 2048 : 4096) ? 2048 : 512);  // Cholesky panels per matrix
    const double per_w = (double)nn * (3 * es + (f64 ? 0 : 8)) + panel_w;
    const double per_q = (double)nn * 12 + panel_w;
    const double budget = std::min(96e9, 0.6 * ((double)free_b + held)) - (double)nn * 12;
    const int WCH = std::max(1, std::min(nw, (int)(budget / per_w)));
    int QG = 1;
    if (WCH == nw && nq > 1) {
        QG = std::max(1, std::min(nq, (int)(budget / (nw * per_w + per_q))));
        if (const char *qg = std::getenv("LIBRPA_AMD_EC_QGROUP")) QG = std::max(1, std::min(QG, std::atoi(qg)));
    }
    const int UCH = QG > 1 ? QG * nw : WCH;  // (q, omega) matrices per pass
    DevBuf &dV = ec_V, &dL32 = ec_L32, &dD = ec_D, &dX = ec_X, &dM = ec_M, &dM64 = ec_M64, &dacc = ec_acc,
           &dVld = ec_Vld, &dS = ec_S;
    dV.reserve(nn * 8 * QG);
    dD.reserve(nn * es * UCH);
    dX.reserve(nn * es * UCH);
    dM.reserve(nn * es * UCH);
    dVld.reserve(sizeof(double) * QG);
    // pivot signs S of V = L S L^T: a Coulomb matrix that is not positive definite keeps
    // det(1 - V chi0) = det(S) det(S - L^T chi0 L) and Tr(V chi0) = n - sum_i S_i M_ii with
    // M = S - L^T chi0 L, so Ec is exact for any V (as the LU of epsilon.cpp:600-693 is)
    dS.reserve((size_t)n * 8 * QG);
    if (!f64) { dL32.reserve(nn * 4 * QG); dM64.reserve(nn * 8 * UCH); }
    const size_t acc_bytes = sizeof(double) * 2 * nq * nw + 64;
    dacc.reserve(acc_bytes);
    HIP_CHECK(hipMemsetAsync(dacc.get(), 0, acc_bytes, stream));
    int *dflag = reinterpret_cast<int *>(dacc.as<char>() + sizeof(double) * 2 * nq * nw);
    CholWork &cw = ec_cw;
    if (v_ibz != ibz) {
        // stage the input's V(q) blocks once per plan (the engine is rebuilt when inputs change)
        std::vector<VBlock> desc;
        std::vector<cplx> store;
        vdesc_q.assign(1, 0);
        for (int iq = 0; iq < nq; ++iq) {
            for (const auto &kv : ds.vq) {
                const int ik = std::get<0>(kv.first), I = std::get<1>(kv.first), J = std::get<2>(kv.first);
                if (ik != ibz[iq] || I > J) continue;
                if (kv.second.size() != (size_t)na[I] * na[J]) LRA_THROW("Coulomb block of the wrong size");
                desc.push_back({(long long)store.size(), (int)abf[I], (int)abf[J], na[I], na[J], I == J ? 1 : 0, iq});
                store.insert(store.end(), kv.second.begin(), kv.second.end());
            }
            vdesc_q.push_back((int)desc.size());
        }
        d_vblk = upload(store, stream);
        d_vdesc = upload(desc, stream);
        HIP_CHECK(hipStreamSynchronize(stream));
        v_ibz = ibz;
    }
    // (q per pass, omega per q, order, precision) -> (X = D L, M = S - L^T X) over the pass's
    // matrices u = qi * cnt + w, whose L is that of q qi; kept with their tuned tiles
    auto get_batches = [&](int qg, int cnt) -> std::pair<GemmBatch, GemmBatch> & {
        const auto key = std::make_tuple(qg, cnt, n, (int)ec_prec);
        auto it = ec_batches.find(key);
        if (it != ec_batches.end()) return it->second;
        auto &pr = ec_batches[key];
        GemmBatch &bx = pr.first, &bm = pr.second;
        bm.trans_a = true;
        bm.lower_only = true;
        for (int qi = 0; qi < qg; ++qi)
            for (int w = 0; w < cnt; ++w) {
                const long long u = ((long long)qi * cnt + w) * (long long)nn, l = (long long)qi * (long long)nn;
                // plane h of X = D L (no conjugate) and of M = L^H X
                for (int h = 0; h < (herm ? 2 : 1); ++h) {
                    GemmProb px = make_prob(n, n, n, u, n, l + h * plane, n, u + h * plane, n);
                    px.kmode = 1;  // L is lower triangular: column tile n0 needs k >= n0 only
                    GemmProb pm = make_prob(n, n, n, l, n, u + h * plane, n, u + h * plane, n);
                    pm.kmode = 2;  // A = L^T: row tile m0 needs k >= m0 only
                    if (herm) {
                        px.sgn2 = h ? 1 : -1;
                        px.a_off2 = u + plane;
                        px.b_off2 = l + (1 - h) * plane;
                        pm.sgn2 = h ? -1 : 1;
                        pm.a_off2 = l + plane;
                        pm.b_off2 = u + (1 - h) * plane;
                    }
                    bx.add(px);
                    bm.add(pm);
                }
            }
        const int cfg = n >= 1024 ? big_tile(ec_prec) : T64x64;
        bx.finalize(cfg, stream);
        bm.finalize(cfg, stream);
        // executed flops of the triangular products
        const double c = (herm ? 4.0 : 1.0) * qg * cnt * (double)n * n * n;
        bx.flops = c;
        bm.flops = c / 3.0;
        return pr;
    };
    for (int iq0 = 0; iq0 < nq; iq0 += QG) {
        const int qg = std::min(QG, nq - iq0);
        if (verbose) {
            HIP_CHECK(hipStreamSynchronize(stream));
            fprintf(stderr, "[librpa-mi355x] Ec: q %d-%d / %d (%.1f s)\n", iq0 + 1, iq0 + qg, nq, now_s() - t0);
            fflush(stderr);
        }
        // dense V(q) from the staged upper atom-pair blocks (Hermitian fill, utils_matrix_m_mpi.h:430-441)
        prof.begin("ec_v_fill", stream);
        HIP_CHECK(hipMemsetAsync(dV.get(), 0, (size_t)qg * nn * 8, stream));
        launch_v_scatter(d_vblk.as<double>(), d_vdesc.as<VBlock>() + vdesc_q[iq0], vdesc_q[iq0 + qg] - vdesc_q[iq0],
                         dV.as<double>(), n, lay, 0, iq0, (long long)nn, stream);
        prof.end("ec_v_fill", stream, 0, (double)qg * nn * 8);
        prof.begin("ec_chol_v", stream);
        cholesky_logdet_batched(dV.as<double>(), (long long)nn, qg, n, n, dVld.as<double>(), 1, dflag + 1, true, cw,
                                stream, -1, dS.as<double>(), n, herm ? plane : 0);
        prof.end("ec_chol_v", stream, (herm ? 4.0 : 1.0) * qg * n * n * n / 3.0);
        const void *Lp = dV.get();
        if (!f64) {
            launch_convert<double, float>(dV.as<double>(), dL32.as<float>(), (long long)qg * nn, stream);
            Lp = dL32.get();
        }
        const int cstep = qg > 1 ? nw : WCH;
        for (int w0 = 0; w0 < nw; w0 += cstep) {
            const int cnt = std::min(cstep, nw - w0);
            const int nu = qg * cnt;
            // tau -> omega (formed once above, or per chunk) and R -> q of chi0s into dense matrices
            prof.begin("chi0_transform", stream);
            std::vector<const double *> kfs(qg);
            for (int qi = 0; qi < qg; ++qi) kfs[qi] = &ds.kfrac[(size_t)ibz[iq0 + qi] * 3];
            assemble_dense_q(g, kfs, w0, cnt, dD.get(), f64, (long long)nn, lay, stream);
            const double tbytes = chiw_ok ? 8.0 * E_tot * cnt * ceil_div(qg, kChi0RqMaxQ) + (double)es * cnt * nn * qg
                                          : ((double)ts * E_tot * ntau_done * ceil_div(cnt, kChi0AssembleMaxW) +
                                             (double)es * cnt * nn) * qg;
            prof.end("chi0_transform", stream, 0, tbytes);
            auto &bb = get_batches(qg, cnt);
            if (autotune && !bb.first.tuned) {
                bb.first.tune(ec_prec, dD.get(), Lp, dX.get(), 1.0, 0.0, stream);
                gemm_run(ec_prec, bb.first, dD.get(), Lp, dX.get(), 1.0, 0.0, stream);
                bb.second.tune(ec_prec, Lp, dX.get(), dM.get(), -1.0, 0.0, stream);
            }
            prof.begin("ec_gemm_x", stream);
            gemm_run(ec_prec, bb.first, dD.get(), Lp, dX.get(), 1.0, 0.0, stream);
            prof.end("ec_gemm_x", stream, bb.first.flops);
            prof.begin("ec_gemm_m", stream);
            gemm_run(ec_prec, bb.second, Lp, dX.get(), dM.get(), -1.0, 0.0, stream);
            prof.end("ec_gemm_m", stream, bb.second.flops);
            double *M64 = dM.as<double>();
            if (!f64) {
                launch_copy_lower_f2d(dM.as<float>(), dM64.as<double>(), n, (long long)nu * (herm ? 2 : 1), plane, stream);
                M64 = dM64.as<double>();
            }
            // accumulators of (q, omega) at 2 (q nw + omega): the pass's matrices are consecutive
            // there (one q per pass, or all omega of each q)
            double *acc0 = dacc.as<double>() + 2 * ((size_t)iq0 * nw + w0);
            prof.begin("ec_logdet", stream);
            // S joins -L^H X here, in FP64 whatever the precision of the products
            launch_add_signs_trace(M64, n, nu, (long long)nn, dS.as<double>(), cnt, acc0, stream);
            cholesky_logdet_batched(M64, (long long)nn, nu, n, n, acc0 + 1, 2, dflag, false, cw, stream, -1, nullptr, 0,
                                    herm ? plane : 0);
            prof.end("ec_logdet", stream, (herm ? 4.0 : 1.0) * nu * n * n * n / 3.0);
        }
    }
    std::vector<double> hacc(2 * (size_t)nq * nw);
    int hflag[2] = {0, 0};
    HIP_CHECK(hipMemcpyAsync(hacc.data(), dacc.get(), hacc.size() * 8, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipMemcpyAsync(hflag, dflag, sizeof(hflag), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    if (hflag[1]) LRA_THROW("Coulomb matrix is singular or not finite (zero pivot in its factorisation)");
    if (hflag[0]) LRA_THROW("1 - V chi0 is singular or not finite at some (q, omega)");
    for (int iq = 0; iq < nq; ++iq)
        for (int iw = 0; iw < nw; ++iw) {
            const double tr = hacc[2 * ((size_t)iq * nw + iw)];
            const double ld = hacc[2 * ((size_t)iq * nw + iw) + 1];
            const double val = (n - tr) + ld;
            res.qcontrib[iq] += cplx(val * g.omega_w[iw] * wq[iq] / (2 * M_PI), 0.0);
        }
    for (auto &c : res.qcontrib) res.ec_re += c.real();
    // a host-staged system needs the device memory back for the next chi0 build
    if (host_staged) release_ec();
    t_ec = now_s() - t0;
    return res;
}

bool RpaEngine::form_chiw(const TFGrid &g, double max_bytes, hipStream_t s) {
    chiw_ok = false;
    const double need = 8.0 * (double)E_tot * g.n;
    // a store kept from an earlier evaluation is reused (its bytes are not in the free memory)
    if (ntau_done != g.n || g.n > kTauOmegaMax || need > max_bytes + (double)d_chiw.bytes()) return false;
    d_chiw.reserve((size_t)need);
    std::vector<double> coef((size_t)g.n * g.n);
    for (int w = 0; w < g.n; ++w)
        for (int t = 0; t < g.n; ++t) coef[(size_t)w * g.n + t] = g.cos_t2f[(size_t)w * g.n + t] * 2.0 / nspin;
    if (host_staged) {
        DevBuf dc = upload(coef, s);
        // slices back through the one-slice device buffer, accumulated tau by tau
        for (int t = 0; t < ntau_done; ++t) {
            HIP_CHECK(hipMemcpyAsync(d_chi0s.get(), h_chi0s[t].data(), ts * (size_t)E_tot, hipMemcpyHostToDevice, s));
            if (prec == Prec::F64)
                launch_tau_accumulate(d_chi0s.as<double>(), E_tot, t, ntau_done, dc.as<double>(), g.n,
                                      d_chiw.as<double>(), s);
            else
                launch_tau_accumulate(d_chi0s.as<float>(), E_tot, t, ntau_done, dc.as<double>(), g.n,
                                      d_chiw.as<double>(), s);
        }
        HIP_CHECK(hipStreamSynchronize(s));
        chiw_ok = true;
        return true;
    }
    if (prec == Prec::F64)
        launch_tau_to_omega(d_chi0s.as<double>(), E_tot, ntau_done, coef, d_table, g.n, d_chiw.as<double>(), s);
    else
        launch_tau_to_omega(d_chi0s.as<float>(), E_tot, ntau_done, coef, d_table, g.n, d_chiw.as<double>(), s);
    chiw_ok = true;
    return true;
}

void RpaEngine::assemble_dense_q(const TFGrid &g, const std::vector<const double *> &kfs, int w0, int cnt,
                                 void *dense, bool f64, long long nn, DenseLayout lay, hipStream_t s) {
    const size_t es = f64 ? 8 : 4;
    if (!chiw_ok) {
        for (size_t qi = 0; qi < kfs.size(); ++qi)
            assemble_dense(g, kfs[qi], w0, cnt, static_cast<char *>(dense) + qi * cnt * nn * es, f64, nn, lay, s);
        return;
    }
    const int n = NABF;
    for (size_t q0 = 0; q0 < kfs.size(); q0 += kChi0RqMaxQ) {
        const int nq = (int)std::min<size_t>(kChi0RqMaxQ, kfs.size() - q0);
        std::vector<double> ph((size_t)nq * nR * 2);
        for (int qi = 0; qi < nq; ++qi) {
            const double *kf = kfs[q0 + qi];
            for (int r = 0; r < nR; ++r) {
                const double ang = 2 * M_PI * (kf[0] * cells[r][0] + kf[1] * cells[r][1] + kf[2] * cells[r][2]);
                ph[((size_t)qi * nR + r) * 2] = std::cos(ang);
                ph[((size_t)qi * nR + r) * 2 + 1] = std::sin(ang);
            }
        }
        const double *cw = d_chiw.as<double>() + (size_t)w0 * E_tot;
        char *Dd = static_cast<char *>(dense) + q0 * cnt * nn * es;
        if (f64)
            launch_chi0_rq_multi<double>(cw, E_tot, d_pairs.as<PairDesc>(), (int)pairs.size(), n_pair_elems,
                                         d_pair_eoff.as<long long>(), nR, ph, d_table, nq, cnt, (double *)Dd, nn,
                                         (long long)cnt * nn, n, lay, s);
        else
            launch_chi0_rq_multi<float>(cw, E_tot, d_pairs.as<PairDesc>(), (int)pairs.size(), n_pair_elems,
                                        d_pair_eoff.as<long long>(), nR, ph, d_table, nq, cnt, (float *)Dd, nn,
                                        (long long)cnt * nn, n, lay, s);
    }
}

void RpaEngine::assemble_dense(const TFGrid &g, const double *kf, int w0, int cnt, void *dense, bool f64, long long nn,
                               DenseLayout lay, hipStream_t s) {
    if (chiw_ok) {
        assemble_dense_q(g, {kf}, w0, cnt, dense, f64, nn, lay, s);
        return;
    }
    const int n = NABF;
    std::vector<double> ph((size_t)nR * 2);
    for (int r = 0; r < nR; ++r) {
        const double ang = 2 * M_PI * (kf[0] * cells[r][0] + kf[1] * cells[r][1] + kf[2] * cells[r][2]);
        ph[2 * r] = std::cos(ang);
        ph[2 * r + 1] = std::sin(ang);
    }
    const size_t es = f64 ? 8 : 4;
    for (int a0 = 0; a0 < cnt; a0 += kChi0AssembleMaxW) {
        const int cw_n = std::min(kChi0AssembleMaxW, cnt - a0);
        std::vector<double> gp((size_t)cw_n * nR * ntau_done * 2, 0.0);
        for (int w = 0; w < cw_n; ++w)
            for (int r = 0; r < nR; ++r)
                for (int t = 0; t < ntau_done; ++t) {
                    const double gam = g.cos_t2f[(size_t)(w0 + a0 + w) * g.n + t] * 2.0 / nspin;
                    gp[(((size_t)w * nR + r) * ntau_done + t) * 2] = gam * ph[2 * r];
                    gp[(((size_t)w * nR + r) * ntau_done + t) * 2 + 1] = gam * ph[2 * r + 1];
                }
        DevBuf dgp = upload(gp, s);
        char *Dd = static_cast<char *>(dense) + (size_t)a0 * nn * es;
        if (prec == Prec::F64 && f64)
            launch_chi0_assemble<double, double>(d_chi0s.as<double>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                                 (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                                 dgp.as<double>(), cw_n, (double *)Dd, nn, n, lay, s);
        else if (prec == Prec::F64)
            launch_chi0_assemble<double, float>(d_chi0s.as<double>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                                (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                                dgp.as<double>(), cw_n, (float *)Dd, nn, n, lay, s);
        else if (f64)
            launch_chi0_assemble<float, double>(d_chi0s.as<float>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                                (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                                dgp.as<double>(), cw_n, (double *)Dd, nn, n, lay, s);
        else
            launch_chi0_assemble<float, float>(d_chi0s.as<float>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                               (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                               dgp.as<double>(), cw_n, (float *)Dd, nn, n, lay, s);
        HIP_CHECK(hipStreamSynchronize(s));  // dgp is freed on return
    }
}

double RpaEngine::ec_bytes() const {
    double held = 0;
    for (const DevBuf *b : {&ec_V, &ec_L32, &ec_D, &ec_X, &ec_M, &ec_M64, &ec_S, &ec_Vld, &ec_acc, &ec_cw.linv,
                            &ec_cw.panel})
        held += (double)b->bytes();
    return held;
}

void RpaEngine::release_ec() {
    for (DevBuf *b : {&ec_V, &ec_L32, &ec_D, &ec_X, &ec_M, &ec_M64, &ec_S, &ec_Vld, &ec_acc, &ec_cw.linv, &ec_cw.panel})
        b->release();
}

void RpaEngine::release_work() {
    d_Ghat.release();
    d_W.release();
}

void RpaEngine::release_stores() {
    release_work();
    release_ec();
    for (DevBuf *b : {&d_chi0s, &d_chiw, &d_Cfin, &d_CWb, &d_Cfin32, &d_CWb32, &d_ZZ, &d_Zs, &d_Mst, &d_Gpm, &d_wre, &d_wim, &d_vblk})
        b->release();
    free_host_store();
    ntau_done = 0;
    chiw_ok = false;
}

void RpaEngine::free_host_store() {
    h_chi0s.clear();
    h_chi0s.shrink_to_fit();
}

RpaEngine::~RpaEngine() {
    hold();
    free_host_store();
}

void RpaEngine::chi0s_block(int it, int I, int J, int r, double *out) {
    for (const auto &o : outs)
        if (o.I == I && o.J == J && o.r == r) {
            const size_t n = (size_t)na[I] * na[J];
            const size_t off = (size_t)it * E_tot + o.eoff;
            if (host_staged) {
                if (it < 0 || it >= (int)h_chi0s.size()) LRA_THROW("tau index out of range");
                if (prec == Prec::F64) {
                    std::memcpy(out, reinterpret_cast<const double *>(h_chi0s[it].data()) + o.eoff, n * 8);
                } else {
                    const float *src = reinterpret_cast<const float *>(h_chi0s[it].data()) + o.eoff;
                    for (size_t i = 0; i < n; ++i) out[i] = src[i];
                }
                return;
            }
            if (prec == Prec::F64) {
                HIP_CHECK(hipMemcpy(out, d_chi0s.as<double>() + off, n * 8, hipMemcpyDeviceToHost));
            } else {
                std::vector<float> tmp(n);
                HIP_CHECK(hipMemcpy(tmp.data(), d_chi0s.as<float>() + off, n * 4, hipMemcpyDeviceToHost));
                for (size_t i = 0; i < n; ++i) out[i] = tmp[i];
            }
            return;
        }
    LRA_THROW("chi0s block not found");
}

void RpaEngine::chi0q_block(const Dataset &ds, const TFGrid &g, int iw, int iq, int I, int J, double *re,
                            double *im) {
    if (host_staged) LRA_THROW("chi0(q, omega) blocks are not kept with the host-staged chi0 store");
    const bool herm = nk > 1;
    const DenseLayout lay = herm ? kPlanar : kReal;
    const int n = NABF;
    const size_t nn = (size_t)n * n * (herm ? 2 : 1);
    DevBuf dD(nn * 8);
    std::vector<double> gp((size_t)nR * ntau_done * 2);
    const double *kf = &ds.kfrac[(size_t)iq * 3];
    for (int r = 0; r < nR; ++r) {
        const double ang = 2 * M_PI * (kf[0] * cells[r][0] + kf[1] * cells[r][1] + kf[2] * cells[r][2]);
        for (int t = 0; t < ntau_done; ++t) {
            const double gam = g.cos_t2f[(size_t)iw * g.n + t] * 2.0 / nspin;
            gp[((size_t)r * ntau_done + t) * 2] = gam * std::cos(ang);
            gp[((size_t)r * ntau_done + t) * 2 + 1] = gam * std::sin(ang);
        }
    }
    DevBuf dgp = upload(gp, stream);
    if (prec == Prec::F64)
        launch_chi0_assemble<double, double>(d_chi0s.as<double>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                             (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                             dgp.as<double>(), 1, dD.as<double>(), 0, n, lay, stream);
    else
        launch_chi0_assemble<float, double>(d_chi0s.as<float>(), E_tot, ntau_done, d_pairs.as<PairDesc>(),
                                            (int)pairs.size(), n_pair_elems, d_pair_eoff.as<long long>(), nR,
                                            dgp.as<double>(), 1, dD.as<double>(), 0, n, lay, stream);
    std::vector<double> h(nn);
    HIP_CHECK(hipMemcpyAsync(h.data(), dD.get(), h.size() * 8, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    for (int mu = 0; mu < na[I]; ++mu)
        for (int nu = 0; nu < na[J]; ++nu) {
            const size_t r = abf[I] + mu, c = abf[J] + nu;
            re[(size_t)mu * na[J] + nu] = h[r * n + c];
            im[(size_t)mu * na[J] + nu] = herm ? h[(n + r) * n + c] : 0.0;
        }
}

}  // namespace lra
