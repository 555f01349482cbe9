// G0W0: screened interaction W(q, i omega) -> W(R, i tau) and the correlation
// self-energy Sigma(R, i tau) = C G W C contraction on top of the chi0 engine.
#pragma once

#include <cstdio>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/librpa_options.h"
#include "dataset.h"
#include "gemm.h"
#include "gw_kernels.h"
#include "kernels.h"
#include "rpa.h"

namespace lra {

// The upper atom-pair blocks (I <= J) of a Coulomb input for a list of k points, on the device for
// launch_v_scatter (VBlock::q: position in the list), with the largest |V| and |Im V| of each.
struct CoulombStage {
    DevBuf blk, desc;
    std::vector<int> first;  // descriptors of point i: [first[i], first[i + 1])
    std::vector<double> vmax, imax;
};

// consecutive 256-byte aligned pieces of a buffer (a null base counts the bytes)
struct Carve {
    char *base;
    size_t at = 0;
    template <class T> T *take(size_t n) {
        T *p = reinterpret_cast<T *>(base + at);
        at += (n * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

struct GwEngine : KeptMemory {
    void give_back() override { work.release(); }
    ~GwEngine() override { hold(); }
    std::shared_ptr<RpaEngine> rpa;  // geometry, G(R, +-tau) builder, chi0(R, tau)
    Prec prec = Prec::F64;
    size_t ts = 8;
    int natom = 0, NAO = 0, NABF = 0, nR = 0, nk = 0, nspin = 1, ntau = 0;
    long long LD = 0;  // nR * NAO: column count of the (cell, atom, orbital) index

    // cell differences R1 - R2 of two BvK cells on an extended (2p - 1)^3 grid
    int E[3] = {1, 1, 1};
    int NE = 1;
    long long c0 = 0;
    long long linr(int x, int y, int z) const { return ((long long)x * E[1] + y) * E[2] + z; }

    int nbatch = 1;  // tau points per pass
    int signs = 2;   // signs of tau per pass: U and Y of both are held, or of one at a time when two do not fit

    // U_J(S) build
    struct UChunk {
        int sg = -1;  // its sign of tau (0: +, 1: -), -1: both
        long long ghat_elems = 0;
        int max_gcol = 0;
        std::vector<GatherJob> jobs;
        std::vector<long long> colsrc;
        DevBuf d_jobs, d_colsrc;
        GemmBatch ub;
    };
    std::vector<UChunk> uchunks;
    std::vector<long long> u_off;  // per (J, S)
    long long u_elems = 0;

    // CW of the atoms [x0, x1) and the contractions that read it
    struct Tasks { int a = 1, b = 1, n = 0; DevBuf d; };  // fragments of a task
    struct XChunk {
        int x0 = 0, x1 = 0;
        long long cw_elems = 0;
        GemmBatch cwb;
        DevBuf d_blks;
        std::vector<Tasks> d, b;
    };
    std::vector<XChunk> xchunks;
    std::vector<Tasks> ytasks;
    DevBuf d_yent;
    GemmBatch a3;
    std::vector<long long> y_off;
    long long y_elems = 0;

    DevBuf d_fold, d_neg;
    // Work memory of W and of Sigma, one after the other in the same bytes.  Kept for the next build up to
    // keep_bytes (allocating and freeing 3 GB took 30 of the 86 ms of a build on 8 atoms and 4 k), as are
    // the chi0 build's buffers and the Cholesky workspace beside it; larger systems give each of them back
    // after every build, finished or failed.
    DevBuf work;
    static double keep_bytes();  // 12 GB, or LIBRPA_AMD_KEEP_BYTES
    struct SigmaWork { char *U, *Ghat, *CW, *Y, *sigma, *Wlow; };  // sigma: sig, s2 and ext of each tau and sign
    void sigma_layout(Carve &c, SigmaWork &w) const;
    CoulombStage vst, vcst;          // the Coulomb inputs of the q in v_qs
    std::vector<int> v_qs;
    bool same_cut = false;           // v_c = v
    // What a build leaves for the getters; replaced when the next one is complete.
    struct Result {
        DevBuf Wrt;       // W(R, tau) [tau][R][NABF][NABF], FP64
        DevBuf Sre, Sim;  // Sigma(R, i omega) [spin][omega][R][NAO][NAO], FP64
        bool w_zero = false;  // no truncated Coulomb given: W = 0
    };
    std::shared_ptr<Result> res;
    mutable std::mutex ks_mu;  // ks_diag's buffers
    DevBuf ks_in, ks_out;

    double flops_sigma = 0, flops_w = 0, t_w = 0, t_sigma = 0;
    long long max_ghat = 0, max_cw = 0;
    bool verbose = false;  // progress lines on stderr
    // eps_mac(i omega_w) per grid frequency: replaces the head of the dielectric matrix at q = 0
    // (replace_w_head with option_dielect_func 0); empty = no replacement
    std::vector<double> head;
    double sqrt_threshold = 0.0;  // sqrt_coulomb_threshold: eigenvalues of v, v_c below it are dropped

    void plan(const Dataset &ds, std::shared_ptr<RpaEngine> r);
    void build_w(const Dataset &ds, const TFGrid &g, Result &out);
    void build_sigma(const Dataset &ds, const TFGrid &g, Result &out);
    void w_block(int it, int I, int J, int r, double *out) const;
    void sigma_block(int spin, int iw, int I, int J, int r, double *re, double *im) const;
    // Sigma_KS(k, i omega)_nn for the given states: [state][omega]
    std::vector<std::vector<cplx>> ks_diag(const Dataset &ds, int spin, int ik, const std::vector<int> &states);
};

// the minimax / time-frequency grid of the current inputs (api.cpp)
void lra_prepare_grid(Dataset &d, const LibrpaOptions &o);

void gw_build_sigma(Dataset &d, const LibrpaOptions &o);
void gw_sigc_kgrid(Dataset &d, const LibrpaOptions &o, int n_spins, int n_kpts_this, const int *iks_this,
                   int i_state_low, int i_state_high, const double *vxc, const double *vexx, double *sigc_re,
                   double *sigc_im);

// Thiele continued-fraction analytic continuation (src/core/analycont.cpp:17-80)
struct PadeAC {
    int n = 0;
    std::vector<cplx> x, y;
    PadeAC(int n_pars, const std::vector<cplx> &xs, const std::vector<cplx> &data);
    cplx operator()(cplx z) const;
};
// Damped fixed-point QP solver (src/core/qpe_solver.cpp:10-55); returns 0 on success
int qpe_solve(const PadeAC &p, double e_mf, double e_fermi, double vxc, double sigx, double &e_qp, cplx &sigc,
              double diff_init = 1e-3, double thres = 1e-5, int n_iter_max = 200);

}  // namespace lra
