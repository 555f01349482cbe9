// Streaming kernels of the G0W0 path (gfx950): W(q, omega) -> W(R, tau) accumulation,
// folding of the self-energy cell images, the tau -> omega fold and the Kohn-Sham
// projection of Sigma(R, i omega).
#pragma once

#include "chi0.h"
#include "common.h"

namespace lra {

// Dense n x n matrices below are real, or Hermitian in two planes (Re, Im) of n x n (pl = 2, im > 0).

// W(R, tau)[a][b] += sum_(q, w) coef[q][w][tau] (ph_qR.x Re W_qw(a, b) + ph_qR.y Im W_qw(a, b)) for all R
// and tau, W_qw = -(trailing block of the partially factorised augmented matrix q * nw + w), that block
// starting at (n, n) of a 2n x 2n matrix (lower triangle valid), matrices stride apart and the
// imaginary plane im after the real one (0: none).  ph [q][R] (cos, sin); Wrt layout: [tau][R][n][n].
void launch_w_accum(const double *aug, long long stride, long long im, int nq, int nw, int n, const double *coef,
                    int ntau, const double *ph, int nR, double *Wrt, hipStream_t s);
// lower triangle of every augmented matrix: [[I, .], [C_q, V_q]]
void launch_fill_aug(double *A, long long stride, long long im, int nq, int nw, int n, const double *C, const double *V,
                     hipStream_t s);

// ---- self-energy contractions (gw.cpp) ----
// CW_IJ(R)[c][i][nu] = sum_mu C^I[(c, i)][mu] W_IJ(R)[mu][nu] and U_J(S)[(X, x)][j][nu] per tau point; c
// runs over the rows (K, R1, k) of atom I's neighbours (Chi0Seg order: (cell, row) of R - R1).
// One (I, J, R).
struct SigBlk {
    long long cw, u;  // CW_IJ(R), U_J(cell 0) (cells NAO nj aj apart)
    int ni, nj, aj, l;
    int rowI, colJ, r;
    int seg0;         // first entry of (I, R) in the segment table
};
// segments [c0, c1) of a block, rows from i0 (or all), columns from j0
struct SigTask { int blk, i0, j0, c0, c1; };
// For nsg signs of tau (2, or 1 at a time: sig, s2 start at that sign then, U and Y hold it alone):
// sig[z][sign][R][NAO][NAO] += D, the label a0b0_a2b2: CW zcw elements per tau point, U's signs usg apart
template <class T>
void launch_sigma_d(const SigTask *tasks, int ntask, int fi, int fj, const SigBlk *blks, const Chi0Seg *segs, const T *CW,
                    long long zcw, const T *U, long long usg, T *sig, long long ssg, int NAO, int nz, int nsg, hipStream_t s);
// s2[z][sign][R][NAO][NAO] += the label a0b0_a1b2, 64 fc segments a task from c0
template <class T>
void launch_sigma_b(const SigTask *tasks, int ntask, int fc, int fj, const SigBlk *blks, const Chi0Seg *segs, const T *CW,
                    long long zcw, const T *U, long long usg, T *s2, long long ssg, int NAO, int nz, int nsg, hipStream_t s);
// One (J, R) that reaches the columns (S, L, .): G_IJ(R) at g, CW_JI(-R)[(L, S - R, l)] at
// b + abf(I) lb + (cb + l nj) ai
struct SigYEnt { long long g, b; int lb, cb, nj, J; };
struct SigYTask {
    long long y;  // Y_I row of (S, L, 0)
    int e0, e1;   // entries of (S, L)
    int ni, ai, ao, abf, l0, nl, mu0, i0;
};
template <class T>
void launch_sigma_y(const SigYTask *tasks, int ntask, int fi, const SigYEnt *ents, const T *CW, long long zcw, const T *G,
                    long long zg, T *Y, long long ysg, int NAO, int x0, int x1, bool first, int nz, int nsg, int sg0, hipStream_t s);

// for nz tau points and both signs: sig[R][a][b] += s2[R][a][b] + s2[-R][b][a] + sum_{e : fold[e] == R} ext[e][a][b]
template <class T>
void launch_sigma_fold(T *sig, const T *s2, const T *ext, const int *fold, const int *neg, int NE, int nR, int n,
                       int nz, hipStream_t s);

// Sigma(R, i w) += 0.5 (S+ + S-) cos_t2f(w) + i 0.5 (S+ - S-) sin_t2f(w) for all w and the tau points
// [it0, it0 + nz) (sig [z][sign][nelem], cw / sw [w][ntau], sre / sim [w][nelem]).
template <class T>
void launch_sigma_freq(const T *sig, long long nelem, const double *cw, const double *sw, int nw, int ntau, int it0,
                       int nz, double *sre, double *sim, hipStream_t s);

// Y[w][a][st] = sum_b sum_R ph[(I(a), J(b), R)] Sigma(R, w)[a][b] U[st][b] for one k point
// (complex, st < nst <= 16); ph layout [I][J][R] (re, im interleaved), U [st][b] (re, im).
void launch_sigma_ks_rows(const double *sre, const double *sim, int nw, int nR, int n, const int *atom_of,
                          int natom, const double *ph, const double *U, int nst, double *Y, hipStream_t s);

// Newton-Schulz square roots of the matrices A + sel[m] * nn, m < nmat (nn = pl n^2 elements each), on
// compact work arrays Y, Z: Y = A / c, Z = I with c = ||A||_F in scale (part: 32 doubles a matrix) ...
void launch_ns_init(const double *A, const int *sel, int nmat, int n, int pl, double *part, double *Y, double *Z,
                    double *scale, hipStream_t s);
// ... P <- 1.5 I - 0.5 P ...
void launch_ns_step(double *P, int nmat, int n, int pl, hipStream_t s);
// ... out[2 m], out[2 m + 1] = max |Yn - Y|, max |Y| (bits of doubles, cleared by the caller) ...
void launch_ns_change(const double *Yn, const double *Y, int nmat, int n, int pl, unsigned long long *out, hipStream_t s);
// ... and A + sel[m] * nn = sqrt(c) Y
void launch_ns_finish(const double *Y, const double *scale, const int *sel, int nmat, int n, int pl, double *A,
                      hipStream_t s);
// A[i][:] *= f[i] (row-major n x n)
void launch_scale_rows(double *A, int n, const double *f, hipStream_t s);

// Head of the dielectric matrix at q = 0 (replace_w_head): for each of cnt matrices eps_w (lower
// triangle valid, rows of length ld, stride apart), q[w] = u^T eps_w u over the n x n block at the
// origin (q is accumulated, clear it first) ...
void launch_head_quad(const double *A, long long stride, int ld, int n, int cnt, const double *u, double *q,
                      hipStream_t s);
// ... then eps_w += (eps_mac[w] - q[w]) u u^T on the lower triangle of that block.
void launch_head_update(double *A, long long stride, int ld, int n, int cnt, const double *u, const double *eps_mac,
                        const double *q, hipStream_t s);

}  // namespace lra
