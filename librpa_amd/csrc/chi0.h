// The chi0(R, tau) contraction: every output block straight from G, W and Cs, one launch per
// tile class.
#pragma once

#include <vector>

#include "common.h"
#include "gemm.h"

namespace lra {

// One output block chi0s(I, J, R).
struct Chi0Out {
    long long cfin;    // Cfin_I [(K, R1, k, i)][mu]
    long long gpm;     // G_IJ(R) in Gpm: element (i, q) at gpm + i * 2 NAO + q, q = (s, j)
    long long wseg;    // W(., J, cell 0); cell S at + S * NAO * 2 nj * aj
    long long xa, xb;  // W(I, -R) rows of J and W(J, R) rows of I (the direct term's operands)
    long long eoff;    // chi0s block, row-major ai x aj
    int ni, nj, ai, aj;
    int I, J, r;
    int lsum;          // segments: rows (K, R1, k) of atom I
    int segtab;        // first entry of (I, R) in the segment table
};
// Segment t of (I, R): W(K, J, R - R1) row k is at wseg + (cell * NAO + row) * 2 nj * aj, its rows
// of Cfin_I start at c * ni.  In the order of (cell, row): the outputs of one R then walk through
// the rows of W and of Cs in step, whatever their I and J.
struct Chi0Seg { int cell, row, c, pad; };
// One workgroup: ns column strips x kp parts of the segments [t0, t1) of output out; segments
// from lsum on are the 2 nj (s', j) terms of the direct contraction.
struct Chi0Task { int out, m0, n0, ns, kp, t0, t1, part; };

// The task lists of one element type (FP64 or FP32), by tile class.
struct Chi0Tasks {
    struct Class {
        int fm, fn, fi, nq;  // row fragments of mu, columns of a lane, fragments of i per pass, unrolled W steps
        std::vector<Chi0Task> tasks;
        int qs = 0;  // LDS steps of the G operand
        DevBuf d_tasks;
    };
    std::vector<Class> classes;
    // nz: tau points per launch; splitk: 0 = by load, 1 = one part per output (no atomic adds: the
    // same bits every run), n = n parts
    void build(const std::vector<Chi0Out> &outs, bool f64, int nz, int splitk, hipStream_t s);
    bool single = false;
};

// chi += contraction for nz tau points (slices zg, zw, zc elements apart).  T is the element type
// of G, W and Cs, TO that of chi.  skip (optional): nz x nout flags of outputs to leave out.
template <class T, class TO>
void launch_chi0_contract(const Chi0Tasks &tk, const Chi0Out *outs, int nout, const Chi0Seg *segs, const T *Gpm,
                          long long zg, const T *W, long long zw, const T *Cfin, TO *chi, long long zc, int NAO,
                          int nz, const unsigned char *skip, hipStream_t s);

// Elements that W and Cfin hold past their last one: a lane's 16-byte load may start at the last
// element of a row.
constexpr int kChi0Pad = 16;

}  // namespace lra
