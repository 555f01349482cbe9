// chi0(R, tau) contraction kernel (gfx950).
//
// An output block sums over the rows (K, R1, k) of atom I ("segments"):
//   chi0s(I,J,R)[mu][nu] += sum_i C^I(K,R1)[mu][(k, i)] T[i][nu],
//   T[i][nu] = sum_(s, j) G^s_IJ(R)[i][(s, j)] W(K,J,R-R1)[(s, j)][k][nu],
// and the direct term sum_(s', j, i) W(I,-R)[(1-s', i)][(J, j)][mu] W(J,R)[(s', j)][(I, i)][nu].
// T is never stored: one wave forms a 16 x 16 fragment of it with MFMA and feeds the accumulator
// registers to the next MFMA as its B operand.  Both the FP64 and the FP32 16x16x4 results hold,
// in register r of lane group kq, one row of the four that step r of the second product contracts
// over (FP64: row 4r + kq; FP32: row 4kq + r, turned into 4r + kq by permuting the rows of G when
// they are staged), so no value crosses a lane.
//
// A wave owns a strip of 16 FN columns over FM row fragments and reads W and Cs straight into
// registers, 16 bytes a lane: an MFMA of these types takes 64 (FP64) or 32 (FP32) cycles for 512
// (256) bytes of operand, so there is nothing to gain from staging them in LDS, and no barrier in
// the loop; only G_IJ, which every segment reuses, is in LDS.  An operand register is loaded again
// as soon as the MFMAs that read it are issued, so a load has 1 to 4 thousand cycles of MFMA to
// arrive.  Measured against the two GEMMs with T between them (38 GB of it per tau point on a
// 64-atom cell), X and T_A and contraction together: 526 -> 411 ms on 64 atoms at Gamma (46 TF/s of
// the sums' own flops; 60- and 120-row blocks and 13- and 27-row T fragments pad the rest), 52 -> 32.7 ms
// on 16 atoms and 8 k (47 TF/s).  On 128 atoms (46 TF/s FP64, 121 ms a tau point) the operands come through
// the L2 at 3.9 TB/s (FP64) and 5.0 TB/s (FP32, 61 ms): FP32 is bound by that, FP64 nearly.
#include "chi0.h"

#include <algorithm>
#include <map>
#include <tuple>
#include <type_traits>

namespace lra {

namespace {
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
// 16-byte buffer loads need dword alignment only (rows of odd basis sizes)
typedef double d2u __attribute__((ext_vector_type(2)));
typedef float f4u __attribute__((ext_vector_type(4)));

typedef double d1u __attribute__((ext_vector_type(1)));
typedef float f2u __attribute__((ext_vector_type(2)));
template <class T> struct CT;  // V: VL values, a 16-byte load; Cols: FN values, that or half of it
template <> struct CT<double> { using V = d2u; using A = v4d; static constexpr int VL = 2; template <int N> using Cols = std::conditional_t<N == 2, d2u, d1u>; };
template <> struct CT<float> { using V = f4u; using A = v4f; static constexpr int VL = 4; template <int N> using Cols = std::conditional_t<N == 4, f4u, f2u>; };

__device__ __forceinline__ v4d mfma(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// One wave a SIMD with long rings, or two with short ones: two hide the instructions between the MFMAs
// (FP32, 120-row blocks of 27-row fragments: 18.7 -> 17.0 ms a 32-atom build) as long as the accumulators
// leave registers for them; 128 + 32 FP64 ones do not (38 spilled: 205 -> 258 ms on 64 atoms), nor do the
// FP64 strips of more than 128 rows (160 or more accumulator registers).
template <class T> constexpr bool one_wave(int fm, int fi) { return sizeof(T) == 8 && (fm > 8 || fm * fi >= 16); }

// An FP32 accumulator takes at most this many steps (of four products) before it is added to chi.  Diagonal
// blocks of the 128-atom cell against FP64: off by 1.28e-6 of their norm (rms) with a segment list in two to
// four accumulators (up to 6400 steps each), by 0.77e-6 with this limit, and the launches 5% shorter (977 ->
// 931 ms for 16 tau points).  The GEMMs over a stored T that took quarters of the list were off by 0.86e-6.
constexpr double kMaxStepsF32 = 1600;

// row fragments of a strip with VL columns a lane at most
constexpr int most_whole(bool f64) { return f64 ? 12 : 8; }

constexpr int kQsMax = 96;  // G steps of a fragment of i kept in LDS (n_b(J) <= 192)

// 16 or 8 bytes at base + o: base in scalar registers, o one vector register (a 64-bit lane address per step
// and fragment, worked out ahead of the loop, took 64 registers and two moves per load)
template <class V, class T> __device__ __forceinline__ V load_at(const T *b, unsigned o) {
    const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(b), 0, -1, 0x00027000);
    if constexpr (sizeof(V) == 16) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
    else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0));
}

// G_IJ rows [i0, i0 + 16 FI) as A fragments: step s of fragment f at P[(f qsl + s) 64 + lane], zero past
// n_b(I) and 2 n_b(J)
template <class T>
__device__ __forceinline__ T g_element(const T *g, int i0, int f, int s, int lane, int ni, int qn, int NAO) {
    const int rho = lane & 15, i = i0 + f * 16 + (sizeof(T) == 8 ? rho : 4 * (rho & 3) + (rho >> 2)), q = 4 * s + (lane >> 4);
    return (i < ni && q < qn) ? g[(long long)i * 2 * NAO + q] : T(0);
}

// chi += the accumulators of a wave: rows from m0 (fragments of VL interleaved ones), 16 FN columns from n0
template <class T, class TO, int FM, int FN, class A>
__device__ __forceinline__ void add_to_chi(TO *chi, const Chi0Out &O, int m0, int n0, int c, int kq, const A (&acc)[FM][FN],
                                           int single) {
    constexpr int VL = CT<T>::VL;
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int rho = sizeof(T) == 8 ? 4 * r + kq : 4 * kq + r;
            const int mu = m0 + ((a / VL) * 16 + rho) * VL + a % VL;
            if (mu >= O.ai) continue;
            TO *dst = chi + O.eoff + (long long)mu * O.aj + n0 + c * FN;
#pragma unroll
            for (int b = 0; b < FN; ++b) {
                if (n0 + c * FN + b >= O.aj) continue;
                if (single) dst[b] += static_cast<TO>(acc[a][b][r]);
                else unsafeAtomicAdd(dst + b, static_cast<TO>(acc[a][b][r]));
            }
        }
}

// the direct term of a wave's strip: segment lsum + (s', j) contracts over i, segments [x0, x1) of it
template <class T, int FM, int FN, int RC, class A>
__device__ __forceinline__ void direct_term(const Chi0Out &O, const T *W, int x0, int x1, int kq, const unsigned (&mul)[FM / CT<T>::VL],
                                            unsigned nul, A (&acc)[FM][FN]) {
    using V = typename CT<T>::V;
    using Q = typename CT<T>::template Cols<FN>;
    constexpr int VL = CT<T>::VL, G = FM / VL;
    constexpr unsigned TS = sizeof(T);
    const int ni = O.ni, ai = O.ai, aj = O.aj, qn = 2 * O.nj;
    const unsigned ao_ = kq * ai * TS, aol = min(kq, (ni - 1) & 3) * ai * TS;
    const unsigned bo = kq * qn * aj * TS + nul, bol = min(kq, (ni - 1) & 3) * qn * aj * TS + nul;
    const int nic = (ni + 4 * RC - 1) / (4 * RC), nu = max(0, (x1 - x0) * nic);
    if (nu == 0) return;
    V ar[RC][G];
    Q br[RC];
    // step s of the u-th (s', j), i block
    const auto load = [&](int u, int s) {
        const int x = x0 + u / nic, i0 = (u % nic) * 4 * RC;
        const int sp = x >= O.nj ? 1 : 0, j = x - sp * O.nj;
        const int is = min(i0 + 4 * s, (ni - 1) & ~3);
        const bool last = is + 4 >= ni;
        const T *ab = W + O.xa + ((long long)j * 2 * ni + (1 - sp) * ni + is) * ai;
        const T *bb = W + O.xb + ((long long)is * qn + sp * O.nj + j) * aj;
#pragma unroll
        for (int g = 0; g < G; ++g) ar[s][g] = load_at<V>(ab, (last ? aol : ao_) + mul[g]);
        br[s] = load_at<Q>(bb, last ? bol : bo);
        if (i0 + 4 * s + kq >= ni)
#pragma unroll
            for (int b = 0; b < FN; ++b) br[s][b] = T(0);
    };
#pragma unroll
    for (int s = 0; s < RC; ++s) load(0, s);
    for (int u = 0; u < nu; ++u) {
        const int un = min(u + 1, nu - 1);
#pragma unroll
        for (int s = 0; s < RC; ++s) {
            if ((u % nic) * 4 * RC + 4 * s < ni)
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int e = 0; e < VL; ++e)
#pragma unroll
                        for (int b = 0; b < FN; ++b)
                            acc[g * VL + e][b] = mfma(ar[s][g][e], br[s][b], acc[g * VL + e][b]);
            load(un, s);
        }
    }
}
}  // namespace

// NQ: steps of W of a segment, unrolled (n_b(J) <= 2 NQ); NQ = 0: up to kQsMax, in a loop over groups of RQ;
// NQ = -1: any number, with G steps past kQsMax read from memory.  (That read in the loop, even where it is
// never taken, makes the step after it wait for every load in flight.)
template <class T, class TO, int FM, int FN, int FI, int NQ>
__global__ __launch_bounds__(256, one_wave<T>(FM, FI) ? 1 : 2) void chi0_contract_kernel(
    const Chi0Task *__restrict__ tasks, const Chi0Out *__restrict__ outs, int nout, const Chi0Seg *__restrict__ segs,
    const T *__restrict__ Gpm, long long zg, const T *__restrict__ W, long long zw, const T *__restrict__ Cfin,
    TO *__restrict__ chi, long long zc, int NAO, int qsl, int single, const unsigned char *__restrict__ skip) {
    using V = typename CT<T>::V;
    using A = typename CT<T>::A;
    using Q = typename CT<T>::template Cols<FN>;
    constexpr int VL = CT<T>::VL, G = FM / VL;
    constexpr unsigned TS = sizeof(T);
    constexpr bool ONE = one_wave<T>(FM, FI);
    constexpr int RQ = ONE || FN < VL ? 8 : 4, RC = (!ONE && (FM * FI >= 12 || FM >= 8)) || FM >= 16 ? 2 : 4;
    static_assert((NQ < 0 || NQ % RQ == 0) && (4 * FI) % RC == 0, "rings");
    static_assert(G * VL == FM && (FN == VL || 2 * FN == VL), "row fragments come in vectors, columns in whole or half ones");
    extern __shared__ __align__(16) char smem[];
    T *P = reinterpret_cast<T *>(smem);

    // contiguous tasks on one XCD: they share the W slab of their J
    const int nb = gridDim.x, per8 = nb / 8, rem = nb % 8, x8 = blockIdx.x & 7, i8 = blockIdx.x >> 3;
    const Chi0Task tk = tasks[x8 < rem ? x8 * (per8 + 1) + i8 : rem * (per8 + 1) + (x8 - rem) * per8 + i8];
    const int z = blockIdx.y;
    if (skip != nullptr && skip[(long long)z * nout + tk.out] != 0) return;
    const Chi0Out O = outs[tk.out];
    Gpm += z * zg;
    W += z * zw;
    chi += z * zc;
    const int lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = tk.ns == 4 ? 0 : tk.ns == 2 ? wave >> 1 : wave;
    const int n0 = tk.n0 + (wave - sub * tk.ns) * 16 * FN;
    const int part = tk.part;  // segments of one wave
    const int ta = tk.t0 + sub * part, tb = sub < tk.kp ? min(tk.t1, ta + part) : ta;
    const bool active = ta < tb && n0 < O.aj;
    const int ni = O.ni, ai = O.ai, aj = O.aj, qn = 2 * O.nj;
    const int QS = (qn + 3) / 4;
    // byte offsets of a lane: its column, and row kq of the four rows of a step of W and of Cs, clamped
    // to the last row (G, and so T, is zero past the end); the base of a segment is wave-uniform
    const unsigned nul = min(n0 + c * FN, aj - 1) * TS;
    const unsigned qstep = 4 * aj * TS, qo = kq * aj * TS + nul, qmax = (qn - 1) * aj * TS + nul;
    const unsigned cstep = 4 * ai * TS, co = kq * ai * TS;
    unsigned mul[G];
#pragma unroll
    for (int g = 0; g < G; ++g) mul[g] = min(tk.m0 + (g * 16 + c) * VL, ai - 1) * TS;
    A acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[a][b] = A{0, 0, 0, 0};

    const int mb = min(tb, O.lsum);
    for (int i0 = 0; i0 < ni; i0 += 16 * FI) {
        if (tk.t0 >= O.lsum) break;
        if (i0 > 0) __syncthreads();
        for (int e = threadIdx.x; e < FI * qsl * 64; e += 256) {
            const int f = (e >> 6) / qsl;
            P[e] = g_element(Gpm + O.gpm, i0, f, (e >> 6) - f * qsl, e & 63, ni, qn, NAO);
        }
        __syncthreads();
        if (!active || ta >= mb) continue;

        const int CS = min(4 * FI, (ni - i0 + 3) / 4);
        const Chi0Seg *st = segs + O.segtab;
        const auto q_base = [&](const Chi0Seg &sg) {
            return W + O.wseg + ((long long)sg.cell * NAO + sg.row) * qn * aj;
        };
        const auto c_base = [&](const Chi0Seg &sg) { return Cfin + O.cfin + ((long long)sg.c * ni + i0) * ai; };
        const unsigned cmax = (ni - 1 - i0) * ai * TS;
        const auto load_q = [&](const T *qb, int s) { return load_at<Q>(qb, min(qo + s * qstep, qmax)); };
        const auto load_c = [&](V *cc, const T *cb, int s) {
            const unsigned o = min(co + s * cstep, cmax);
#pragma unroll
            for (int g = 0; g < G; ++g) cc[g] = load_at<V>(cb, o + mul[g]);
        };
        A tf[FI][FN];
        const auto zero_t = [&]() {
#pragma unroll
            for (int f = 0; f < FI; ++f)
#pragma unroll
                for (int b = 0; b < FN; ++b) tf[f][b] = A{0, 0, 0, 0};
        };
        T pn[FI];
        const auto load_p = [&](int s) {
#pragma unroll
            for (int f = 0; f < FI; ++f)
                pn[f] = NQ >= 0 || s < qsl ? P[(f * qsl + s) * 64 + lane] : g_element(Gpm + O.gpm, i0, f, s, lane, ni, qn, NAO);
        };
        const bool two = i0 + 16 < ni;  // more than one fragment of rows in this pass
        const auto t_step = [&](const T *p, const Q &q) {
#pragma unroll
            for (int f = 0; f < FI; ++f) {
                if (NQ <= 0 && f > 0 && !two) break;
#pragma unroll
                for (int b = 0; b < FN; ++b) tf[f][b] = mfma(p[f], q[b], tf[f][b]);
            }
        };
        const auto c_step = [&](const V *cc, int s) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int e = 0; e < VL; ++e)
#pragma unroll
                    for (int b = 0; b < FN; ++b)
                        acc[g * VL + e][b] = mfma(cc[g][e], tf[s / 4][b][s % 4], acc[g * VL + e][b]);
        };
        // RQ steps of W and RC steps of Cs in flight: each register is loaded again as soon as the
        // MFMAs that read it are issued
        Q qr[RQ];
        V cr[RC][G];
        Chi0Seg s0 = st[ta], s1 = st[min(ta + 1, mb - 1)];
        const T *qb = q_base(s0), *cb = c_base(s0);
#pragma unroll
        for (int s = 0; s < RQ; ++s) qr[s] = load_q(qb, s);
        load_p(0);
        for (int t = ta; t < mb; ++t) {
            // (opaque: comparisons with the steps stay in the loop, two scalar instructions each; ahead of it
            // they were two dozen masks, spilled)
            int qsteps = QS, csteps = CS;
            asm volatile("" : "+s"(qsteps), "+s"(csteps));
            const T *qn_ = q_base(s1), *cn_ = c_base(s1);
            s1 = st[min(t + 2, mb - 1)];
#pragma unroll
            for (int s = 0; s < RC; ++s) load_c(cr[s], cb, s);
            zero_t();
            // a group of RQ steps from g0 on; their registers go on with the steps from g1 on of `from`
            const auto group = [&](int g0, int all, const T *from, int g1) {
#pragma unroll
                for (int u = 0; u < RQ; ++u) {
                    T pc[FI];
#pragma unroll
                    for (int f = 0; f < FI; ++f) pc[f] = pn[f];
                    load_p(g0 + u + 1 < all ? g0 + u + 1 : 0);
                    if (g0 + u < qsteps) t_step(pc, qr[u]);
                    qr[u] = load_q(from, g1 + u);
                }
            };
            if constexpr (NQ > 0) {
#pragma unroll
                for (int g = 0; g < NQ; g += RQ) group(g, NQ, g + RQ < NQ ? qb : qn_, g + RQ < NQ ? g + RQ : 0);
            } else {
                int g = 0;
                for (; g + RQ < qsteps; g += RQ) group(g, qsteps, qb, g + RQ);
                group(g, qsteps, qn_, 0);
            }
#pragma unroll
            for (int s = 0; s < 4 * FI; ++s) {
                if (s < csteps) c_step(cr[s % RC], s);
                if (s + RC < 4 * FI) load_c(cr[s % RC], cb, s + RC);
            }
            qb = qn_;
            cb = cn_;
        }
    }
    if (active) direct_term<T, FM, FN, RC>(O, W, max(ta, O.lsum) - O.lsum, tb - O.lsum, kq, mul, nul, acc);

    // the kp parts of a strip are summed in LDS, so that one wave adds to chi (an FP64 atomic add per
    // part and element took as long as the products on small blocks: 58 million of them in 1.4 ms)
    for (int k = 1; k < tk.kp; ++k) {
        T *slot = P + (wave - sub * tk.ns) * (FM * FN * 256) + lane * 4;
        __syncthreads();
        if (sub == k)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) *reinterpret_cast<A *>(slot + (a * FN + b) * 256) = acc[a][b];
        __syncthreads();
        if (sub == 0)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] += *reinterpret_cast<const A *>(slot + (a * FN + b) * 256);
    }
    if (sub != 0 || n0 >= aj) return;
    add_to_chi<T, TO, FM, FN>(chi, O, tk.m0, n0, c, kq, acc, single);
}

void Chi0Tasks::build(const std::vector<Chi0Out> &outs, bool f64, int nz, int splitk, hipStream_t s) {
    classes.clear();
    single = splitk == 1;
    const int VL = f64 ? 2 : 4;
    // Tile class of an output: row fragments of a strip and the number of strips, columns of a lane.  A strip
    // holds all rows where it can, so that T is formed once for them (40 functions, 180 rows: T is as many
    // MFMAs as its contraction with 96 rows): up to 128 rows (FP64: 192) in strips of VL columns a lane, more in
    // strips of half the columns and up to 320 (FP64) or 256 rows.  A call (FP64 / FP32, ms) with the GEMMs
    // over a stored T, with strips of 64 rows for every n_b(J) > 32 and loads waited for, and now:
    //   33 functions,  150 rows,  8 atoms at Gamma   27.8 / 22.0    34.5 / 20.5    20.7 / 11.9
    //   40, 180, 16 atoms                             226 / 141      397 / 194      205 / 107
    //   50, 230, 16 atoms                             546 / 325          -          548 / 255
    //   70, 300,  8 atoms                             277 / 174      599 / 273      268 / 156
    //   100, 400, 2 atoms and 4 k                     365 / 247      908 / 403      362 / 174
    //   27, 140,  8 atoms                            19.4 / 15.8    12.5 / 9.2     11.0 / 7.5
    // Bound, where T is long, by the reads of Cs from L2 (0.5 KB a row fragment and step, each for FN MFMAs:
    // MFMAs take 55 to 65% of the launch).
    struct Shape { int fm, fn, strips; };
    auto shape_of = [&](const Chi0Out &o) {
        const int fr = std::max(1, ceil_div(o.ai, 16));
        if (o.nj > 2 * kQsMax) return Shape{4, VL, ceil_div(fr, 4)};
        const int strips = ceil_div(fr, f64 ? 20 : 16);
        const int fm = ceil_div(ceil_div(fr, strips), VL) * VL;
        return Shape{fm, fm <= most_whole(f64) ? VL : VL / 2, strips};
    };
    // MFMAs of one wave over all segments of a strip
    auto cost = [&](const Chi0Out &o, const Shape &h, double &main, double &direct) {
        main = direct = 0;
        // an atom without basis or auxiliary functions: no sum, and no rows for the kernel to clamp to
        if (o.ni == 0 || o.nj == 0 || o.ai == 0 || o.aj == 0) return 0.0;
        const int qs = (2 * o.nj + 3) / 4;
        main = (double)ceil_div(o.ni, 16) * h.fn * qs + (double)h.fm * h.fn * ceil_div(o.ni, 4);
        direct = (double)h.fm * h.fn * ceil_div(o.ni, 4);
        return o.lsum * main + 2.0 * o.nj * direct;
    };
    double total = 0;
    for (const auto &o : outs) {
        const Shape h = shape_of(o);
        double m, d;
        total += cost(o, h, m, d) * h.strips * ceil_div(o.aj, 16 * h.fn);
    }
    // parts: about 16384 waves a launch (8 rounds of 2 waves on each of the 1024 SIMDs, so that the
    // last round is a small share), but no part under 768 MFMAs, whose prologue and atomic adds
    // would show (10 to 20 us of MFMA time)
    const double per = std::max(768.0, total * nz / 16384.0);
    std::map<std::tuple<int, int, int, int>, size_t> at;
    for (size_t oi = 0; oi < outs.size(); ++oi) {
        const auto &o = outs[oi];
        const Shape h = shape_of(o);
        const int nq = o.nj > 2 * kQsMax ? -1 : o.nj > 32 || h.fm > 8 ? 0 : o.nj > 16 ? 16 : 8;
        const int fi = nq >= 0 && o.ni <= 16 ? 1 : 2;
        double cm, cd;
        const double cst = cost(o, h, cm, cd);
        if (cst <= 0) continue;
        const auto key = std::make_tuple(h.fm, h.fn, fi, nq);
        auto it = at.find(key);
        if (it == at.end()) {
            it = at.emplace(key, classes.size()).first;
            classes.emplace_back();
            classes.back().fm = h.fm;
            classes.back().fn = h.fn;
            classes.back().fi = fi;
            classes.back().nq = nq;
        }
        Class &cl = classes[it->second];
        cl.qs = nq > 0 ? nq : std::max(cl.qs, std::min(kQsMax, (2 * o.nj + 3) / 4));
        const int strips = ceil_div(o.aj, 16 * h.fn), nseg = o.lsum + 2 * o.nj;
        for (int n = 0; n < strips;) {
            const int left = strips - n, ns = left >= 4 ? 4 : left >= 2 ? 2 : 1;
            const int kp = single ? 1 : 4 / ns;
            int parts = splitk > 0 ? ceil_div(splitk, kp) : (int)std::max(1.0, std::min(cst / (per * kp) + 0.5, 4096.0));
            if (!f64 && splitk == 0) parts = std::max(parts, (int)std::ceil((double)o.lsum * ceil_div(o.ni, 4) / (kp * kMaxStepsF32)));
            parts = std::min(parts, std::max(1, nseg / kp));
            // segment where the share f of the cost is reached
            auto seg_at = [&](double f) {
                const double want = f * cst;
                const double t = want <= o.lsum * cm ? want / cm : o.lsum + (want - o.lsum * cm) / cd;
                return std::max(0, std::min(nseg, (int)(t + 0.5)));
            };
            for (int p = 0; p < parts; ++p) {
                const int t0 = p == 0 ? 0 : seg_at((double)p / parts), t1 = p + 1 == parts ? nseg : seg_at((double)(p + 1) / parts);
                if (t0 >= t1) continue;
                for (int m = 0; m < h.strips; ++m) cl.tasks.push_back({(int)oi, m * h.fm * 16, n * 16 * h.fn, ns, kp, t0, t1, ceil_div(t1 - t0, kp)});
            }
            n += ns;
        }
    }
    // workgroups that run side by side: one J, the same share of the segments, different I and R.
    // (Blocks of 4 to 16 I x 4 to 16 J of one R measured the same within 1%, 16 x 16 10% slower; one I and R
    // with different J, which share Cs and walk in step, 4% slower.)  Past 128 rows, where Cs is most of what is
    // read, the column strips of an output beside each other as well (70 functions, 300 rows: 277 -> 269 ms).
    for (auto &cl : classes) {
        std::stable_sort(cl.tasks.begin(), cl.tasks.end(), [&](const Chi0Task &a, const Chi0Task &b) {
            const auto key = [&](const Chi0Task &t) {
                const auto &o = outs[t.out];
                const float share = (float)t.t0 / std::max(1, o.lsum + 2 * o.nj);
                return cl.fm > 8 ? std::make_tuple(o.J, share, (float)t.n0) : std::make_tuple(o.J, (float)t.n0, share);
            };
            return key(a) < key(b);
        });
        cl.d_tasks = upload(cl.tasks, s);
    }
}

template <class T, class TO>
void launch_chi0_contract(const Chi0Tasks &tk, const Chi0Out *outs, int nout, const Chi0Seg *segs, const T *Gpm,
                          long long zg, const T *W, long long zw, const T *Cfin, TO *chi, long long zc, int NAO,
                          int nz, const unsigned char *skip, hipStream_t s) {
    for (const auto &cl : tk.classes) {
        if (cl.tasks.empty()) continue;
        constexpr int VL = CT<T>::VL;
        const size_t lds = sizeof(T) * std::max(64 * cl.qs * cl.fi, tk.single ? 0 : 2 * cl.fm * cl.fn * 256);
        bool done = false;
        const auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)cl.tasks.size(), nz), dim3(256), lds, s, cl.d_tasks.as<Chi0Task>(),
                               outs, nout, segs, Gpm, zg, W, zw, Cfin, chi, zc, NAO, cl.qs, (int)tk.single, skip);
            HIP_CHECK(hipGetLastError());
            done = true;
        };
        const auto rows = [&](auto fm) {
            constexpr int FM = decltype(fm)::value;
            if constexpr (FM % VL == 0) {
                if (cl.fm != FM) return;
                if constexpr (FM > 8) {
                    constexpr int FN = FM <= most_whole(sizeof(T) == 8) ? VL : VL / 2;
                    if (cl.fi == 1) go(chi0_contract_kernel<T, TO, FM, FN, 1, 0>);
                    else go(chi0_contract_kernel<T, TO, FM, FN, 2, 0>);
                } else if (cl.nq < 0) {
                    if constexpr (FM == 4) go(chi0_contract_kernel<T, TO, 4, VL, 2, -1>);
                } else if (cl.fi == 1) {
                    if (cl.nq == 8) go(chi0_contract_kernel<T, TO, FM, VL, 1, 8>);
                    else if (cl.nq == 16) go(chi0_contract_kernel<T, TO, FM, VL, 1, 16>);
                    else go(chi0_contract_kernel<T, TO, FM, VL, 1, 0>);
                } else {
                    if (cl.nq == 8) go(chi0_contract_kernel<T, TO, FM, VL, 2, 8>);
                    else if (cl.nq == 16) go(chi0_contract_kernel<T, TO, FM, VL, 2, 16>);
                    else go(chi0_contract_kernel<T, TO, FM, VL, 2, 0>);
                }
            }
        };
        rows(std::integral_constant<int, 2>());
        rows(std::integral_constant<int, 4>());
        rows(std::integral_constant<int, 6>());
        rows(std::integral_constant<int, 8>());
        rows(std::integral_constant<int, 10>());
        rows(std::integral_constant<int, 12>());
        rows(std::integral_constant<int, 14>());
        rows(std::integral_constant<int, 16>());
        if constexpr (sizeof(T) == 8) {
            rows(std::integral_constant<int, 18>());
            rows(std::integral_constant<int, 20>());
        }
        if (!done) LRA_THROW("chi0 contraction: tile class");
    }
}
template void launch_chi0_contract<double, double>(const Chi0Tasks &, const Chi0Out *, int, const Chi0Seg *,
                                                   const double *, long long, const double *, long long, const double *,
                                                   double *, long long, int, int, const unsigned char *, hipStream_t);
template void launch_chi0_contract<float, double>(const Chi0Tasks &, const Chi0Out *, int, const Chi0Seg *,
                                                  const float *, long long, const float *, long long, const float *,
                                                  double *, long long, int, int, const unsigned char *, hipStream_t);
template void launch_chi0_contract<float, float>(const Chi0Tasks &, const Chi0Out *, int, const Chi0Seg *,
                                                 const float *, long long, const float *, long long, const float *,
                                                 float *, long long, int, int, const unsigned char *, hipStream_t);

}  // namespace lra
