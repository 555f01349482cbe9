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

namespace lra {

namespace {
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
// 16-byte buffer loads need dword alignment only (rows of odd basis sizes)
typedef double d2u __attribute__((ext_vector_type(2)));
typedef float f4u __attribute__((ext_vector_type(4)));

template <class T> struct CT;
template <> struct CT<double> { using V = d2u; using A = v4d; static constexpr int VL = 2; };
template <> struct CT<float> { using V = f4u; using A = v4f; static constexpr int VL = 4; };

__device__ __forceinline__ v4d mfma(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// One wave a SIMD with long rings, or two with short ones: two hide the instructions between the MFMAs
// (FP32, 120-row blocks of 27-row fragments: 18.7 -> 17.0 ms a 32-atom build) as long as the accumulators
// leave registers for them; 128 + 32 FP64 ones do not (38 spilled: 205 -> 258 ms on 64 atoms).
template <class T> constexpr bool one_wave(int fm, int fi) { return sizeof(T) == 8 && fm * fi >= 16; }

// An FP32 accumulator takes at most this many steps (of four products) before it is added to chi.  Diagonal
// blocks of the 128-atom cell against FP64: off by 1.28e-6 of their norm (rms) with a segment list in two to
// four accumulators (up to 6400 steps each), by 0.77e-6 with this limit, and the launches 5% shorter (977 ->
// 931 ms for 16 tau points).  The GEMMs over a stored T that took quarters of the list were off by 0.86e-6.
constexpr double kMaxStepsF32 = 1600;

constexpr int kQsMax = 64;  // G steps kept in LDS (n_b(J) <= 128); later ones are read from memory
}  // namespace

// NQ: steps of W held in registers (n_b(J) <= 2 NQ); NQ = 0 for larger n_b(J), whose steps are
// read four at a time.
template <class T, class TO, int FM, int FI, int NQ>
__global__ __launch_bounds__(256, one_wave<T>(FM, FI) ? 1 : 2) void chi0_contract_kernel(
    const Chi0Task *__restrict__ tasks, const Chi0Out *__restrict__ outs, int nout, const Chi0Seg *__restrict__ segs,
    const T *__restrict__ Gpm, long long zg, const T *__restrict__ W, long long zw, const T *__restrict__ Cfin,
    TO *__restrict__ chi, long long zc, int NAO, int qsl, int single, const unsigned char *__restrict__ skip) {
    using V = typename CT<T>::V;
    using A = typename CT<T>::A;
    constexpr int VL = CT<T>::VL, FN = VL, G = FM / VL;
    constexpr unsigned TS = sizeof(T);
    constexpr bool ONE = one_wave<T>(FM, FI);
    constexpr int RQ = NQ > 0 ? (ONE ? 8 : 4) : 1, RC = !ONE && (FM * FI >= 12 || FM == 8) ? 2 : 4;
    static_assert(NQ % RQ == 0 && (4 * FI) % RC == 0, "rings");
    static_assert(G * VL == FM, "row fragments come in vectors");
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
    const unsigned nul = min(n0 + c * VL, aj - 1) * TS;
    const unsigned qstep = 4 * aj * TS, qo = kq * aj * TS + nul, qmax = (qn - 1) * aj * TS + nul;
    const unsigned cstep = 4 * ai * TS, co = kq * ai * TS;
    unsigned mul[G];
#pragma unroll
    for (int g = 0; g < G; ++g) mul[g] = min(tk.m0 + (g * 16 + c) * VL, ai - 1) * TS;
    // 16 bytes at base + o: base in scalar registers, o one vector register (a 64-bit lane address per step
    // and fragment, worked out ahead of the loop, took 64 registers and two moves per load)
    const auto at = [](const T *b, unsigned o) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(b), 0, -1, 0x00027000);
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
    };

    A acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[a][b] = A{0, 0, 0, 0};

    const int mb = min(tb, O.lsum);
    for (int i0 = 0; i0 < ni; i0 += 16 * FI) {
        if (tk.t0 >= O.lsum) break;
        // G_IJ rows [i0, i0 + 16 FI) as A fragments: step s of fragment f at P[(f qsl + s) 64 + lane],
        // zero past n_b(I) and 2 n_b(J)
        if (i0 > 0) __syncthreads();
        for (int e = threadIdx.x; e < FI * qsl * 64; e += 256) {
            const int l = e & 63, f = (e >> 6) / qsl, s = (e >> 6) - f * qsl;
            const int rho = l & 15;
            const int i = i0 + f * 16 + (TS == 8 ? rho : 4 * (rho & 3) + (rho >> 2));
            const int q = 4 * s + (l >> 4);
            P[e] = (i < ni && q < qn) ? Gpm[O.gpm + (long long)i * 2 * NAO + q] : T(0);
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
        const auto load_q = [&](const T *qb, int s) { return at(qb, min(qo + s * qstep, qmax)); };
        const auto load_c = [&](V *cc, const T *cb, int s) {
            const unsigned o = min(co + s * cstep, cmax);
#pragma unroll
            for (int g = 0; g < G; ++g) cc[g] = at(cb, o + mul[g]);
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
            for (int f = 0; f < FI; ++f) pn[f] = P[(f * qsl + s) * 64 + lane];
        };
        const auto t_step = [&](const T *p, const V &q) {
#pragma unroll
            for (int f = 0; f < FI; ++f)
#pragma unroll
                for (int b = 0; b < FN; ++b) tf[f][b] = mfma(p[f], q[b], tf[f][b]);
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
        if constexpr (NQ > 0) {
            // RQ steps of W and RC steps of Cs in flight: each register is loaded again as soon as the
            // MFMAs that read it are issued
            V qr[RQ], cr[RC][G];
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
#pragma unroll
                for (int s = 0; s < NQ; ++s) {
                    T pc[FI];
#pragma unroll
                    for (int f = 0; f < FI; ++f) pc[f] = pn[f];
                    load_p(s + 1 < NQ ? s + 1 : 0);
                    if (s < qsteps) t_step(pc, qr[s % RQ]);
                    if (s + RQ < NQ) qr[s % RQ] = load_q(qb, s + RQ);
                    else qr[s % RQ] = load_q(qn_, s + RQ - NQ);
                }
#pragma unroll
                for (int s = 0; s < 4 * FI; ++s) {
                    if (s < csteps) c_step(cr[s % RC], s);
                    if (s + RC < 4 * FI) load_c(cr[s % RC], cb, s + RC);
                }
                qb = qn_;
                cb = cn_;
            }
        } else {
            for (int t = ta; t < mb; ++t) {
                const Chi0Seg sg = st[t];
                const T *qb = q_base(sg), *cb = c_base(sg);
                zero_t();
                for (int s0 = 0; s0 < QS; s0 += 4) {
                    V q[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) q[u] = load_q(qb, s0 + u);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int s = s0 + u;
                        if (s >= QS) break;
                        if (s < qsl) {
                            load_p(s);
                            t_step(pn, q[u]);
                        } else {  // G steps past the LDS share
#pragma unroll
                            for (int f = 0; f < FI; ++f) {
                                const int i = i0 + f * 16 + (TS == 8 ? c : 4 * (c & 3) + (c >> 2)), qi = 4 * s + kq;
                                const T p = (i < ni && qi < qn) ? Gpm[O.gpm + (long long)i * 2 * NAO + qi] : T(0);
#pragma unroll
                                for (int b = 0; b < FN; ++b) tf[f][b] = mfma(p, q[u][b], tf[f][b]);
                            }
                        }
                    }
                }
#pragma unroll
                for (int s = 0; s < 4 * FI; ++s)
                    if (s < CS) {
                        V cc[G];
                        load_c(cc, cb, s);
                        c_step(cc, s);
                    }
            }
        }
    }
    // direct term: segment lsum + (s', j) contracts over i
    const unsigned ao_ = kq * ai * TS, aol = min(kq, (ni - 1) & 3) * ai * TS;
    const unsigned bo = kq * qn * aj * TS + nul, bol = min(kq, (ni - 1) & 3) * qn * aj * TS + nul;
    const int xa0 = max(ta, O.lsum) - O.lsum, nic = (ni + 4 * RC - 1) / (4 * RC), nu = active ? max(0, (tb - O.lsum - xa0) * nic) : 0;
    if (nu > 0) {
        V ar[RC][G], br[RC];
        // step s of the u-th (s', j), i block
        const auto load = [&](int u, int s) {
            const int x = xa0 + u / nic, i0 = (u % nic) * 4 * RC;
            const int sp = x >= O.nj ? 1 : 0, j = x - sp * O.nj;
            const int is = min(i0 + 4 * s, (ni - 1) & ~3);
            const bool last = is + 4 >= ni;
            const T *ab = W + O.xa + ((long long)j * 2 * ni + (1 - sp) * ni + is) * ai;
            const T *bb = W + O.xb + ((long long)is * qn + sp * O.nj + j) * aj;
#pragma unroll
            for (int g = 0; g < G; ++g) ar[s][g] = at(ab, (last ? aol : ao_) + mul[g]);
            br[s] = at(bb, last ? bol : bo);
            if (i0 + 4 * s + kq >= ni)
#pragma unroll
                for (int b = 0; b < VL; ++b) br[s][b] = T(0);
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

#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int rho = TS == 8 ? 4 * r + kq : 4 * kq + r;
            const int mu = tk.m0 + ((a / VL) * 16 + rho) * VL + a % VL;
            if (mu >= ai) continue;
            TO *dst = chi + O.eoff + (long long)mu * aj + n0 + c * VL;
#pragma unroll
            for (int b = 0; b < FN; ++b) {
                if (n0 + c * VL + b >= aj) continue;
                if (single) dst[b] += static_cast<TO>(acc[a][b][r]);
                else unsafeAtomicAdd(dst + b, static_cast<TO>(acc[a][b][r]));
            }
        }
}

void Chi0Tasks::build(const std::vector<Chi0Out> &outs, bool f64, int nz, int splitk, hipStream_t s) {
    classes.clear();
    single = splitk == 1;
    const int VL = f64 ? 2 : 4, FN = VL;
    auto fm_of = [&](int ai, int &strips) {
        const int fr = ceil_div(ai, 16);
        strips = std::max(1, ceil_div(fr, 8));
        return std::max(VL, ceil_div(ceil_div(fr, strips), VL) * VL);
    };
    // MFMAs of one wave over all segments of a strip
    auto cost = [&](const Chi0Out &o, int fm, double &main, double &direct) {
        main = direct = 0;
        // an atom without basis or auxiliary functions: no sum, and no rows for the kernel to clamp to
        if (o.ni == 0 || o.nj == 0 || o.ai == 0 || o.aj == 0) return 0.0;
        const int qs = (2 * o.nj + 3) / 4;
        main = (double)ceil_div(o.ni, 16) * FN * qs + (double)fm * FN * ceil_div(o.ni, 4);
        direct = (double)fm * FN * ceil_div(o.ni, 4);
        return o.lsum * main + 2.0 * o.nj * direct;
    };
    double total = 0;
    for (const auto &o : outs) {
        int ms = 1;
        const int fm = fm_of(o.ai, ms);
        double m, d;
        total += cost(o, fm, m, d) * ms * ceil_div(o.aj, 16 * FN);
    }
    // parts: about 16384 waves a launch (8 rounds of 2 waves on each of the 1024 SIMDs, so that the
    // last round is a small share), but no part under 768 MFMAs, whose prologue and atomic adds
    // would show (10 to 20 us of MFMA time)
    const double per = std::max(768.0, total * nz / 16384.0);
    std::map<std::tuple<int, int, int>, size_t> at;
    for (size_t oi = 0; oi < outs.size(); ++oi) {
        const auto &o = outs[oi];
        int ms = 1;
        const int fm0 = fm_of(o.ai, ms), nq = o.nj <= 16 ? 8 : o.nj <= 32 ? 16 : 0;
        const int fm = nq > 0 ? fm0 : 4, fi = nq > 0 && o.ni <= 16 ? 1 : 2;
        if (nq == 0) ms = ceil_div(o.ai, 64);
        double cm, cd;
        const double cst = cost(o, fm, cm, cd);
        if (cst <= 0) continue;
        auto it = at.find({fm, fi, nq});
        if (it == at.end()) {
            it = at.emplace(std::make_tuple(fm, fi, nq), classes.size()).first;
            classes.emplace_back();
            classes.back().fm = fm;
            classes.back().fi = fi;
            classes.back().nq = nq;
        }
        Class &cl = classes[it->second];
        cl.qs = nq > 0 ? nq : std::max(cl.qs, std::min(kQsMax, (2 * o.nj + 3) / 4));
        const int strips = ceil_div(o.aj, 16 * FN), nseg = o.lsum + 2 * o.nj;
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
                for (int m = 0; m < ms; ++m) cl.tasks.push_back({(int)oi, m * fm * 16, n * 16 * FN, ns, kp, t0, t1, ceil_div(t1 - t0, kp)});
            }
            n += ns;
        }
    }
    // workgroups that run side by side: one J, the same share of the segments, different I and R.
    // (Blocks of 4 to 16 I x 4 to 16 J of one R measured the same within 1%, 16 x 16 10% slower; one I and R
    // with different J, which share Cs and walk in step, 4% slower.)
    for (auto &cl : classes) {
        std::stable_sort(cl.tasks.begin(), cl.tasks.end(), [&](const Chi0Task &a, const Chi0Task &b) {
            const auto key = [&](const Chi0Task &t) {
                const auto &o = outs[t.out];
                return std::make_tuple(o.J, t.n0, (float)t.t0 / std::max(1, o.lsum + 2 * o.nj));
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
        const int fn = sizeof(T) == 8 ? 2 : 4;
        const size_t lds = sizeof(T) * std::max(64 * cl.qs * cl.fi, tk.single ? 0 : 2 * cl.fm * fn * 256);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)cl.tasks.size(), nz), dim3(256), lds, s, cl.d_tasks.as<Chi0Task>(),
                               outs, nout, segs, Gpm, zg, W, zw, Cfin, chi, zc, NAO, cl.qs, (int)tk.single, skip);
            HIP_CHECK(hipGetLastError());
        };
        const auto by_fi_nq = [&](auto fm) {
            constexpr int FM = decltype(fm)::value;
            if (cl.fi == 1 && cl.nq == 8) go(chi0_contract_kernel<T, TO, FM, 1, 8>);
            else if (cl.fi == 1 && cl.nq == 16) go(chi0_contract_kernel<T, TO, FM, 1, 16>);
            else if (cl.fi == 2 && cl.nq == 8) go(chi0_contract_kernel<T, TO, FM, 2, 8>);
            else if (cl.fi == 2 && cl.nq == 16) go(chi0_contract_kernel<T, TO, FM, 2, 16>);
            else LRA_THROW("chi0 contraction: tile class");
        };
        if (cl.nq == 0 && cl.fm == 4 && cl.fi == 2) go(chi0_contract_kernel<T, TO, 4, 2, 0>);
        else if (cl.fm == 4) by_fi_nq(std::integral_constant<int, 4>());
        else if (cl.fm == 8) by_fi_nq(std::integral_constant<int, 8>());
        else if (cl.fm == 2 && sizeof(T) == 8) by_fi_nq(std::integral_constant<int, sizeof(T) == 8 ? 2 : 4>());
        else if (cl.fm == 6 && sizeof(T) == 8) by_fi_nq(std::integral_constant<int, sizeof(T) == 8 ? 6 : 4>());
        else LRA_THROW("chi0 contraction: tile class");
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
