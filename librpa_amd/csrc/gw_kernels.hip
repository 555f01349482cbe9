// Streaming kernels of the G0W0 path (gfx950).
#include "gw_kernels.h"

#include <cmath>
#include <type_traits>

namespace lra {

// One element of (a, b), kWTau tau points and kWCells cells a thread: sums over the frequencies of each q
// of the pass first, then over q with its phases, so that W(q, omega) is read once per four tau points
// and eight cells and W(R, tau) is written once per pass over q (it was read and written again for
// every q and eight frequencies).
constexpr int kWTau = 4, kWCells = 8;
__global__ __launch_bounds__(256) void w_accum_kernel(const double *__restrict__ aug, long long stride, long long im,
                                                      int nq, int nw, int n, const double *__restrict__ coef, int ntau,
                                                      const double *__restrict__ ph, int nR, double *__restrict__ Wrt) {
    const long long nn = (long long)n * n;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nn) return;
    const int a = (int)(idx / n), b = (int)(idx % n), N = 2 * n;
    const int t0 = blockIdx.y * kWTau, r0 = blockIdx.z * kWCells;
    const long long at = (long long)(n + max(a, b)) * N + n + min(a, b);
    const double sgn = a < b ? -1.0 : 1.0;  // Im W_ab = -Im W_ba
    double acc[kWTau][kWCells];
#pragma unroll
    for (int t = 0; t < kWTau; ++t)
#pragma unroll
        for (int r = 0; r < kWCells; ++r) acc[t][r] = 0;
    for (int q = 0; q < nq; ++q) {
        double x[kWTau], y[kWTau];
#pragma unroll
        for (int t = 0; t < kWTau; ++t) x[t] = y[t] = 0;
        for (int w = 0; w < nw; ++w) {
            const double *A = aug + ((long long)q * nw + w) * stride + at;
            const double re = -A[0], ii = im ? -sgn * A[im] : 0.0;
#pragma unroll
            for (int t = 0; t < kWTau; ++t) {
                const double c = coef[((long long)q * nw + w) * ntau + min(t0 + t, ntau - 1)];
                x[t] += c * re;
                y[t] += c * ii;
            }
        }
#pragma unroll
        for (int r = 0; r < kWCells; ++r) {
            const double *p = ph + 2 * ((long long)q * nR + min(r0 + r, nR - 1));
#pragma unroll
            for (int t = 0; t < kWTau; ++t) acc[t][r] += p[0] * x[t] + p[1] * y[t];
        }
    }
#pragma unroll
    for (int t = 0; t < kWTau; ++t)
#pragma unroll
        for (int r = 0; r < kWCells; ++r)
            if (t0 + t < ntau && r0 + r < nR) Wrt[((long long)(t0 + t) * nR + r0 + r) * nn + idx] += acc[t][r];
}

void launch_w_accum(const double *aug, long long stride, long long im, int nq, int nw, int n, const double *coef,
                    int ntau, const double *ph, int nR, double *Wrt, hipStream_t s) {
    hipLaunchKernelGGL(w_accum_kernel, dim3(ceil_div((long long)n * n, 256), ceil_div(ntau, kWTau), ceil_div(nR, kWCells)),
                       dim3(256), 0, s, aug, stride, im, nq, nw, n, coef, ntau, ph, nR, Wrt);
    HIP_CHECK(hipGetLastError());
}

// lower triangle (whole rows of the lower left block) of matrix blockIdx.y = q * nw + w, plane blockIdx.z
__global__ __launch_bounds__(256) void fill_aug_kernel(double *__restrict__ A, long long stride, long long im, int nw, int n,
                                                       const double *__restrict__ C, const double *__restrict__ V,
                                                       long long nn) {
    const int N = 2 * n;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)N * N) return;
    const int i = (int)(idx / N), j = (int)(idx % N);
    if (j > i) return;
    const long long src = (blockIdx.y / nw) * nn + blockIdx.z * (long long)n * n;
    double v;
    if (i < n) v = (i == j && blockIdx.z == 0) ? 1.0 : 0.0;
    else if (j < n) v = C[src + (long long)(i - n) * n + j];
    else v = V[src + (long long)(i - n) * n + j - n];
    A[blockIdx.y * stride + blockIdx.z * im + idx] = v;
}
void launch_fill_aug(double *A, long long stride, long long im, int nq, int nw, int n, const double *C, const double *V,
                     hipStream_t s) {
    const int pl = im ? 2 : 1;
    hipLaunchKernelGGL(fill_aug_kernel, dim3(ceil_div(4LL * n * n, 256), nq * nw, pl), dim3(256), 0, s, A, stride, im, nw,
                       n, C, V, (long long)pl * n * n);
    HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// self-energy contractions
// ------------------------------------------------------------------------------------
namespace {
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
// 16-byte loads at element alignment (rows of odd basis sizes)
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
template <class T> struct SV;
template <> struct SV<double> { using A = v4d; using V = d2u; static constexpr int VL = 2; };
template <> struct SV<float> { using A = v4f; using V = f4u; static constexpr int VL = 4; };
__device__ __forceinline__ v4d mfma(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// row of a 16 x 16 result that register r of lane group kq holds
template <class T> __device__ __forceinline__ int acc_row(int r, int kq) { return sizeof(T) == 8 ? 4 * r + kq : 4 * kq + r; }

// elements [0, n) of p (n <= 4), zero past them
template <class T>
__device__ __forceinline__ void load4(T (&v)[4], const T *p, int n) {
    using V = typename SV<T>::V;
    constexpr int VL = SV<T>::VL;
    if (n >= 4) {
#pragma unroll
        for (int g = 0; g < 4 / VL; ++g) {
            const V x = *reinterpret_cast<const V *>(p + g * VL);
#pragma unroll
            for (int e = 0; e < VL; ++e) v[g * VL + e] = x[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = e < n ? p[e] : T(0);
    }
}
}  // namespace

// Sigma_IJ(R)[i][j] += sum_(c, nu) CW_IJ(R)[c][i][nu] U_J(S_c)[row_c][j][nu] over segments [c0, c1) of a
// task, both signs at once: a wave takes every fourth segment, FI x FJ fragments of 16 x 16, and 16 nu
// at a time, four consecutive ones a lane (any assignment of nu to the steps of an MFMA will do when
// both operands share it).  The four waves are summed in LDS before one atomic add per element.
// Bound by the reads of CW (each element once per pass) and, for small n_b, by U from L2: an MFMA
// multiplies a fragment pair of 1 KB in 64 (FP64) cycles, so the next fragments are in flight
// meanwhile.  8 atoms, 4 k: 24 such contractions of T = W U through an 8-workgroup GEMM took 35 ms.
template <class T, int FI, int FJ, int NSG>
__global__ __launch_bounds__(256, 2) void sigma_d_kernel(const SigTask *__restrict__ tasks, const SigBlk *__restrict__ blks,
                                                         const Chi0Seg *__restrict__ segs, const T *__restrict__ CW,
                                                         long long zcw, const T *__restrict__ U, long long usg,
                                                         T *__restrict__ sig, long long ssg, int NAO) {
    using A = typename SV<T>::A;
    __shared__ __align__(16) T red[FI * FJ * NSG * 256];
    const SigTask tk = tasks[blockIdx.x];
    const SigBlk B = blks[tk.blk];
    CW += blockIdx.y * zcw + B.cw;
    U += blockIdx.y * NSG * usg + B.u;
    sig += blockIdx.y * 2 * ssg;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, kq = lane >> 4;
    const int ni = B.ni, nj = B.nj, aj = B.aj;
    const Chi0Seg *st = segs + B.seg0;
    int ao[FI], uo[FJ];
#pragma unroll
    for (int f = 0; f < FI; ++f) ao[f] = min(tk.i0 + 16 * f + c16, ni - 1) * aj + 4 * kq;
#pragma unroll
    for (int g = 0; g < FJ; ++g) uo[g] = min(tk.j0 + 16 * g + c16, nj - 1) * aj + 4 * kq;
    A acc[FI][FJ][NSG];
#pragma unroll
    for (int f = 0; f < FI; ++f)
#pragma unroll
        for (int g = 0; g < FJ; ++g)
#pragma unroll
            for (int s = 0; s < NSG; ++s) acc[f][g][s] = A{0, 0, 0, 0};
    struct Frag { T a[FI][4], u[NSG][FJ][4]; };
    auto load = [&](Frag &x, int t, int k0) {
        const Chi0Seg sg = st[t];
        const T *ab = CW + (long long)sg.c * ni * aj + k0;
        const T *ub = U + ((long long)sg.cell * NAO + sg.row) * nj * aj + k0;
        const int n = aj - k0 - 4 * kq;
#pragma unroll
        for (int f = 0; f < FI; ++f) load4(x.a[f], ab + ao[f], n);
#pragma unroll
        for (int s = 0; s < NSG; ++s)
#pragma unroll
            for (int g = 0; g < FJ; ++g) load4(x.u[s][g], ub + s * usg + uo[g], n);
    };
    auto use = [&](const Frag &x) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int s = 0; s < NSG; ++s)
#pragma unroll
                for (int f = 0; f < FI; ++f)
#pragma unroll
                    for (int g = 0; g < FJ; ++g) acc[f][g][s] = mfma(x.a[f][e], x.u[s][g][e], acc[f][g][s]);
    };
    int t = tk.c0 + wave, k0 = 0;
    if (t < tk.c1) {
        Frag x, y;
        load(x, t, k0);
        for (;;) {
            k0 += 16;
            if (k0 >= aj) { k0 = 0; t += 4; }
            const bool more = t < tk.c1;
            if (more) load(y, t, k0);
            use(x);
            if (!more) break;
            x = y;
        }
    }
    for (int w = 1; w < 4; ++w) {
        __syncthreads();
        if (wave == w)
#pragma unroll
            for (int f = 0; f < FI; ++f)
#pragma unroll
                for (int g = 0; g < FJ; ++g)
#pragma unroll
                    for (int s = 0; s < NSG; ++s) *reinterpret_cast<A *>(&red[(((f * FJ + g) * NSG + s) * 64 + lane) * 4]) = acc[f][g][s];
        __syncthreads();
        if (wave == 0)
#pragma unroll
            for (int f = 0; f < FI; ++f)
#pragma unroll
                for (int g = 0; g < FJ; ++g)
#pragma unroll
                    for (int s = 0; s < NSG; ++s) acc[f][g][s] += *reinterpret_cast<const A *>(&red[(((f * FJ + g) * NSG + s) * 64 + lane) * 4]);
    }
    if (wave != 0) return;
#pragma unroll
    for (int f = 0; f < FI; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = tk.i0 + 16 * f + acc_row<T>(r, kq);
            if (i >= ni) continue;
#pragma unroll
            for (int g = 0; g < FJ; ++g) {
                const int j = tk.j0 + 16 * g + c16;
                if (j >= nj) continue;
                T *dst = sig + ((long long)B.r * NAO + B.rowI + i) * NAO + B.colJ + j;
#pragma unroll
                for (int s = 0; s < NSG; ++s) unsafeAtomicAdd(dst + s * ssg, acc[f][g][s][r]);
            }
        }
}

// S2(S_c)[row_c][j] += sum_(i, nu) CW_IJ(R)[c][(i, nu)] U_J(R)[(I, i)][j][nu] for the 16 FC segments of a
// wave (64 FC of a task, from c0), FJ fragments of j and both signs; operands as in sigma_d_kernel.
template <class T, int FC, int FJ, int NSG>
__global__ __launch_bounds__(256, 2) void sigma_b_kernel(const SigTask *__restrict__ tasks, const SigBlk *__restrict__ blks,
                                                         const Chi0Seg *__restrict__ segs, const T *__restrict__ CW,
                                                         long long zcw, const T *__restrict__ U, long long usg,
                                                         T *__restrict__ s2, long long ssg, int NAO) {
    using A = typename SV<T>::A;
    const SigTask tk = tasks[blockIdx.x];
    const SigBlk B = blks[tk.blk];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, kq = lane >> 4;
    const int ni = B.ni, nj = B.nj, aj = B.aj, t0 = tk.c0 + 16 * FC * wave;
    if (t0 >= B.l) return;
    CW += blockIdx.y * zcw + B.cw;
    U += blockIdx.y * NSG * usg + B.u + ((long long)B.r * NAO + B.rowI) * nj * aj;
    s2 += blockIdx.y * 2 * ssg;
    const Chi0Seg *st = segs + B.seg0;
    const T *ap[FC];
#pragma unroll
    for (int f = 0; f < FC; ++f) ap[f] = CW + (long long)st[min(t0 + 16 * f + c16, B.l - 1)].c * ni * aj + 4 * kq;
    int uo[FJ];
#pragma unroll
    for (int g = 0; g < FJ; ++g) uo[g] = min(tk.j0 + 16 * g + c16, nj - 1) * aj + 4 * kq;
    A acc[FC][FJ][NSG];
#pragma unroll
    for (int f = 0; f < FC; ++f)
#pragma unroll
        for (int g = 0; g < FJ; ++g)
#pragma unroll
            for (int s = 0; s < NSG; ++s) acc[f][g][s] = A{0, 0, 0, 0};
    struct Frag { T a[FC][4], u[NSG][FJ][4]; };
    auto load = [&](Frag &x, int i, int k0) {
        const int n = aj - k0 - 4 * kq;
        const T *ub = U + (long long)i * nj * aj + k0;
#pragma unroll
        for (int f = 0; f < FC; ++f) load4(x.a[f], ap[f] + i * aj + k0, n);
#pragma unroll
        for (int s = 0; s < NSG; ++s)
#pragma unroll
            for (int g = 0; g < FJ; ++g) load4(x.u[s][g], ub + s * usg + uo[g], n);
    };
    int i = 0, k0 = 0;
    Frag x, y;
    load(x, i, k0);
    for (;;) {
        k0 += 16;
        if (k0 >= aj) { k0 = 0; ++i; }
        const bool more = i < ni;
        if (more) load(y, i, k0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int s = 0; s < NSG; ++s)
#pragma unroll
                for (int f = 0; f < FC; ++f)
#pragma unroll
                    for (int g = 0; g < FJ; ++g) acc[f][g][s] = mfma(x.a[f][e], x.u[s][g][e], acc[f][g][s]);
        if (!more) break;
        x = y;
    }
#pragma unroll
    for (int f = 0; f < FC; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = t0 + 16 * f + acc_row<T>(r, kq);
            if (t >= B.l) continue;
            const Chi0Seg sg = st[t];
#pragma unroll
            for (int g = 0; g < FJ; ++g) {
                const int j = tk.j0 + 16 * g + c16;
                if (j >= nj) continue;
                T *dst = s2 + ((long long)sg.cell * NAO + sg.row) * NAO + B.colJ + j;
#pragma unroll
                for (int s = 0; s < NSG; ++s) unsafeAtomicAdd(dst + s * ssg, acc[f][g][s][r]);
            }
        }
}

// Y_I[(S, L, l)][i][mu] (+)= sum_(J, R, j) G_IJ(R)[i][j] CW_JI(-R)[(L, S - R, l)][j][mu], both signs: a wave
// takes one column (S, L, l), 16 FI rows i and 64 mu, and the entries (J, R) of (S, L) with J in
// [x0, x1) (first chunk: Y is overwritten).  Each element of CW is read once, 16 bytes a lane, for
// 2 FI MFMAs; G_IJ comes from L2.
template <class T, int FI, int NSG>
__global__ __launch_bounds__(256, 2) void sigma_y_kernel(const SigYTask *__restrict__ tasks, const SigYEnt *__restrict__ ents,
                                                         const T *__restrict__ CW, long long zcw, const T *__restrict__ G,
                                                         long long zg, T *__restrict__ Y, long long ysg, int NAO, int x0,
                                                         int x1, int first, int sg0) {
    using A = typename SV<T>::A;
    using V = typename SV<T>::V;
    constexpr int VL = SV<T>::VL, NV = 4 / VL;
    const SigYTask tk = tasks[blockIdx.x];
    const int lane = threadIdx.x & 63, c16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = tk.l0 + wave;
    if (l >= tk.nl) return;
    CW += blockIdx.y * zcw;
    G += blockIdx.y * zg + (long long)tk.ao * 2 * NAO;
    Y += blockIdx.y * NSG * ysg + tk.y;
    const int ni = tk.ni, ai = tk.ai;
    int go[FI], mo[NV];
#pragma unroll
    for (int f = 0; f < FI; ++f) go[f] = min(tk.i0 + 16 * f + c16, ni - 1) * 2 * NAO;
#pragma unroll
    for (int v = 0; v < NV; ++v) mo[v] = min(tk.mu0 + (16 * v + c16) * VL, ai - 1);
    A acc[FI][4][NSG];
#pragma unroll
    for (int f = 0; f < FI; ++f)
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int q = 0; q < NSG; ++q) acc[f][m][q] = A{0, 0, 0, 0};
    struct Frag { T g[NSG][FI]; V w[NV]; };
    int e = tk.e0 - 1, s = 0, ns = 0, nj = 0;
    const T *pg = nullptr, *pw = nullptr;
    auto next_entry = [&]() {
        for (++e; e < tk.e1; ++e) {
            const SigYEnt E = ents[e];
            if (E.J < x0 || E.J >= x1) continue;
            nj = E.nj;
            ns = (nj + 3) / 4;
            pg = G + E.g;
            pw = CW + E.b + (long long)tk.abf * E.lb + (long long)(E.cb + l * nj) * ai;
            return true;
        }
        return false;
    };
    auto load = [&](Frag &x) {
        const int j = 4 * s + kq, jc = min(j, nj - 1);
#pragma unroll
        for (int f = 0; f < FI; ++f)
#pragma unroll
            for (int q = 0; q < NSG; ++q) {
                const T v = pg[go[f] + (sg0 + q) * nj + jc];
                x.g[q][f] = j < nj ? v : T(0);
            }
#pragma unroll
        for (int v = 0; v < NV; ++v) x.w[v] = *reinterpret_cast<const V *>(pw + (long long)jc * ai + mo[v]);
    };
    if (next_entry()) {
        Frag x, y;
        load(x);
        for (;;) {
            bool more = true;
            if (++s >= ns) { s = 0; more = next_entry(); }
            if (more) load(y);
#pragma unroll
            for (int q = 0; q < NSG; ++q)
#pragma unroll
                for (int f = 0; f < FI; ++f)
#pragma unroll
                    for (int m = 0; m < 4; ++m) acc[f][m][q] = mfma(x.g[q][f], x.w[m / VL][m % VL], acc[f][m][q]);
            if (!more) break;
            x = y;
        }
    }
#pragma unroll
    for (int f = 0; f < FI; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = tk.i0 + 16 * f + acc_row<T>(r, kq);
            if (i >= ni) continue;
#pragma unroll
            for (int q = 0; q < NSG; ++q) {
                T *dst = Y + q * ysg + ((long long)l * ni + i) * ai;
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const int mu = tk.mu0 + (16 * (m / VL) + c16) * VL + m % VL;
                    if (mu >= ai) continue;
                    if (first) dst[mu] = acc[f][m][q][r];
                    else dst[mu] += acc[f][m][q][r];
                }
            }
        }
}

namespace {
// f of a, b and n (1 or 2 each) as constants
template <class F> void by_two(int a, int b, int n, F f) {
    const auto with_b = [&](auto ca) {
        const auto with_n = [&](auto cb) {
            if (n == 1) f(ca, cb, std::integral_constant<int, 1>());
            else f(ca, cb, std::integral_constant<int, 2>());
        };
        if (b == 1) with_n(std::integral_constant<int, 1>());
        else with_n(std::integral_constant<int, 2>());
    };
    if (a == 1) with_b(std::integral_constant<int, 1>());
    else with_b(std::integral_constant<int, 2>());
}
}  // namespace

template <class T>
void launch_sigma_d(const SigTask *tasks, int ntask, int fi, int fj, const SigBlk *blks, const Chi0Seg *segs, const T *CW,
                    long long zcw, const T *U, long long usg, T *sig, long long ssg, int NAO, int nz, int nsg,
                    hipStream_t s) {
    if (ntask <= 0) return;
    by_two(fi, fj, nsg, [&](auto a, auto b, auto n) {
        hipLaunchKernelGGL((sigma_d_kernel<T, decltype(a)::value, decltype(b)::value, decltype(n)::value>),
                           dim3(ntask, nz), dim3(256), 0, s, tasks, blks, segs, CW, zcw, U, usg, sig, ssg, NAO);
    });
    HIP_CHECK(hipGetLastError());
}
template <class T>
void launch_sigma_b(const SigTask *tasks, int ntask, int fc, int fj, const SigBlk *blks, const Chi0Seg *segs, const T *CW,
                    long long zcw, const T *U, long long usg, T *s2, long long ssg, int NAO, int nz, int nsg,
                    hipStream_t s) {
    if (ntask <= 0) return;
    by_two(fc, fj, nsg, [&](auto a, auto b, auto n) {
        hipLaunchKernelGGL((sigma_b_kernel<T, decltype(a)::value, decltype(b)::value, decltype(n)::value>),
                           dim3(ntask, nz), dim3(256), 0, s, tasks, blks, segs, CW, zcw, U, usg, s2, ssg, NAO);
    });
    HIP_CHECK(hipGetLastError());
}
template <class T>
void launch_sigma_y(const SigYTask *tasks, int ntask, int fi, const SigYEnt *ents, const T *CW, long long zcw, const T *G,
                    long long zg, T *Y, long long ysg, int NAO, int x0, int x1, bool first, int nz, int nsg, int sg0,
                    hipStream_t s) {
    if (ntask <= 0) return;
    by_two(fi, 1, nsg, [&](auto a, auto, auto n) {
        hipLaunchKernelGGL((sigma_y_kernel<T, decltype(a)::value, decltype(n)::value>), dim3(ntask, nz), dim3(256), 0, s,
                           tasks, ents, CW, zcw, G, zg, Y, ysg, NAO, x0, x1, (int)first, sg0);
    });
    HIP_CHECK(hipGetLastError());
}
#define LRA_SIGMA(T)                                                                                                    \
    template void launch_sigma_d<T>(const SigTask *, int, int, int, const SigBlk *, const Chi0Seg *, const T *, long long, \
                                    const T *, long long, T *, long long, int, int, int, hipStream_t);                  \
    template void launch_sigma_b<T>(const SigTask *, int, int, int, const SigBlk *, const Chi0Seg *, const T *, long long, \
                                    const T *, long long, T *, long long, int, int, int, hipStream_t);                  \
    template void launch_sigma_y<T>(const SigYTask *, int, int, const SigYEnt *, const T *, long long, const T *, long long, \
                                    T *, long long, int, int, int, bool, int, int, int, hipStream_t);
LRA_SIGMA(double)
LRA_SIGMA(float)
#undef LRA_SIGMA

// blockIdx.y: tau point and sign
template <class T>
__global__ void sigma_fold_kernel(T *__restrict__ sig, const T *__restrict__ s2, const T *__restrict__ ext,
                                  const int *__restrict__ fold, const int *__restrict__ neg, int NE, int nR, int n) {
    const long long nn = (long long)n * n;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nn * nR) return;
    sig += blockIdx.y * nn * nR;
    s2 += blockIdx.y * nn * nR;
    ext += blockIdx.y * nn * NE;
    const int R = (int)(idx / nn);
    const long long ab = idx % nn;
    const int a = (int)(ab / n), b = (int)(ab % n);
    T acc = s2[idx] + s2[neg[R] * nn + (long long)b * n + a];
    for (int e = 0; e < NE; ++e)
        if (fold[e] == R) acc += ext[(long long)e * nn + ab];
    sig[idx] += acc;
}

template <class T>
void launch_sigma_fold(T *sig, const T *s2, const T *ext, const int *fold, const int *neg, int NE, int nR, int n,
                       int nz, hipStream_t s) {
    hipLaunchKernelGGL(sigma_fold_kernel<T>, dim3(ceil_div((long long)n * n * nR, 256), 2 * nz), dim3(256), 0, s, sig,
                       s2, ext, fold, neg, NE, nR, n);
    HIP_CHECK(hipGetLastError());
}
template void launch_sigma_fold<double>(double *, const double *, const double *, const int *, const int *, int, int,
                                        int, int, hipStream_t);
template void launch_sigma_fold<float>(float *, const float *, const float *, const int *, const int *, int, int, int,
                                       int, hipStream_t);

// blockIdx.y: frequency; the tau points of a pass are added in their order
template <class T>
__global__ void sigma_freq_kernel(const T *__restrict__ sig, long long nelem, const double *__restrict__ cw,
                                  const double *__restrict__ sw, int ntau, int it0, int nz, double *__restrict__ sre,
                                  double *__restrict__ sim) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nelem) return;
    const int w = blockIdx.y;
    double re = sre[(long long)w * nelem + i], im = sim[(long long)w * nelem + i];
    for (int z = 0; z < nz; ++z) {
        const double p = static_cast<double>(sig[2ll * z * nelem + i]), m = static_cast<double>(sig[(2ll * z + 1) * nelem + i]);
        re += 0.5 * (p + m) * cw[w * ntau + it0 + z];
        im += 0.5 * (p - m) * sw[w * ntau + it0 + z];
    }
    sre[(long long)w * nelem + i] = re;
    sim[(long long)w * nelem + i] = im;
}

template <class T>
void launch_sigma_freq(const T *sig, long long nelem, const double *cw, const double *sw, int nw, int ntau, int it0,
                       int nz, double *sre, double *sim, hipStream_t s) {
    hipLaunchKernelGGL(sigma_freq_kernel<T>, dim3(ceil_div(nelem, 256), nw), dim3(256), 0, s, sig, nelem, cw, sw, ntau,
                       it0, nz, sre, sim);
    HIP_CHECK(hipGetLastError());
}
template void launch_sigma_freq<double>(const double *, long long, const double *, const double *, int, int, int, int,
                                        double *, double *, hipStream_t);
template void launch_sigma_freq<float>(const float *, long long, const double *, const double *, int, int, int, int,
                                       double *, double *, hipStream_t);

constexpr int kStMax = 16;

// one workgroup per (row a, omega); threads stride over the columns b.  Under 256 columns the threads left over
// share the cells of a column (26 functions on 8 k kept 26 threads waiting for 8 cells in turn).
__global__ __launch_bounds__(256) void sigma_ks_rows_kernel(const double *__restrict__ sre,
                                                            const double *__restrict__ sim, int nR, int n,
                                                            const int *__restrict__ atom_of, int natom,
                                                            const double *__restrict__ ph,
                                                            const double *__restrict__ U, int nst,
                                                            double *__restrict__ Y) {
    const int a = blockIdx.x, w = blockIdx.y;
    const int t = threadIdx.x;
    const int I = atom_of[a];
    double ar[kStMax], ai[kStMax];
#pragma unroll
    for (int st = 0; st < kStMax; ++st) { ar[st] = 0; ai[st] = 0; }
    const long long nn = (long long)n * n;
    const int G = n >= 256 ? 1 : min(nR, 256 / n), g = G > 1 ? t / n : 0;
    for (int b = G > 1 ? t % n : t; b < n && g < G; b += G > 1 ? n : 256) {
        const double *p = ph + ((long long)I * natom + atom_of[b]) * nR * 2;
        double vr = 0, vi = 0;
        for (int R = g; R < nR; R += G) {
            const long long e = ((long long)w * nR + R) * nn + (long long)a * n + b;
            const double sr = sre[e], si = sim[e];
            const double cr = p[2 * R], ci = p[2 * R + 1];
            vr += cr * sr - ci * si;
            vi += cr * si + ci * sr;
        }
#pragma unroll
        for (int st = 0; st < kStMax; ++st) {
            if (st < nst) {
                const double ur = U[((long long)st * n + b) * 2], ui = U[((long long)st * n + b) * 2 + 1];
                ar[st] += vr * ur - vi * ui;
                ai[st] += vr * ui + vi * ur;
            }
        }
    }
    __shared__ double red[4][2 * kStMax];
    const int lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int st = 0; st < kStMax; ++st) {
        if (st >= nst) break;
        double x = ar[st], y = ai[st];
        for (int o = 32; o > 0; o >>= 1) {
            x += __shfl_xor(x, o, 64);
            y += __shfl_xor(y, o, 64);
        }
        if (lane == 0) { red[wave][2 * st] = x; red[wave][2 * st + 1] = y; }
    }
    __syncthreads();
    if (t < 2 * nst) {
        const double v = red[0][t] + red[1][t] + red[2][t] + red[3][t];
        Y[((long long)w * n + a) * nst * 2 + t] = v;
    }
}

void launch_sigma_ks_rows(const double *sre, const double *sim, int nw, int nR, int n, const int *atom_of,
                          int natom, const double *ph, const double *U, int nst, double *Y, hipStream_t s) {
    if (nst < 1 || nst > kStMax) LRA_THROW("sigma_ks_rows: 1..16 states per launch");
    hipLaunchKernelGGL(sigma_ks_rows_kernel, dim3(n, nw), dim3(256), 0, s, sre, sim, nR, n, atom_of, natom, ph, U,
                       nst, Y);
    HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// Newton-Schulz square roots of several matrices (blockIdx.y), pl planes of n x n each
// ------------------------------------------------------------------------------------
constexpr int kNsBlocks = 32;  // partial sums and maxima per matrix

__global__ __launch_bounds__(256) void ns_norm_kernel(const double *__restrict__ A, const int *__restrict__ sel,
                                                      long long nn, double *__restrict__ part) {
    __shared__ double red[256];
    const double *M = A + sel[blockIdx.y] * nn;
    double v = 0;
    for (long long i = blockIdx.x * 256 + threadIdx.x; i < nn; i += kNsBlocks * 256) v += M[i] * M[i];
    red[threadIdx.x] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.y * kNsBlocks + blockIdx.x] = red[0];
}

__device__ __forceinline__ double ns_scale(const double *part) {
    double v = 0;
    for (int i = 0; i < kNsBlocks; ++i) v += part[i];
    return sqrt(v);
}

// Y = A / c, Z = I with c = ||A||_F (kept in scale)
__global__ __launch_bounds__(256) void ns_init_kernel(const double *__restrict__ A, const int *__restrict__ sel, int n,
                                                      long long nn, const double *__restrict__ part,
                                                      double *__restrict__ Y, double *__restrict__ Z,
                                                      double *__restrict__ scale) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    const double c = ns_scale(part + blockIdx.y * kNsBlocks);
    if (i == 0) scale[blockIdx.y] = c;
    Y[blockIdx.y * nn + i] = A[sel[blockIdx.y] * nn + i] * (1.0 / c);
    Z[blockIdx.y * nn + i] = (i < (long long)n * n && i / n == i % n) ? 1.0 : 0.0;
}
void launch_ns_init(const double *A, const int *sel, int nmat, int n, int pl, double *part, double *Y, double *Z,
                    double *scale, hipStream_t s) {
    const long long nn = (long long)pl * n * n;
    hipLaunchKernelGGL(ns_norm_kernel, dim3(kNsBlocks, nmat), dim3(256), 0, s, A, sel, nn, part);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(ns_init_kernel, dim3(ceil_div(nn, 256), nmat), dim3(256), 0, s, A, sel, n, nn, part, Y, Z, scale);
    HIP_CHECK(hipGetLastError());
}

// T = 1.5 I - 0.5 P, in place
__global__ __launch_bounds__(256) void ns_step_kernel(double *P, int n, long long nn) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    const bool diag = i < (long long)n * n && i / n == i % n;
    P[blockIdx.y * nn + i] = -0.5 * P[blockIdx.y * nn + i] + (diag ? 1.5 : 0.0);
}
void launch_ns_step(double *P, int nmat, int n, int pl, hipStream_t s) {
    const long long nn = (long long)pl * n * n;
    hipLaunchKernelGGL(ns_step_kernel, dim3(ceil_div(nn, 256), nmat), dim3(256), 0, s, P, n, nn);
    HIP_CHECK(hipGetLastError());
}

// out[2 m] = max |Yn - Y|, out[2 m + 1] = max |Y| of matrix m, as the bits of non-negative doubles (which
// order as integers); a NaN counts as infinity.  out starts from zero.
__global__ __launch_bounds__(256) void ns_change_kernel(const double *__restrict__ Yn, const double *__restrict__ Y,
                                                        long long nn, unsigned long long *__restrict__ out) {
    double d = 0, m = 0;
    const auto up = [](double &m_, double v) {
        v = fabs(v);
        if (!(v <= m_)) m_ = v < INFINITY ? v : INFINITY;
    };
    for (long long i = blockIdx.x * 256 + threadIdx.x; i < nn; i += kNsBlocks * 256) {
        const double y = Y[blockIdx.y * nn + i];
        up(d, Yn[blockIdx.y * nn + i] - y);
        up(m, y);
    }
    for (int o = 32; o > 0; o >>= 1) {
        d = fmax(d, __shfl_xor(d, o, 64));
        m = fmax(m, __shfl_xor(m, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(out + 2 * blockIdx.y, (unsigned long long)__double_as_longlong(d));
        atomicMax(out + 2 * blockIdx.y + 1, (unsigned long long)__double_as_longlong(m));
    }
}
void launch_ns_change(const double *Yn, const double *Y, int nmat, int n, int pl, unsigned long long *out, hipStream_t s) {
    hipLaunchKernelGGL(ns_change_kernel, dim3(kNsBlocks, nmat), dim3(256), 0, s, Yn, Y, (long long)pl * n * n, out);
    HIP_CHECK(hipGetLastError());
}

// A[sel] = sqrt(c) Y
__global__ __launch_bounds__(256) void ns_finish_kernel(const double *__restrict__ Y, const double *__restrict__ scale,
                                                        const int *__restrict__ sel, long long nn, double *__restrict__ A) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < nn) A[sel[blockIdx.y] * nn + i] = sqrt(scale[blockIdx.y]) * Y[blockIdx.y * nn + i];
}
void launch_ns_finish(const double *Y, const double *scale, const int *sel, int nmat, int n, int pl, double *A,
                      hipStream_t s) {
    const long long nn = (long long)pl * n * n;
    hipLaunchKernelGGL(ns_finish_kernel, dim3(ceil_div(nn, 256), nmat), dim3(256), 0, s, Y, scale, sel, nn, A);
    HIP_CHECK(hipGetLastError());
}

__global__ void scale_rows_kernel(double *__restrict__ A, int n, const double *__restrict__ f) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n * n) return;
    A[idx] *= f[idx / n];
}
void launch_scale_rows(double *A, int n, const double *f, hipStream_t s) {
    hipLaunchKernelGGL(scale_rows_kernel, dim3(ceil_div((long long)n * n, 256)), dim3(256), 0, s, A, n, f);
    HIP_CHECK(hipGetLastError());
}

// one workgroup per (row i, matrix w): u_i (eps_ii u_i + 2 sum_{j<i} eps_ij u_j), summed into q[w]
__global__ __launch_bounds__(256) void head_quad_kernel(const double *__restrict__ A, long long stride, int ld,
                                                        const double *__restrict__ u, double *q) {
    __shared__ double red[256];
    const int i = blockIdx.x, w = blockIdx.y;
    const double *row = A + (long long)w * stride + (long long)i * ld;
    double acc = 0.0;
    for (int j = threadIdx.x; j < i; j += blockDim.x) acc += row[j] * u[j];
    acc *= 2.0;
    if (threadIdx.x == 0) acc += row[i] * u[i];
    red[threadIdx.x] = acc * u[i];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(q + w, red[0]);
}
void launch_head_quad(const double *A, long long stride, int ld, int n, int cnt, const double *u, double *q,
                      hipStream_t s) {
    hipLaunchKernelGGL(head_quad_kernel, dim3(n, cnt), dim3(256), 0, s, A, stride, ld, u, q);
    HIP_CHECK(hipGetLastError());
}

__global__ __launch_bounds__(256) void head_update_kernel(double *__restrict__ A, long long stride, int ld,
                                                          const double *__restrict__ u,
                                                          const double *__restrict__ eps_mac,
                                                          const double *__restrict__ q) {
    const int i = blockIdx.x, w = blockIdx.y;
    const double d = (eps_mac[w] - q[w]) * u[i];
    double *row = A + (long long)w * stride + (long long)i * ld;
    for (int j = threadIdx.x; j <= i; j += blockDim.x) row[j] += d * u[j];
}
void launch_head_update(double *A, long long stride, int ld, int n, int cnt, const double *u, const double *eps_mac,
                        const double *q, hipStream_t s) {
    hipLaunchKernelGGL(head_update_kernel, dim3(n, cnt), dim3(256), 0, s, A, stride, ld, u, eps_mac, q);
    HIP_CHECK(hipGetLastError());
}

}  // namespace lra
