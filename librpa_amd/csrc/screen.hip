// Block norms and the screener MLP (forward, backward, Adam) on gfx950.
//
// MLP, FP32: z1 = x W1 + b1, h1 = silu(z1), z2 = h1 W2 + b2, h2 = silu(z2), y = h2 w3 + b3.
// Parameter vector: W1[8][64], b1[64], W2[64][64], b2[64], w3[64], b3.
// Training: full-batch mean squared error; one kernel takes tiles of 64 samples from the forward pass
// to partial parameter gradients, a second sums those; Adam updates the parameters in place.
#include "screen.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

namespace lra {

namespace {
constexpr int OW1 = 0, OB1 = MLP_NFEAT * MLP_H, OW2 = OB1 + MLP_H, OB2 = OW2 + MLP_H * MLP_H, OW3 = OB2 + MLP_H,
              OB3 = OW3 + MLP_H;
static_assert(OB3 + 1 == MLP_NPARAM, "parameter layout");
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sig(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ __forceinline__ double block_sum(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    return s;
}
}  // namespace

template <class T>
__global__ __launch_bounds__(256) void block_norms_kernel(const T *__restrict__ base, long long ld,
                                                          const BlockRef *__restrict__ blocks, double *out) {
    __shared__ double red[4];
    const BlockRef b = blocks[blockIdx.x];
    const int n = b.rows * b.cols;
    double v = 0;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const double x = static_cast<double>(base[b.off + (long long)(e / b.cols) * ld + e % b.cols]);
        v += x * x;
    }
    const double s = block_sum(v, red);
    if (threadIdx.x == 0) out[blockIdx.x] = sqrt(s);
}

template <class T>
void launch_block_norms(const T *base, long long ld, const BlockRef *blocks, int nblocks, double *out, hipStream_t s) {
    if (nblocks <= 0) return;
    hipLaunchKernelGGL(block_norms_kernel<T>, dim3(nblocks), dim3(256), 0, s, base, ld, blocks, out);
    HIP_CHECK(hipGetLastError());
}
template void launch_block_norms<double>(const double *, long long, const BlockRef *, int, double *, hipStream_t);
template void launch_block_norms<float>(const float *, long long, const BlockRef *, int, double *, hipStream_t);

template <class T>
__global__ __launch_bounds__(256) void chi0_block_norms_kernel(const T *__restrict__ chi0s, long long E_tot,
                                                               const long long *__restrict__ eoff,
                                                               const int *__restrict__ esize, int nout,
                                                               double *out) {
    __shared__ double red[4];
    const int o = blockIdx.x, t = blockIdx.y;
    const T *p = chi0s + (long long)t * E_tot + eoff[o];
    double v = 0;
    for (int e = threadIdx.x; e < esize[o]; e += blockDim.x) {
        const double x = static_cast<double>(p[e]);
        v += x * x;
    }
    const double s = block_sum(v, red);
    if (threadIdx.x == 0) out[(long long)t * nout + o] = sqrt(s);
}

template <class T>
void launch_chi0_block_norms(const T *chi0s, long long E_tot, int ntau, const long long *eoff, const int *esize,
                             int nout, double *out, hipStream_t s) {
    if (nout <= 0 || ntau <= 0) return;
    hipLaunchKernelGGL(chi0_block_norms_kernel<T>, dim3(nout, ntau), dim3(256), 0, s, chi0s, E_tot, eoff, esize,
                       nout, out);
    HIP_CHECK(hipGetLastError());
}
template void launch_chi0_block_norms<double>(const double *, long long, int, const long long *, const int *, int,
                                              double *, hipStream_t);
template void launch_chi0_block_norms<float>(const float *, long long, int, const long long *, const int *, int,
                                             double *, hipStream_t);

__global__ __launch_bounds__(256) void mlp_forward_kernel(const float *__restrict__ params,
                                                          const float *__restrict__ X, int n, float *__restrict__ y) {
    __shared__ float P[MLP_NPARAM];
    for (int i = threadIdx.x; i < MLP_NPARAM; i += blockDim.x) P[i] = params[i];
    __syncthreads();
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    float x[MLP_NFEAT];
#pragma unroll
    for (int i = 0; i < MLP_NFEAT; ++i) x[i] = X[(long long)s * MLP_NFEAT + i];
    float h1[MLP_H];
#pragma unroll
    for (int j = 0; j < MLP_H; ++j) {
        float z = P[OB1 + j];
#pragma unroll
        for (int i = 0; i < MLP_NFEAT; ++i) z += x[i] * P[OW1 + i * MLP_H + j];
        h1[j] = z * sig(z);
    }
    float out = P[OB3];
    for (int j = 0; j < MLP_H; ++j) {
        float z = P[OB2 + j];
#pragma unroll
        for (int k = 0; k < MLP_H; ++k) z += h1[k] * P[OW2 + k * MLP_H + j];
        out += z * sig(z) * P[OW3 + j];
    }
    y[s] = out;
}

void launch_mlp_forward(const float *params, const float *X, int n, float *y, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, params, X, n, y);
    HIP_CHECK(hipGetLastError());
}

// Loss and gradient in two launches.  The first keeps a tile of 64 samples on chip from the forward
// pass to its share of every parameter's gradient, all products on the FP32 matrix units: a wave
// holds 16 samples as the columns of Z1^T, Z2^T and the deltas, and passes them from product to
// product through its own rows in LDS.  The terms are taken in the order of the hidden units: z2 and
// y are the sums that one thread per sample would form, bit by bit.  The products over samples (W1,
// b1, W2) read h1 and the deltas of all four waves; b2 and w3 are summed in registers.  A workgroup
// takes tiles blockIdx.x, + gridDim.x, ... and writes one partial gradient; the second launch adds the
// partials in FP64.
//
// Bound by the chain of one tile: 232 MFMAs a wave are 3 us, the rest is the latency of the first
// loads and of the code itself, so the products are loops.  A call on 20000 samples takes 25 us;
// with all products unrolled and registers for one workgroup a CU 31, with a thread per sample and
// activations in memory (two launches over 20 MB of them) 168.  Rows of 68 floats keep the lanes of a step
// on different banks (W2 rows in the forward product: two to a bank).
constexpr int TS = 64, LDH = MLP_H + 4, LDX = 20;

__device__ __forceinline__ v4f mfma_f32(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// sum over the 16 lanes of a lane group (every lane gets it)
__device__ __forceinline__ float row_sum(float v) {
    const auto dpp = [](float x, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v += dpp(v, std::integral_constant<int, 0xB1>());   // lane ^ 1
    v += dpp(v, std::integral_constant<int, 0x4E>());   // lane ^ 2
    v += dpp(v, std::integral_constant<int, 0x141>());  // mirror of 8 lanes
    v += dpp(v, std::integral_constant<int, 0x140>());  // mirror of 16 lanes
    return v;
}

__global__ __launch_bounds__(256, 2) void mlp_tile_grad_kernel(const float *__restrict__ params, const float *__restrict__ X,
                                                            const float *__restrict__ t, int n, int ntile,
                                                            float *__restrict__ part, double *__restrict__ lossp) {
    __shared__ __align__(16) float W2s[MLP_H * LDH], H1[TS * LDH], D1[TS * LDH], D2[TS * LDH], Xs[TS * LDX];
    __shared__ float w3s[MLP_H];
    __shared__ float red[2][4][MLP_H], red3[4];
    __shared__ double redl[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, kq = lane >> 4;
    for (int i = tid; i < MLP_H * MLP_H; i += 256) W2s[(i / MLP_H) * LDH + i % MLP_H] = params[OW2 + i];
    if (tid < MLP_H) w3s[tid] = params[OW3 + tid];
    // columns 8 to 15 of X: the ones of b1, then zeros
    for (int i = tid; i < TS * 8; i += 256) Xs[(i >> 3) * LDX + 8 + (i & 7)] = (i & 7) == 0 ? 1.0f : 0.0f;
    float w1[2][4], b1[4][4], b2[4][4], w3[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
#pragma unroll
        for (int st = 0; st < 2; ++st) w1[st][m] = params[OW1 + (4 * st + kq) * MLP_H + 16 * m + c];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 16 * m + 4 * kq + r;
            b1[m][r] = params[OB1 + j];
            b2[m][r] = params[OB2 + j];
            w3[m][r] = params[OW3 + j];
        }
    }
    const float b3 = params[OB3];
    v4f g2[4], g1 = {0, 0, 0, 0}, gb2[4], gw3[4];  // W2 rows of this wave, W1 and b1 columns of it, b2, w3
#pragma unroll
    for (int m = 0; m < 4; ++m) g2[m] = gb2[m] = gw3[m] = v4f{0, 0, 0, 0};
    float gb3 = 0;
    double loss = 0;
    for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int s = tile * TS + 16 * wave + c;
        float xb[2];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            xb[st] = s < n ? X[(long long)s * MLP_NFEAT + 4 * st + kq] : 0.0f;
            Xs[(16 * wave + c) * LDX + 4 * st + kq] = xb[st];
        }
        const float ts = s < n ? t[s] : 0.0f;
        v4f s1[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            v4f z = {b1[m][0], b1[m][1], b1[m][2], b1[m][3]};
#pragma unroll
            for (int st = 0; st < 2; ++st) z = mfma_f32(w1[st][m], xb[st], z);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float g = sig(z[r]);
                s1[m][r] = g * (1.0f + z[r] * (1.0f - g));
                z[r] *= g;
            }
            *reinterpret_cast<v4f *>(&H1[(16 * wave + c) * LDH + 16 * m + 4 * kq]) = z;
        }
        __syncthreads();
        v4f d[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) d[m] = v4f{b2[m][0], b2[m][1], b2[m][2], b2[m][3]};
#pragma unroll 4
        for (int st = 0; st < 16; ++st) {
            const float h = H1[(16 * wave + c) * LDH + 4 * st + kq];
#pragma unroll
            for (int m = 0; m < 4; ++m) d[m] = mfma_f32(W2s[(4 * st + kq) * LDH + 16 * m + c], h, d[m]);
        }
        v4f h2[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float z = d[m][r], g = sig(z);
                h2[m][r] = z * g;
                d[m][r] = g * (1.0f + z * (1.0f - g));
            }
            *reinterpret_cast<v4f *>(&D1[(16 * wave + c) * LDH + 16 * m + 4 * kq]) = h2[m];
        }
        __syncthreads();
        v4f y = {b3, b3, b3, b3};  // the same in all four rows
#pragma unroll 4
        for (int st = 0; st < 16; ++st) y = mfma_f32(w3s[4 * st + kq], D1[(16 * wave + c) * LDH + 4 * st + kq], y);
        const float res = s < n ? y[0] - ts : 0.0f;
        const float dy = 2.0f * res / (float)n;
        if (kq == 0) {
            gb3 += dy;
            loss += (double)res * (double)res;
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gw3[m][r] += s < n ? dy * h2[m][r] : 0.0f;  // (h2 of a padding lane can overflow where no sample's does)
                d[m][r] = s < n ? d[m][r] * dy * w3[m][r] : 0.0f;
                gb2[m][r] += d[m][r];
            }
            *reinterpret_cast<v4f *>(&D2[(16 * wave + c) * LDH + 16 * m + 4 * kq]) = d[m];
        }
        __syncthreads();
        // dz1 = (W2 dz2) silu'(z1)
        v4f e[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) e[m] = v4f{0, 0, 0, 0};
#pragma unroll 4
        for (int st = 0; st < 16; ++st) {
            const float x = D2[(16 * wave + c) * LDH + 4 * st + kq];
#pragma unroll
            for (int m = 0; m < 4; ++m) e[m] = mfma_f32(W2s[(16 * m + c) * LDH + 4 * st + kq], x, e[m]);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma unroll
            for (int r = 0; r < 4; ++r) e[m][r] *= s1[m][r];
            *reinterpret_cast<v4f *>(&D1[(16 * wave + c) * LDH + 16 * m + 4 * kq]) = e[m];
        }
        __syncthreads();
        // products over the tile's samples, step (q, u) over samples 16 q + 4 kq + u
#pragma unroll 1
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = 16 * q + 4 * kq + u;
                const float a = H1[k * LDH + 16 * wave + c];
#pragma unroll
                for (int m = 0; m < 4; ++m) g2[m] = mfma_f32(a, D2[k * LDH + 16 * m + c], g2[m]);
                g1 = mfma_f32(Xs[k * LDX + c], D1[k * LDH + 16 * wave + c], g1);
            }
        __syncthreads();
    }
    float *out = part + (long long)blockIdx.x * MLP_NPARAM;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 4 * kq + r;  // rows 0 to 7 of W1, then b1
        if (i <= MLP_NFEAT) out[(i < MLP_NFEAT ? OW1 + i * MLP_H : OB1) + 16 * wave + c] = g1[r];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            out[OW2 + (16 * wave + 4 * kq + r) * MLP_H + 16 * m + c] = g2[m][r];
            const float x = row_sum(gb2[m][r]), z = row_sum(gw3[m][r]);
            if (c == 0) {
                red[0][wave][16 * m + 4 * kq + r] = x;
                red[1][wave][16 * m + 4 * kq + r] = z;
            }
        }
    }
    gb3 = row_sum(gb3);
    for (int o = 8; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (lane == 0) {
        red3[wave] = gb3;
        redl[wave] = loss;
    }
    __syncthreads();
    if (tid < 2 * MLP_H) {
        const int w = tid / MLP_H, j = tid % MLP_H;
        out[(w ? OW3 : OB2) + j] = red[w][0][j] + red[w][1][j] + red[w][2][j] + red[w][3][j];
    }
    if (tid == 0) {
        out[OB3] = red3[0] + red3[1] + red3[2] + red3[3];
        lossp[blockIdx.x] = redl[0] + redl[1] + redl[2] + redl[3];
    }
}

// grad = sum of the partials, 64 parameters a workgroup, wave w the partials w, w + 16, ...; the last
// workgroup: the mean loss
__global__ __launch_bounds__(1024) void mlp_grad_sum_kernel(const float *__restrict__ part,
                                                            const double *__restrict__ lossp, int npart, int n,
                                                            float *__restrict__ grad, double *__restrict__ loss) {
    __shared__ double red[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double s = 0;
    if (blockIdx.x == gridDim.x - 1) {
        for (int i = threadIdx.x; i < npart; i += 1024) s += lossp[i];
        const double v = block_sum(s, &red[0][0]);
        if (threadIdx.x == 0) *loss = v / (double)n;
        return;
    }
    const int p = blockIdx.x * 64 + lane;
    if (p < MLP_NPARAM) {
#pragma unroll 8
        for (int i = wave; i < npart; i += 16) s += part[(long long)i * MLP_NPARAM + p];
    }
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && p < MLP_NPARAM) {
        s = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) s += red[w][lane];
        grad[p] = (float)s;
    }
}

namespace {
// at most two workgroups (of 78 KB of LDS) on each of the 256 CUs: one round, one partial each
constexpr int kMlpParts = 512;
constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t kPartBytes = align256(sizeof(float) * (size_t)kMlpParts * MLP_NPARAM);

// The two launches on caller-provided work memory of kMlpNoallocScratchBytes: partial gradients, then
// partial losses.  Every entry the second launch reads is written by the first, so the work memory
// needs no clearing.
void loss_grad_launches(const float *params, const float *X, const float *t, int n, float *grad, double *loss,
                        char *work, hipStream_t s) {
    float *part = reinterpret_cast<float *>(work);
    double *lossp = reinterpret_cast<double *>(work + kPartBytes);
    const int ntile = ceil_div(n, TS), npart = std::min(ntile, kMlpParts);
    hipLaunchKernelGGL(mlp_tile_grad_kernel, dim3(npart), dim3(256), 0, s, params, X, t, n, ntile, part, lossp);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(mlp_grad_sum_kernel, dim3(ceil_div(MLP_NPARAM, 64) + 1), dim3(1024), 0, s, part, lossp, npart, n,
                       grad, loss);
    HIP_CHECK(hipGetLastError());
}
static_assert(kPartBytes + align256(sizeof(double) * kMlpParts) == kMlpNoallocScratchBytes, "scratch size");
}  // namespace

// Work memory of the allocation-free loss and gradient (about 10 MB): each GPU the library runs
// on holds its own copy from the code object's load until the process ends.  Host code reaches it
// only through the per-device address from hipGetSymbolAddress below, never through this name.
static __device__ __align__(256) double scratch[kMlpNoallocScratchBytes / sizeof(double)];

namespace {
std::mutex g_scratch_mu;
std::map<int, char *> g_scratch_dev;  // device ordinal -> device address of scratch
}  // namespace

char *mlp_noalloc_setup() {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch_dev.find(dev);
    if (it != g_scratch_dev.end()) return it->second;
    void *p = nullptr;
    const hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (rc != hipSuccess || p == nullptr)
        LRA_THROW(std::string("hipGetSymbolAddress of the MLP scratch array failed: ") + hipGetErrorString(rc));
    g_scratch_dev[dev] = static_cast<char *>(p);
    return static_cast<char *>(p);
}

void mlp_loss_grad_noalloc(const float *params, const float *X, const float *t, int n, float *grad, double *loss,
                           hipStream_t s) {
    if (n <= 0) LRA_THROW("mlp: no samples");
    if (n > kMlpNoallocMax)
        LRA_THROW("allocation-free MLP loss/gradient: " + std::to_string(n) + " samples exceed the maximum of " +
                  std::to_string(kMlpNoallocMax));
    if (!params || !X || !t || !grad || !loss) LRA_THROW("allocation-free MLP loss/gradient: null device pointer");
    loss_grad_launches(params, X, t, n, grad, loss, mlp_noalloc_setup(), s);
}

void mlp_loss_grad(const float *params, const float *X, const float *t, int n, float *grad, double *loss,
                   MlpWork &w, hipStream_t s) {
    if (n <= 0) LRA_THROW("mlp: no samples");
    w.part.reserve(kMlpNoallocScratchBytes);
    loss_grad_launches(params, X, t, n, grad, loss, w.part.as<char>(), s);
}

__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, int n, float lr, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

void launch_adam(float *params, const float *grad, float *m, float *v, int n, float lr, int step, hipStream_t s) {
    const float c1 = 1.0f - powf(0.9f, (float)step), c2 = 1.0f - powf(0.999f, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, params, grad, m, v, n, lr, c1, c2);
    HIP_CHECK(hipGetLastError());
}

}  // namespace lra
