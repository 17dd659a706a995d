// spz_mlp.hip -- bf16 MFMA kernels of the subtree-size predictor (see
// spz_mlp.h): forward, backward, Adam, and frontier prediction.
#include "spz_mlp.h"
#include "spz_board.h"

#include <vector>

namespace spz {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u); // round to nearest even
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// C(m,n) = sum_k A(m,k) B(k,n), bf16 operands, fp32 accumulate, using
// v_mfma_f32_16x16x16_bf16.  A(m,k) = A[m*sam + k*sak], B(k,n) =
// B[k*sbk + n*sbn], N columns (a multiple of 16), C row-major with leading
// dimension N.  One wave per 16x16 output tile, four waves per block along M.
// Operand layout of the instruction: lane l holds A(l%16, 4(l/16)+j) and
// B(4(l/16)+j, l%16), and receives D(4(l/16)+j, l%16), j = 0..3.  KA, KB: k is
// the operand's contiguous index (sak = 1, sbk = 1; rows 8-byte aligned), so a
// lane's four values are one load.  The products are small (1024 x 640 x 256:
// 0.3 GFLOP) and the loads' latency bounds them, so a wave has the loads of
// kGemmDeep steps in flight; the sum's order over k is that of single steps.
// Five products of a gradient over 1024 rows: 119 us with a step's loads at a
// time and a value each, now 53.
// EPI, what becomes of an element v of C: kEpiStore, c = v; kEpiAct, z = v +
// bias of its column to c and bf16(relu(z)) to cb; kEpiGrad, v where zin > 0,
// else 0, to c and in bf16 to cb.
constexpr int kGemmDeep = 8;
enum : int { kEpiStore = 0, kEpiAct = 1, kEpiGrad = 2 };
template <bool KA, bool KB, int EPI>
__global__ void __launch_bounds__(256) k_gemm_bf16(const uint16_t *__restrict__ A, int sam, int sak,
                                                   const uint16_t *__restrict__ B, int sbk, int sbn, float *c,
                                                   uint16_t *cb, const float *bias, const float *zin, int M, int N,
                                                   int K) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = (blockIdx.y * 4 + wave) * 16, n0 = blockIdx.x * 16;
    if (m0 >= M) return; // wave-uniform
    const int r = lane & 15, q = lane >> 4;
    // rows past M take the last row's values; they are not stored
    const uint16_t *a0 = A + (size_t)min(m0 + r, M - 1) * sam + (size_t)(q * 4) * sak;
    const uint16_t *b0 = B + (size_t)(n0 + r) * sbn + (size_t)(q * 4) * sbk;
    auto load = [](const uint16_t *p, int stride, bool vec) -> bf16x4 {
        bf16x4 v;
        if (vec) {
            v = *(const bf16x4 *)p;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (short)p[(size_t)j * stride];
        }
        return v;
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int k0 = 0;
    for (; k0 + 16 * kGemmDeep <= K; k0 += 16 * kGemmDeep) {
        bf16x4 a[kGemmDeep], b[kGemmDeep];
#pragma unroll
        for (int u = 0; u < kGemmDeep; ++u) {
            a[u] = load(a0 + (size_t)(k0 + 16 * u) * sak, sak, KA);
            b[u] = load(b0 + (size_t)(k0 + 16 * u) * sbk, sbk, KB);
        }
#pragma unroll
        for (int u = 0; u < kGemmDeep; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[u], b[u], acc, 0, 0, 0);
    }
    for (; k0 < K; k0 += 16) {
        bf16x4 a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool kin = k0 + q * 4 + j < K;
            a[j] = (short)(kin ? a0[(size_t)(k0 + j) * sak] : 0);
            b[j] = (short)(kin ? b0[(size_t)(k0 + j) * sbk] : 0);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = m0 + q * 4 + j, col = n0 + r;
        if (row >= M) continue;
        const size_t at = (size_t)row * N + col;
        float v = acc[j];
        if constexpr (EPI == kEpiAct) {
            v += bias[col];
            cb[at] = f2bf(v > 0.f ? v : 0.f);
        }
        if constexpr (EPI == kEpiGrad) {
            v = zin[at] > 0.f ? v : 0.f;
            cb[at] = f2bf(v);
        }
        c[at] = v;
    }
}

template <bool KA, bool KB, int EPI>
static hipError_t gemm(const uint16_t *A, int sam, int sak, const uint16_t *B, int sbk, int sbn, float *c,
                       uint16_t *cb, const float *bias, const float *zin, int M, int N, int K, hipStream_t s) {
    dim3 grid((unsigned)(N / 16), (unsigned)((M + 63) / 64));
    hipLaunchKernelGGL((k_gemm_bf16<KA, KB, EPI>), grid, dim3(256), 0, s, A, sam, sak, B, sbk, sbn, c, cb, bias, zin,
                       M, N, K);
    return hipGetLastError();
}

// features of Items at thresholds (one wave per row, 10 columns per lane);
// with perm, row r is built from items[perm[r]] (and its target copied)
template <int W>
__global__ void k_features(const Item *items, const int *thr, int n, uint16_t *x, const int *perm, const float *tgt,
                           float *tout) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    const int src = perm ? perm[row] : row;
    const Item it = items[src];
    if (perm && lane == 0) tout[row] = tgt[src];
    Board<W> bd;
    bd.unpack(it.b);
    const int h = meta_h(it.meta);
    const int L = thr[src];
    constexpr int N2 = W * W;
    for (int k = lane; k < kMlpIn; k += 64) {
        float v = 0.f;
        if (k < N2 * N2) {
            int t = k / N2, c = k - t * N2;
            v = (bd.tile(c) == t) ? 1.f : 0.f;
        } else if (k == 625) {
            v = h * (1.f / 32.f);
        } else if (k == 626) {
            v = (L - h) * (1.f / 32.f);
        }
        x[(long)row * kMlpIn + k] = f2bf(v);
    }
}

// y = h2 . w3 + b3 (one wave per row; bf16 weights, fp32 sum)
__global__ void k_out(const uint16_t *h2, const uint16_t *wbf, const float *master, float *y, int n) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    float acc = 0.f;
    for (int j = lane; j < kMlpH; j += 64) acc += bf2f(h2[(long)row * kMlpH + j]) * bf2f(wbf[kMlpOffW3 + j]);
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) y[row] = acc + master[kMlpOffB3];
}

// The output layer both ways, one wave per row: y as k_out has it, the row's
// squared error / n to e, dy = 2 (y - t) / n, and dz2[j] = dy w3[j] [z2 > 0]
// (fp32 and bf16)
__global__ void __launch_bounds__(256) k_out_loss(const uint16_t *h2, const float *z2, const uint16_t *wbf,
                                                  const float *master, const float *t, int n, float *dy, float *e,
                                                  float *dz, uint16_t *dzb) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    float acc = 0.f, w[kMlpH / 64], z[kMlpH / 64];
#pragma unroll
    for (int u = 0; u < kMlpH / 64; ++u) {
        const int j = u * 64 + lane;
        w[u] = bf2f(wbf[kMlpOffW3 + j]);
        z[u] = z2[(size_t)row * kMlpH + j];
        acc += bf2f(h2[(size_t)row * kMlpH + j]) * w[u];
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    const float d = acc + master[kMlpOffB3] - t[row];
    const float g = 2.f * d / n;
    if (lane == 0) {
        dy[row] = g;
        e[row] = d * d / n;
    }
#pragma unroll
    for (int u = 0; u < kMlpH / 64; ++u) {
        const size_t at = (size_t)row * kMlpH + u * 64 + lane;
        const float v = z[u] > 0.f ? g * w[u] : 0.f;
        dz[at] = v;
        dzb[at] = f2bf(v);
    }
}

// Column sums over n rows of 256 columns in two passes with a fixed order
// (so training is deterministic): block b sums rows [b*kSumRows, ...) into
// part[b][j], then k_grad_fin adds the parts.  Block row 1 of the grid, where
// there is one, sums bf16 a[i][j] * w[i] into part_w (the output weights'
// gradient, h2^T dy).  All of a block's loads are in flight at once: with
// those of 16 rows a sum took 11 us over 1024 rows, row after row 15, so 4.6.
constexpr int kSumRows = 64, kSumDeep = 16;
__global__ void __launch_bounds__(256) k_colsum_part(const float *a, float *part, const uint16_t *aw, const float *w,
                                                     float *part_w, int n) {
    const int j = threadIdx.x, b = blockIdx.x, i0 = b * kSumRows;
    const int rows = min(n - i0, kSumRows);
    float v[kSumRows], s = 0.f;
    if (blockIdx.y) {
#pragma unroll
        for (int u = 0; u < kSumRows; ++u) {
            const int row = i0 + min(u, rows - 1);
            v[u] = bf2f(aw[(size_t)row * kMlpH + j]) * w[row];
        }
    } else {
#pragma unroll
        for (int u = 0; u < kSumRows; ++u) v[u] = a[(size_t)(i0 + min(u, rows - 1)) * kMlpH + j];
    }
#pragma unroll
    for (int u = 0; u < kSumRows; ++u) s += u < rows ? v[u] : 0.f;
    (blockIdx.y ? part_w : part)[(size_t)b * kMlpH + j] = s;
}

// What is left of a gradient, a block each: the sums of the parts of gw3
// (block 0), gb2 (1) and gb1 (2), the output bias gradient sum dy (3) and the
// loss, sum e, added to *loss (4; `fresh`: stored).
__device__ __forceinline__ float block_sum(const float *v, int n) {
    __shared__ float sh[4];
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += v[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}
__global__ void __launch_bounds__(256) k_grad_fin(const float *part, int nparts, int part_stride, const float *dy,
                                                  const float *e, int n, float *grad, float *loss, int fresh) {
    const int j = threadIdx.x, b = blockIdx.x;
    if (b < 3) {
        const float *p = part + (size_t)b * part_stride + j;
        float s = 0.f;
        int k = 0;
        for (; k + kSumDeep <= nparts; k += kSumDeep) {
            float v[kSumDeep];
#pragma unroll
            for (int u = 0; u < kSumDeep; ++u) v[u] = p[(size_t)(k + u) * kMlpH];
#pragma unroll
            for (int u = 0; u < kSumDeep; ++u) s += v[u];
        }
        for (; k < nparts; ++k) s += p[(size_t)k * kMlpH];
        grad[(b == 0 ? kMlpOffW3 : b == 1 ? kMlpOffB2 : kMlpOffB1) + j] = s;
    } else {
        const float s = block_sum(b == 3 ? dy : e, n);
        if (j == 0) {
            if (b == 3)
                grad[kMlpOffB3] = s;
            else
                *loss = fresh ? s : *loss + s;
        }
    }
}

__global__ void k_adam(float *w, const float *g, float *m, float *v, uint16_t *wbf, long n, float lr, float b1t,
                       float b2t) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float gi = g[i];
    float mi = b1 * m[i] + (1.f - b1) * gi;
    float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    float mh = mi / (1.f - b1t), vh = vi / (1.f - b2t);
    float wi = w[i] - lr * mh / (sqrtf(vh) + eps);
    w[i] = wi;
    wbf[i] = f2bf(wi);
}

__global__ void k_to_bf16(const float *w, uint16_t *wbf, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wbf[i] = f2bf(w[i]);
}

// ---------------------------------------------------------------------------
hipError_t mlp_alloc(MlpState &m) {
    hipError_t e;
    if ((e = hipMalloc(&m.master, kMlpParams * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.wbf, kMlpParams * 2)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.grad, (kMlpParams + 1) * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.adam_m, kMlpParams * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.adam_v, kMlpParams * 4)) != hipSuccess) return e;
    m.loss = m.grad + kMlpParams;
    return hipSuccess;
}

static void fr(void *p) {
    if (p) (void)hipFree(p);
}

static void free_scratch(MlpState &m) {
    fr(m.x);
    fr(m.z1);
    fr(m.z2);
    fr(m.h1);
    fr(m.h2);
    fr(m.y);
    fr(m.dz);
    fr(m.dzb);
    fr(m.e);
    fr(m.part);
    m.part = nullptr;
    m.x = nullptr;
    m.z1 = m.z2 = nullptr;
    m.h1 = m.h2 = nullptr;
    m.y = nullptr;
    m.dz = nullptr;
    m.dzb = nullptr;
    m.e = nullptr;
    m.cap = 0;
}

void mlp_free(MlpState &m) {
    free_scratch(m);
    fr(m.master);
    fr(m.wbf);
    fr(m.grad);
    fr(m.adam_m);
    fr(m.adam_v);
    fr(m.w2frag);
    m = MlpState();
}

hipError_t mlp_reserve(MlpState &m, size_t rows) {
    if (rows <= m.cap) return hipSuccess;
    free_scratch(m);
    hipError_t e;
    if ((e = hipMalloc(&m.x, rows * kMlpIn * 2)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.z1, rows * kMlpH * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.z2, rows * kMlpH * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.h1, rows * kMlpH * 2)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.h2, rows * kMlpH * 2)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.y, rows * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.dz, rows * kMlpH * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.dzb, rows * kMlpH * 2)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.e, rows * 4)) != hipSuccess) return e;
    if ((e = hipMalloc(&m.part, 3 * ((rows + kSumRows - 1) / kSumRows) * kMlpH * 4)) != hipSuccess) return e;
    m.cap = rows;
    return hipSuccess;
}

static hipError_t refresh_bf16(MlpState &m, hipStream_t s) {
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((kMlpParams + 255) / 256)), dim3(256), 0, s, m.master, m.wbf,
                       (long)kMlpParams);
    return hipGetLastError();
}

hipError_t mlp_set_params(MlpState &m, const float *host, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(m.master, host, kMlpParams * 4, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(m.adam_m, 0, kMlpParams * 4, s);
    if (e == hipSuccess) e = hipMemsetAsync(m.adam_v, 0, kMlpParams * 4, s);
    if (e == hipSuccess) e = refresh_bf16(m, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    m.adam_t = 0;
    m.ready = (e == hipSuccess);
    return e;
}

hipError_t mlp_get_params(MlpState &m, float *host, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(host, m.master, kMlpParams * 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e;
}

// He-uniform initialisation from a seeded splitmix64 stream
hipError_t mlp_init_random(MlpState &m, uint64_t seed, hipStream_t s) {
    std::vector<float> p(kMlpParams, 0.f);
    uint64_t x = seed;
    auto next = [&]() {
        uint64_t z = (x += 0x9e3779b97f4a7c15ULL);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
        z ^= z >> 31;
        return (double)(z >> 11) / 9007199254740992.0; // [0,1)
    };
    const double a1 = sqrt(6.0 / 64.0), a2 = sqrt(6.0 / kMlpH), a3 = sqrt(6.0 / kMlpH);
    for (size_t i = 0; i < (size_t)kMlpIn * kMlpH; ++i) p[kMlpOffW1 + i] = (float)((2 * next() - 1) * a1 * 0.25);
    for (size_t i = 0; i < (size_t)kMlpH * kMlpH; ++i) p[kMlpOffW2 + i] = (float)((2 * next() - 1) * a2);
    for (int i = 0; i < kMlpH; ++i) p[kMlpOffW3 + i] = (float)((2 * next() - 1) * a3);
    for (int i = 0; i < kMlpH; ++i) p[kMlpOffB1 + i] = 0.05f;
    for (int i = 0; i < kMlpH; ++i) p[kMlpOffB2 + i] = 0.05f;
    p[kMlpOffB3] = 10.f; // log2 sizes are O(10)
    return mlp_set_params(m, p.data(), s);
}

hipError_t mlp_features_items(MlpState &m, int width, const Item *items, const int *thr, int n, hipStream_t s) {
    dim3 grid((unsigned)((n + 3) / 4));
    if (width == 4)
        hipLaunchKernelGGL((k_features<4>), grid, dim3(256), 0, s, items, thr, n, m.x, nullptr, nullptr, nullptr);
    else
        hipLaunchKernelGGL((k_features<5>), grid, dim3(256), 0, s, items, thr, n, m.x, nullptr, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t mlp_features_gather(MlpState &m, int width, const Item *items, const int *thr, const float *tgt,
                               const int *perm, int n, float *tout, hipStream_t s) {
    dim3 grid((unsigned)((n + 3) / 4));
    if (width == 4)
        hipLaunchKernelGGL((k_features<4>), grid, dim3(256), 0, s, items, thr, n, m.x, perm, tgt, tout);
    else
        hipLaunchKernelGGL((k_features<5>), grid, dim3(256), 0, s, items, thr, n, m.x, perm, tgt, tout);
    return hipGetLastError();
}

hipError_t mlp_hidden(MlpState &m, int n, hipStream_t s) {
    // z1 = x W1 + b1, h1 = relu(z1); z2 = h1 W2 + b2, h2 = relu(z2)
    const hipError_t e = gemm<true, false, kEpiAct>(m.x, kMlpIn, 1, m.wbf + kMlpOffW1, kMlpH, 1, m.z1, m.h1,
                                                    m.master + kMlpOffB1, nullptr, n, kMlpH, kMlpIn, s);
    if (e != hipSuccess) return e;
    return gemm<true, false, kEpiAct>(m.h1, kMlpH, 1, m.wbf + kMlpOffW2, kMlpH, 1, m.z2, m.h2, m.master + kMlpOffB2,
                                      nullptr, n, kMlpH, kMlpH, s);
}

hipError_t mlp_forward(MlpState &m, int n, hipStream_t s) {
    const hipError_t e = mlp_hidden(m, n, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_out, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, m.h2, m.wbf, m.master, m.y, n);
    return hipGetLastError();
}

// Weights and activations are bf16, biases fp32 (their gradients are fp32
// sums of the fp32 dz).
hipError_t mlp_backward(MlpState &m, const float *target, int n, hipStream_t s, float *loss_acc) {
    hipError_t e;
    const int nb = (n + kSumRows - 1) / kSumRows;
    const size_t part_n = (size_t)nb * kMlpH;
    float *dy = m.y;
    hipLaunchKernelGGL(k_out_loss, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, m.h2, m.z2, m.wbf, m.master, target,
                       n, dy, m.e, m.dz, m.dzb);
    // parts of gb2 = sum dz2 and gw3 = h2^T dy
    hipLaunchKernelGGL(k_colsum_part, dim3((unsigned)nb, 2), dim3(kMlpH), 0, s, m.dz, m.part + part_n, m.h2, dy,
                       m.part, n);
    // gW2 = h1^T dz2
    if ((e = gemm<false, false, kEpiStore>(m.h1, 1, kMlpH, m.dzb, kMlpH, 1, m.grad + kMlpOffW2, nullptr, nullptr,
                                           nullptr, kMlpH, kMlpH, n, s)) != hipSuccess)
        return e;
    // dz1 = dz2 W2^T [z1 > 0]: fp32 over dz2's, whose bf16 form is the
    // operand; bf16 to h2, which nothing reads any more
    uint16_t *const dz1b = m.h2;
    if ((e = gemm<true, true, kEpiGrad>(m.dzb, kMlpH, 1, m.wbf + kMlpOffW2, 1, kMlpH, m.dz, dz1b, nullptr, m.z1, n,
                                        kMlpH, kMlpH, s)) != hipSuccess)
        return e;
    // gW1 = x^T dz1; parts of gb1 = sum dz1
    if ((e = gemm<false, false, kEpiStore>(m.x, 1, kMlpIn, dz1b, kMlpH, 1, m.grad + kMlpOffW1, nullptr, nullptr,
                                           nullptr, kMlpIn, kMlpH, n, s)) != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_colsum_part, dim3((unsigned)nb, 1), dim3(kMlpH), 0, s, m.dz, m.part + 2 * part_n, nullptr,
                       nullptr, nullptr, n);
    hipLaunchKernelGGL(k_grad_fin, dim3(5), dim3(kMlpH), 0, s, m.part, nb, (int)part_n, dy, m.e, n, m.grad,
                       loss_acc ? loss_acc : m.loss, loss_acc ? 0 : 1);
    return hipGetLastError();
}

hipError_t mlp_adam_step(MlpState &m, float lr, hipStream_t s) {
    m.adam_t += 1;
    float b1t = powf(0.9f, (float)m.adam_t), b2t = powf(0.999f, (float)m.adam_t);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((kMlpParams + 255) / 256)), dim3(256), 0, s, m.master, m.grad,
                       m.adam_m, m.adam_v, m.wbf, (long)kMlpParams, lr, b1t, b2t);
    return hipGetLastError();
}

// W2 in the B-fragment order of v_mfma_f32_16x16x16_bf16: fragment
// (kb, nb) of lane l holds W2[kb*16 + 4(l/16) + j][nb*16 + l%16], j = 0..3,
// so each lane loads its 4 values as one 8-byte word.
__global__ void k_w2frag(const uint16_t *wbf, uint16_t *frag) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x; // (kb*16 + nb)*64 + lane
    if (t >= 16 * 16 * 64) return;
    const int lane = t & 63, f = t >> 6, kb = f >> 4, nb = f & 15;
    const int q = lane >> 4, r = lane & 15;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        frag[(size_t)t * 4 + j] = wbf[kMlpOffW2 + (size_t)(kb * 16 + q * 4 + j) * kMlpH + nb * 16 + r];
}

// Fused prediction: NP nodes per wave, a node's kPredThr = 16 thresholds
// L0 + 2m (m = 0..15) as the 16 rows of an MFMA tile.  Layer 1 of a row is
// the node's one-hot and h/32 columns of W1 (shared by the 16 rows) plus
// (L - h)/32 times row 626 of W1; layers 2 and 3 follow in registers.
// Waves map to node slots (g, i), g < n_groups, i < stride, NP consecutive ones
// each; a slot is live if i < count[g] (or count is null).  L0 = h of roots[g]
// if given, else thr0[g*stride + i].  Rounding follows the forward pass: bf16
// inputs and weights, fp32 sums, bf16 activations after ReLU.
//
// A wave reads all of W2, 128 KB, from L2: with a node a wave that traffic
// bounds it (6001 nodes: 0.8 GB, 61 us), so a wave takes kPredNodes nodes
// through each fragment it loads where there are enough nodes to keep every
// SIMD at work all the same (6001 nodes: 40 us; a call of 3000 takes 77 us a
// node a wave and 80 two, of 4000 90 and 85, of 20,000 308 and 239; four a wave:
// 90, 95, 238).  Layer 1's columns go four a lane, in one load each.
constexpr int kPredNodes = 2;
__device__ __forceinline__ f32x4 four(uint2 w) {
    return f32x4{bf2f((uint16_t)w.x), bf2f((uint16_t)(w.x >> 16)), bf2f((uint16_t)w.y), bf2f((uint16_t)(w.y >> 16))};
}
template <int W, int NP>
__global__ void __launch_bounds__(256) k_predict16(const Item *items, int stride, const unsigned *count, int n_groups,
                                                   const Item *roots, const int *thr0, const uint16_t *wbf,
                                                   const float *master, const uint16_t *w2frag, float *out) {
    __shared__ f32x4 base_s[4][kMlpH / 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const long slot0 = ((long)blockIdx.x * 4 + wave) * NP;
    constexpr int N2 = W * W;
    f32x4 *base = base_s[wave];
    bool live[NP], any = false; // wave-uniform
    bf16x4 a[NP][16];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        const long slot = slot0 + u;
        const int g = (int)(slot / stride), i = (int)(slot - (long)g * stride);
        live[u] = g < n_groups && (!count || (unsigned)i < count[g]);
        any |= live[u];
#pragma unroll
        for (int kb = 0; kb < 16; ++kb) a[u][kb] = bf16x4{0, 0, 0, 0};
        if (!live[u]) continue;
        const Item it = items[slot];
        Board<W> bd;
        bd.unpack(it.b);
        const int h = meta_h(it.meta);
        const int L0 = roots ? meta_h(roots[g].meta) : thr0[slot];
        const float xh = bf2f(f2bf(h * (1.f / 32.f)));
        // layer 1, shared part: sum of the one-hot rows, the h row and b1; a
        // lane has four adjacent columns
        const uint2 *w1 = (const uint2 *)(wbf + kMlpOffW1) + lane;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < N2; ++c) sum += four(w1[(bd.tile(c) * N2 + c) * (kMlpH / 4)]);
        const f32x4 wh = four(w1[625 * (kMlpH / 4)]), b1 = ((const f32x4 *)(master + kMlpOffB1))[lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] += xh * wh[j];
        base[lane] = sum + b1;
        // base is this wave's own: LDS accesses of a wave complete in order, so
        // only the compiler must keep the reads after the writes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // layer 1 rows in A-fragment order: lane l holds row m = l%16 (threshold
        // L0 + 2m), columns kb*16 + 4(l/16) + j
        const float xs = bf2f(f2bf((L0 + 2 * r - h) * (1.f / 32.f)));
        const uint2 *wl = (const uint2 *)(wbf + kMlpOffW1 + (size_t)626 * kMlpH) + q;
#pragma unroll
        for (int kb = 0; kb < 16; ++kb) {
            const f32x4 bs = base[kb * 4 + q], w = four(wl[kb * 4]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = bs[j] + xs * w[j];
                a[u][kb][j] = (short)f2bf(v > 0.f ? v : 0.f);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (!any) return;
    // layers 2 and 3: per output block nb, 16 MFMAs over K a node, then bias,
    // ReLU, bf16, and the dot product with w3 (lane holds rows 4q+j, column
    // nb*16+r)
    float part[NP][4];
#pragma unroll
    for (int u = 0; u < NP; ++u)
        for (int j = 0; j < 4; ++j) part[u][j] = 0.f;
    const uint2 *fr = (const uint2 *)w2frag + lane;
#pragma unroll 1
    for (int nb = 0; nb < 16; ++nb) {
        f32x4 acc[NP];
#pragma unroll
        for (int u = 0; u < NP; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 16; ++kb) {
            const uint2 w = fr[(kb * 16 + nb) * 64];
            bf16x4 b;
            memcpy(&b, &w, 8);
#pragma unroll
            for (int u = 0; u < NP; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[u][kb], b, acc[u], 0, 0, 0);
        }
        const int col = nb * 16 + r;
        const float b2 = master[kMlpOffB2 + col];
        const float w3 = bf2f(wbf[kMlpOffW3 + col]);
#pragma unroll
        for (int u = 0; u < NP; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float z = acc[u][j] + b2;
                part[u][j] += bf2f(f2bf(z > 0.f ? z : 0.f)) * w3;
            }
    }
    // sum over the 16 lanes holding the same rows
#pragma unroll
    for (int u = 0; u < NP; ++u) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            for (int off = 8; off > 0; off >>= 1) part[u][j] += __shfl_xor(part[u][j], off, 16);
        if (r == 0 && live[u]) {
            const float b3 = master[kMlpOffB3];
#pragma unroll
            for (int j = 0; j < 4; ++j) out[(slot0 + u) * kPredThr + q * 4 + j] = part[u][j] + b3;
        }
    }
}

// node slots from which a wave takes kPredNodes of them: two waves a SIMD
constexpr long kPredWide = 4096;

static hipError_t predict_launch(MlpState &m, int width, const Item *items, int stride, const unsigned *count,
                                 int n_groups, const Item *roots, const int *thr0, float *out, hipStream_t s) {
    hipError_t e = hipSuccess;
    if (!m.w2frag && (e = hipMalloc(&m.w2frag, (size_t)16 * 16 * 64 * 4 * 2)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_w2frag, dim3(64), dim3(256), 0, s, m.wbf, m.w2frag);
    const long slots = (long)n_groups * stride;
    const bool wide = slots >= kPredWide;
    const long waves = wide ? (slots + kPredNodes - 1) / kPredNodes : slots;
    auto *const k = width == 4 ? (wide ? &k_predict16<4, kPredNodes> : &k_predict16<4, 1>)
                               : (wide ? &k_predict16<5, kPredNodes> : &k_predict16<5, 1>);
    hipLaunchKernelGGL(k, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, items, stride, count, n_groups, roots,
                       thr0, m.wbf, m.master, m.w2frag, out);
    return hipGetLastError();
}

hipError_t mlp_predict_frontier(MlpState &m, int width, const Item *frontier, const unsigned *nfront,
                                const Item *roots, int n_inst, int capl, float *pred, hipStream_t s) {
    return predict_launch(m, width, frontier, capl, nfront, n_inst, roots, nullptr, pred, s);
}

hipError_t mlp_predict_items(MlpState &m, int width, const Item *items, const int *thr0, int n, float *out,
                             hipStream_t s) {
    return predict_launch(m, width, items, n, nullptr, 1, nullptr, thr0, out, s);
}

} // namespace spz
