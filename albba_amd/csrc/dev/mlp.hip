// FP32 MLP 12 -> 32 -> 32 -> 4 (ReLU, ReLU, linear) of the learned direction
// selector: forward, mean-squared-error loss with its exact gradient, Adam,
// and the single-vector decision used inside the BFS level loop.
//
// Parameter layout (1604 floats): W1[32][12], b1[32], W2[32][32], b2[32],
// W3[4][32], b3[4]; W[j][i] multiplies input i into unit j.
//
// The gradient is computed in two deterministic passes without atomics: a
// block per chunk of 64 samples runs them forward and backward in LDS and sums
// every parameter's contributions over its chunk in sample order; then the
// chunks' partial sums are added in chunk order, and a training step updates
// the parameters in the same pass.  A run reproduces bit for bit and can be
// compared with a CPU restatement.
#include "dev_common.h"
#include "../../../include/albba.h"

namespace {

constexpr int NI = ALBBA_MLP_IN, H1 = ALBBA_MLP_H1, H2 = ALBBA_MLP_H2, NO = ALBBA_MLP_OUT;
constexpr int OW1 = 0, OB1 = OW1 + H1 * NI, OW2 = OB1 + H1, OB2 = OW2 + H2 * H1,
              OW3 = OB2 + H2, OB3 = OW3 + NO * H2, NP = OB3 + NO;
static_assert(NP == ALBBA_MLP_NPARAM, "parameter count");

__device__ __forceinline__ void load_params(const float *params, float *sp)
{
    for (int i = threadIdx.x; i < NP; i += blockDim.x) sp[i] = params[i];
    __syncthreads();
}

__device__ __forceinline__ void forward_one(const float *sp, const float *x, float *h1, float *h2,
                                            float *y)
{
    for (int j = 0; j < H1; ++j) {
        float a = sp[OB1 + j];
        for (int i = 0; i < NI; ++i) a = fmaf(sp[OW1 + j * NI + i], x[i], a);
        h1[j] = a > 0.f ? a : 0.f;
    }
    for (int j = 0; j < H2; ++j) {
        float a = sp[OB2 + j];
        for (int i = 0; i < H1; ++i) a = fmaf(sp[OW2 + j * H1 + i], h1[i], a);
        h2[j] = a > 0.f ? a : 0.f;
    }
    for (int k = 0; k < NO; ++k) {
        float a = sp[OB3 + k];
        for (int i = 0; i < H2; ++i) a = fmaf(sp[OW3 + k * H2 + i], h2[i], a);
        y[k] = a;
    }
}

__global__ __launch_bounds__(256) void k_forward(const float *params, const float *x, int32_t ns,
                                                 float *out)
{
    __shared__ float sp[NP];
    load_params(params, sp);
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ns) return;
    float xi[NI], h1[H1], h2[H2], y[NO];
    for (int i = 0; i < NI; ++i) xi[i] = x[(size_t)s * NI + i];
    forward_one(sp, xi, h1, h2, y);
    for (int k = 0; k < NO; ++k) out[(size_t)s * NO + k] = y[k];
}

// Loss and gradient of a chunk of CH samples, one block each: partial[c][p]
// for every parameter p, partial[c][NP] the chunk's squared errors.
//
// Activations and errors stay in LDS, unit-major (a unit's samples are
// consecutive), so that a thread works on one unit and four samples, or on two
// weights and four samples at a time, with 16-byte LDS reads; every sum
// runs in the order of the forward above and, over the samples, in sample
// order.  The rows are padded against bank conflicts: activations to CH + 4
// (rows stay 16-byte aligned), weights to an odd length.  Writing the
// activations to memory for a second kernel, one thread per sample with its
// vectors in scratch memory, took 23 + 13 us at 9 000 samples (141 chunks);
// this takes 10.2 us there with 512 threads and 13.4 with 256, latency of LDS
// and barriers: the arithmetic is 0.6 us.
constexpr int CH = ALBD_MLP_CHUNK;
constexpr int PS = ALBD_MLP_PARTIAL; // floats per chunk's partial sums
constexpr int LS = CH + 4;
constexpr int S1 = NI + 1, S2 = H1 + 1, S3 = H2 + 1;
static_assert(CH == 64 && H1 == 32 && H2 == 32 && NO == 4 && NI % 4 == 0, "the block's work split");
static_assert(PS >= NP + 1, "a chunk's sums");

struct ChunkLds {
    float w1[H1 * S1], b1[H1], w2[H2 * S2], b2[H2], w3[NO * S3], b3[NO];
    alignas(16) float x[NI * LS], h1[H1 * LS], h2[H2 * LS], e[NO * LS], dy[NO * LS], d1[H1 * LS], d2[H2 * LS],
        lv[LS];
};

constexpr int GT = 512;                // threads per block
constexpr int U = CH * 32 / GT;        // samples per thread
static_assert(U % 4 == 0, "16-byte reads");

// acc[u] += w * v[u]
__device__ __forceinline__ void fma_samples(float (&acc)[U], float w, const float *v)
{
#pragma unroll
    for (int u = 0; u < U; u += 4) {
        const float4 p = *reinterpret_cast<const float4 *>(v + u);
        acc[u] = fmaf(w, p.x, acc[u]);
        acc[u + 1] = fmaf(w, p.y, acc[u + 1]);
        acc[u + 2] = fmaf(w, p.z, acc[u + 2]);
        acc[u + 3] = fmaf(w, p.w, acc[u + 3]);
    }
}

// sum over the chunk's samples, in order, of a[q] * b[q]
__device__ __forceinline__ float dot_samples(const float *a, const float *b)
{
    float g = 0.f;
#pragma unroll
    for (int q = 0; q < CH; q += 4) {
        const float4 u = *reinterpret_cast<const float4 *>(a + q), v = *reinterpret_cast<const float4 *>(b + q);
        g = fmaf(u.x, v.x, g);
        g = fmaf(u.y, v.y, g);
        g = fmaf(u.z, v.z, g);
        g = fmaf(u.w, v.w, g);
    }
    return g;
}

__device__ __forceinline__ float sum_samples(const float *a)
{
    float g = 0.f;
#pragma unroll
    for (int q = 0; q < CH; q += 4) {
        const float4 u = *reinterpret_cast<const float4 *>(a + q);
        g += u.x;
        g += u.y;
        g += u.z;
        g += u.w;
    }
    return g;
}

__global__ __launch_bounds__(GT) void k_chunk_grad(const float *params, const float *x, const float *t, int32_t ns,
                                                    float *partial)
{
    __shared__ ChunkLds S;
    const int tid = threadIdx.x, c = blockIdx.x;
    const size_t s0 = (size_t)c * CH;
    const int m = (int)((size_t)ns - s0 < (size_t)CH ? (size_t)ns - s0 : (size_t)CH);
    // samples past the last one stay zero in every array, so that they add
    // nothing to the sums
    for (int i = tid; i < CH * NI; i += GT) S.x[(i % NI) * LS + i / NI] = i < m * NI ? x[s0 * NI + i] : 0.f;
    for (int i = tid; i < H1 * NI; i += GT) S.w1[(i / NI) * S1 + i % NI] = params[OW1 + i];
    for (int i = tid; i < H2 * H1; i += GT) S.w2[(i / H1) * S2 + i % H1] = params[OW2 + i];
    for (int i = tid; i < NO * H2; i += GT) S.w3[(i / H2) * S3 + i % H2] = params[OW3 + i];
    if (tid < H1) S.b1[tid] = params[OB1 + tid];
    else if (tid < H1 + H2) S.b2[tid - H1] = params[OB2 + tid - H1];
    else if (tid < H1 + H2 + NO) S.b3[tid - H1 - H2] = params[OB3 + tid - H1 - H2];
    __syncthreads();
    const int j = tid & 31, q0 = (tid >> 5) * U; // this thread's unit and samples
    float acc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = S.b1[j];
#pragma unroll
    for (int i = 0; i < NI; ++i) fma_samples(acc, S.w1[j * S1 + i], &S.x[i * LS + q0]);
#pragma unroll
    for (int u = 0; u < U; ++u) S.h1[j * LS + q0 + u] = q0 + u < m && acc[u] > 0.f ? acc[u] : 0.f;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = S.b2[j];
#pragma unroll 8
    for (int i = 0; i < H1; ++i) fma_samples(acc, S.w2[j * S2 + i], &S.h1[i * LS + q0]);
#pragma unroll
    for (int u = 0; u < U; ++u) S.h2[j * LS + q0 + u] = q0 + u < m && acc[u] > 0.f ? acc[u] : 0.f;
    __syncthreads();
    if (tid < CH * NO) {
        const int q = tid >> 2, k = tid & 3;
        float a = S.b3[k];
#pragma unroll 8
        for (int i = 0; i < H2; ++i) a = fmaf(S.w3[k * S3 + i], S.h2[i * LS + q], a);
        const float scale = 2.0f / ((float)ns * (float)NO);
        const float e = q < m ? a - t[(s0 + q) * NO + k] : 0.f;
        S.e[k * LS + q] = e;
        S.dy[k * LS + q] = q < m ? scale * e : 0.f;
    }
    __syncthreads();
    if (tid < CH) {
        float l = 0.f;
#pragma unroll
        for (int k = 0; k < NO; ++k) l = fmaf(S.e[k * LS + tid], S.e[k * LS + tid], l);
        S.lv[tid] = l;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = 0.f;
#pragma unroll
    for (int k = 0; k < NO; ++k) fma_samples(acc, S.w3[k * S3 + j], &S.dy[k * LS + q0]);
#pragma unroll
    for (int u = 0; u < U; ++u)
        S.d2[j * LS + q0 + u] = q0 + u < m && S.h2[j * LS + q0 + u] > 0.f ? acc[u] : 0.f;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = 0.f;
#pragma unroll 8
    for (int i = 0; i < H2; ++i) fma_samples(acc, S.w2[i * S2 + j], &S.d2[i * LS + q0]);
#pragma unroll
    for (int u = 0; u < U; ++u)
        S.d1[j * LS + q0 + u] = q0 + u < m && S.h1[j * LS + q0 + u] > 0.f ? acc[u] : 0.f;
    __syncthreads();
    float *out = partial + (size_t)c * PS;
    {
        // W2[jj][ii .. ii + WU - 1]
        constexpr int WU = H2 * H1 / GT;
        const int jj = tid / (H1 / WU), ii = tid % (H1 / WU) * WU;
        float g[WU];
#pragma unroll
        for (int u = 0; u < WU; ++u) g[u] = 0.f;
#pragma unroll 4
        for (int q = 0; q < CH; q += 4) {
            const float4 d = *reinterpret_cast<const float4 *>(&S.d2[jj * LS + q]);
#pragma unroll
            for (int u = 0; u < WU; ++u) {
                const float4 h = *reinterpret_cast<const float4 *>(&S.h1[(ii + u) * LS + q]);
                g[u] = fmaf(d.x, h.x, g[u]);
                g[u] = fmaf(d.y, h.y, g[u]);
                g[u] = fmaf(d.z, h.z, g[u]);
                g[u] = fmaf(d.w, h.w, g[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < WU; ++u) out[OW2 + jj * H1 + ii + u] = g[u];
    }
    constexpr int N1 = H1 * NI, N3 = NO * H2;
    for (int p = tid; p < N1 + N3 + H1 + H2 + NO + 1; p += GT) {
        int r = p;
        if (r < N1) {
            out[OW1 + r] = dot_samples(&S.d1[(r / NI) * LS], &S.x[(r % NI) * LS]);
        } else if ((r -= N1) < N3) {
            out[OW3 + r] = dot_samples(&S.dy[(r / H2) * LS], &S.h2[(r % H2) * LS]);
        } else if ((r -= N3) < H1) {
            out[OB1 + r] = sum_samples(&S.d1[r * LS]);
        } else if ((r -= H1) < H2) {
            out[OB2 + r] = sum_samples(&S.d2[r * LS]);
        } else if ((r -= H2) < NO) {
            out[OB3 + r] = sum_samples(&S.dy[r * LS]);
        } else {
            out[NP] = sum_samples(S.lv);
        }
    }
}

struct AdamArgs {
    float *params, *m, *v; // params null: no update
    float lr, b1, b2, eps, c1, c2;
};

// grad[p] = the chunks' partial sums in chunk order, loss = the mean of the
// squared errors, and with A.params the Adam step on the gradient.
//
// A sum has one addition per chunk, in order; what must not wait in turn are
// its loads.  A block takes 64 parameters: its 16 waves load the partial sums
// of 256 chunks into LDS, 16 loads in flight each, and one wave adds them.
// One thread per parameter walking the chunks took 33 us at 141 chunks, and
// Adam its own launch 5 us; this takes 4.3.  A step at 200, 9 000 and 33 000
// samples: 36, 72 and 172 us before, 12, 14 and 26 now, with the same bits.
constexpr int RT = 256; // chunks per tile

__global__ __launch_bounds__(1024) void k_reduce_adam(const float *partial, int32_t nchunks, int32_t ns, float *grad,
                                                      float *loss, AdamArgs A)
{
    __shared__ float tile[RT * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    float g = 0.f;
    for (int c0 = 0; c0 < nchunks; c0 += RT) {
        float r[RT / 16];
#pragma unroll
        for (int k = 0; k < RT / 16; ++k) {
            const int c = c0 + wave + 16 * k;
            r[k] = c < nchunks && p <= NP ? partial[(size_t)c * PS + p] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < RT / 16; ++k) tile[(wave + 16 * k) * 64 + lane] = r[k];
        __syncthreads();
        if (wave == 0) {
            const int cnt = nchunks - c0 < RT ? nchunks - c0 : RT;
            int c = 0;
            for (; c + 16 <= cnt; c += 16) {
                float v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = tile[(c + k) * 64 + lane];
#pragma unroll
                for (int k = 0; k < 16; ++k) g += v[k];
            }
            for (; c < cnt; ++c) g += tile[c * 64 + lane];
        }
        __syncthreads(); // the tile is loaded again
    }
    if (wave != 0 || p > NP) return;
    if (p == NP) {
        *loss = g / ((float)ns * (float)NO);
        return;
    }
    grad[p] = g;
    if (A.params) {
        const float mm = A.b1 * A.m[p] + (1.f - A.b1) * g;
        const float vv = A.b2 * A.v[p] + (1.f - A.b2) * g * g;
        A.m[p] = mm;
        A.v[p] = vv;
        A.params[p] -= A.lr * (mm / A.c1) / (sqrtf(vv / A.c2) + A.eps);
    }
}

int loss_grad(albd_ctx *c, const float *params, const float *x, const float *t, int32_t ns, float *scratch,
              float *grad, float *loss, const AdamArgs &A)
{
    if (ns <= 0) return albd_set_error_msg(ALBBA_EINVAL, "mlp: no samples");
    hipStream_t s = albd_stream(c);
    const int32_t nchunks = (int32_t)(((int64_t)ns + CH - 1) / CH);
    hipLaunchKernelGGL(k_chunk_grad, dim3(nchunks), dim3(GT), 0, s, params, x, t, ns, scratch);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce_adam, dim3((NP + 1 + 63) / 64), dim3(1024), 0, s, scratch, nchunks, ns, grad, loss, A);
    HIPCHK(hipGetLastError());
    return 0;
}

} // namespace

extern "C" {

int albd_mlp_forward(albd_ctx *c, const float *params, const float *x, int32_t ns, float *out)
{
    if (ns <= 0) return 0;
    hipLaunchKernelGGL(k_forward, dim3((ns + 255) / 256), dim3(256), 0, albd_stream(c), params, x, ns, out);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_mlp_loss_grad(albd_ctx *c, const float *params, const float *x, const float *t, int32_t ns,
                       float *scratch, float *grad, float *loss)
{
    return loss_grad(c, params, x, t, ns, scratch, grad, loss, AdamArgs{});
}

int albd_mlp_train_step(albd_ctx *c, float *params, const float *x, const float *t, int32_t ns, float *scratch,
                        float *grad, float *loss, float *m, float *v, float lr, float b1, float b2, float eps,
                        int32_t step)
{
    const AdamArgs A{params, m, v, lr, b1, b2, eps, 1.f - powf(b1, (float)step), 1.f - powf(b2, (float)step)};
    return loss_grad(c, params, x, t, ns, scratch, grad, loss, A);
}

} // extern "C"
