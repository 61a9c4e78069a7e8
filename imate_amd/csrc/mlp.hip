// Learned surrogate of the SLQ path: a 2 -> 128 -> 128 -> 1 MLP with SiLU
// activations, trained on the GPU by hand-written forward / backward / Adam
// kernels (FP32) and evaluated by an inference kernel whose 128 x 128 layer
// runs on the matrix cores (BF16 inputs, FP32 accumulation).
//
// Parameter layout (flat FP32, kMlpParams = 17025 values):
//   W1[128][2] | b1[128] | W2[128][128] (row = output unit) | b2[128] |
//   W3[128] | b3
// Loss: mean squared error over the batch.
//
// No reference counterpart: imate's own surrogates over t are the
// interpolators (imate/interpolator, restated in imate_amd/interpolator).

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "lanes.hpp"
#include "slq_internal.hpp"

namespace slq {

namespace {

constexpr int H = 128;
constexpr int kW1 = 0;
constexpr int kB1 = kW1 + 2 * H;
constexpr int kW2 = kB1 + H;
constexpr int kB2 = kW2 + H * H;
constexpr int kW3 = kB2 + H;
constexpr int kB3 = kW3 + H;
constexpr int kMlpParams = kB3 + 1;

__device__ __forceinline__ float sigm(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigm(z); }
__device__ __forceinline__ float dsilu(float z)
{
    const float s = sigm(z);
    return s + z * s * (1.0f - s);
}

// ---------------------------------------------------------------- training

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kTrainThreads = 512;           // 8 wavefronts, 16 hidden units each
constexpr int kTrainWaves = kTrainThreads / 64;
constexpr int kTrainTiles = 1;               // 16-sample tiles a workgroup holds
constexpr int kTrainSamples = 16 * kTrainTiles;
constexpr int kTrainGroups = 256;            // most workgroups (partial gradients)
constexpr int kFirst = kTrainSamples * H / kTrainThreads;   // first-layer values per thread
constexpr int kPad = H + 4;                  // LDS row stride, see below
static_assert(kTrainWaves * 16 == H && kTrainSamples <= 64, "wavefront split");

// Samples per workgroup for a batch of B: one tile each up to half a
// workgroup per CU, then at least two (half the partial gradients to write
// and add: 96 steps at B = 4000 took 2.79 against 2.91 ms), and no more
// workgroups than CUs (64000 samples: 9.9 ms, 16.5 ms on half of the CUs).
inline int train_chunk(int B)
{
    const int tiles = (B + kTrainSamples - 1) / kTrainSamples;
    if (tiles <= kTrainGroups / 2) return kTrainSamples;
    const int per = (tiles + kTrainGroups - 1) / kTrainGroups;
    return (per > 2 ? per : 2) * kTrainSamples;
}

inline int train_groups(int B)
{
    const int chunk = train_chunk(B);
    return (B + chunk - 1) / chunk;
}

// Loss and gradient of a chunk of samples in one launch: forward,
// back-propagation and the sums over the chunk, the three 128 x 128 products
// on the FP32 matrix instruction (v_mfma_f32_16x16x4_f32: lane l holds
// A[l % 16][l / 16] and B[l / 16][l % 16], and D[4 (l / 16) + i][l % 16]).
//
// Wavefront w owns hidden units 16 w .. 16 w + 15 (columns of z2 and z1, rows
// of dW2). Its rows and its columns of W2 stay in registers; activations
// cross between wavefronts through LDS. The order of the reduction index
// within an operand is free as long as both operands agree: lane group g
// takes indices 4 g .. 4 g + 3 of each 16, which makes the reads of h1 and d2
// by row 16 bytes wide, and the row stride of 132 words keeps them, and the
// reads by column of the gradient's product, on distinct LDS banks.
//
// What bounds it: latency, not the 98 kFLOP per sample (0.2 GFLOP, 1.3 us at
// the matrix rate, for B = 2000): the loads of W2, a chain of 32 matrix
// instructions per product, four exchanges through LDS, and the 68 KB of
// sums per workgroup. 14.9 us at B = 2000 with 16 samples per workgroup
// (17.2 with 32, 25.2 with 64); a workgroup per sample for the forward pass
// and the back-propagation and a thread per parameter for the sums, which
// this replaces, took 27.2 us together and 36.8 us.
//
// A chunk's sums go to partial[chunk]; mlp_update_kernel adds the chunks in
// order, so results do not depend on scheduling. step, if given, is advanced
// here: the update of the previous step has read it, the next has not.
__global__ __launch_bounds__(kTrainThreads) void mlp_train_kernel(
    const float* __restrict__ P, const float* __restrict__ x,
    const float* __restrict__ target, int B, int chunk, float* __restrict__ partial,
    float* __restrict__ loss_partial, int* __restrict__ step)
{
    __shared__ __align__(16) float h1[kTrainSamples][kPad];
    __shared__ __align__(16) float d2[kTrainSamples][kPad];
    __shared__ float xs[kTrainSamples][2];
    __shared__ float ys[kTrainWaves][kTrainSamples];
    __shared__ float d3[kTrainSamples];
    const int lane = threadIdx.x % 64;
    const int w = threadIdx.x / 64;
    const int col = lane % 16, g = lane / 16;
    const int unit = 16 * w + col;
    const int b0 = blockIdx.x * chunk;
    const int b1 = b0 + chunk < B ? b0 + chunk : B;
    if (step && blockIdx.x == 0 && threadIdx.x == 0) *step += 1;

    // loads in the order of their use: a wait for one waits for all before it
    const int j1 = threadIdx.x % H;          // unit of the thread's first layer
    const int s1 = threadIdx.x / H;          // its samples: s1, s1 + kTrainThreads / H, ...
    float xin[kFirst][2], tin;
    const auto load_samples = [&](int b) {
        const int n = b1 - b;
#pragma unroll
        for (int i = 0; i < kFirst; ++i)
        {
            const int s = s1 + i * (kTrainThreads / H);
            xin[i][0] = s < n ? x[2 * (b + s)] : 0.f;
            xin[i][1] = s < n ? x[2 * (b + s) + 1] : 0.f;
        }
        const int s = threadIdx.x;
        tin = s < kTrainSamples && s < n ? target[b + s] : 0.f;
    };
    load_samples(b0);
    const float v1x = P[kW1 + 2 * j1], v1y = P[kW1 + 2 * j1 + 1], c1 = P[kB1 + j1];
    const float w1x = P[kW1 + 2 * unit], w1y = P[kW1 + 2 * unit + 1], bias1 = P[kB1 + unit];
    const float bias2 = P[kB2 + unit], w3 = P[kW3 + unit], bias3 = P[kB3];
    f32x4 wrow[H / 16];             // W2[unit][16 k + 4 g + 0..3]
    float wcol[H / 16][4];          // W2[16 k + 4 g + 0..3][unit]
#pragma unroll
    for (int k = 0; k < H / 16; ++k)
        wrow[k] = *(const f32x4*) (P + kW2 + unit * H + 16 * k + 4 * g);
#pragma unroll
    for (int k = 0; k < H / 16; ++k)
#pragma unroll
        for (int t = 0; t < 4; ++t) wcol[k][t] = P[kW2 + (16 * k + 4 * g + t) * H + unit];

    f32x4 gw2[H / 16] = {};
    float gw1x = 0.f, gw1y = 0.f, gb1 = 0.f, gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, loss = 0.f;
    for (int b = b0; b < b1; b += kTrainSamples)
    {
        // samples past the chunk's end count as zero in every sum
        const int n = b1 - b;
#pragma unroll
        for (int i = 0; i < kFirst; ++i)
        {
            const int s = s1 + i * (kTrainThreads / H);
            h1[s][j1] = s < n ? silu(v1x * xin[i][0] + v1y * xin[i][1] + c1) : 0.f;
            if (j1 < 2) xs[s][j1] = j1 ? xin[i][1] : xin[i][0];
        }
        const float tnow = tin;
        load_samples(b + kTrainSamples);
        __syncthreads();
        f32x4 z[kTrainTiles], sz[kTrainTiles], dz[kTrainTiles];
#pragma unroll
        for (int m = 0; m < kTrainTiles; ++m) z[m] = f32x4{bias2, bias2, bias2, bias2};
#pragma unroll
        for (int k = 0; k < H / 16; ++k)
#pragma unroll
            for (int m = 0; m < kTrainTiles; ++m)
            {
                const f32x4 a = *(const f32x4*) &h1[16 * m + col][16 * k + 4 * g];
#pragma unroll
                for (int t = 0; t < 4; ++t) z[m] = mfma(a[t], wrow[k][t], z[m]);
            }
#pragma unroll
        for (int m = 0; m < kTrainTiles; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const float s = sigm(z[m][i]);
                sz[m][i] = z[m][i] * s;
                dz[m][i] = s + z[m][i] * s * (1.0f - s);
                const float y = lanes_sum<16>(w3 * sz[m][i]);
                if (col == 0) ys[w][16 * m + 4 * g + i] = y;
            }
        __syncthreads();
        if (threadIdx.x < kTrainSamples)
        {
            const int s = threadIdx.x;
            float y = 0.f;
#pragma unroll
            for (int q = 0; q < kTrainWaves; ++q) y += ys[q][s];
            const float e = s < n ? y + bias3 - tnow : 0.f;
            loss += e * e;
            const float d = 2.0f * e / (float) B;
            gb3 += d;
            d3[s] = d;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < kTrainTiles; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int s = 16 * m + 4 * g + i;
                const float d = d3[s];
                const float v = s < n ? d * w3 * dz[m][i] : 0.f;
                d2[s][unit] = v;
                gb2 += v;
                gw3 += s < n ? d * sz[m][i] : 0.f;
            }
        __syncthreads();
        f32x4 d1[kTrainTiles] = {};
#pragma unroll
        for (int k = 0; k < H / 16; ++k)
#pragma unroll
            for (int m = 0; m < kTrainTiles; ++m)
            {
                const f32x4 a = *(const f32x4*) &d2[16 * m + col][16 * k + 4 * g];
#pragma unroll
                for (int t = 0; t < 4; ++t) d1[m] = mfma(a[t], wcol[k][t], d1[m]);
            }
#pragma unroll
        for (int m = 0; m < kTrainTiles; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int s = 16 * m + 4 * g + i;
                const float x0 = xs[s][0], x1 = xs[s][1];
                const float v =
                    s < n ? d1[m][i] * dsilu(w1x * x0 + w1y * x1 + bias1) : 0.f;
                gb1 += v;
                gw1x += v * x0;
                gw1y += v * x1;
            }
#pragma unroll
        for (int m = 0; m < kTrainTiles; ++m)
#pragma unroll
            for (int t = 0; t < 4; ++t)
            {
                const int s = 16 * m + 4 * g + t;
                const float a = d2[s][unit];
#pragma unroll
                for (int k = 0; k < H / 16; ++k) gw2[k] = mfma(a, h1[s][16 * k + col], gw2[k]);
            }
        __syncthreads();
    }

    float* out = partial + (size_t) blockIdx.x * kMlpParams;
#pragma unroll
    for (int k = 0; k < H / 16; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[kW2 + (16 * w + 4 * g + i) * H + 16 * k + col] = gw2[k][i];
    // the sums over samples of one unit are spread over the four lane groups
    float* sums[5] = {&gw1x, &gw1y, &gb1, &gb2, &gw3};
#pragma unroll
    for (int q = 0; q < 5; ++q)
    {
        *sums[q] += __shfl_xor(*sums[q], 16);
        *sums[q] += __shfl_xor(*sums[q], 32);
    }
    if (g == 0)
    {
        out[kW1 + 2 * unit] = gw1x;
        out[kW1 + 2 * unit + 1] = gw1y;
        out[kB1 + unit] = gb1;
        out[kB2 + unit] = gb2;
        out[kW3 + unit] = gw3;
    }
    if (w == 0)
    {
        gb3 = lanes_sum<64>(gb3);
        loss = lanes_sum<64>(loss);
        if (lane == 0)
        {
            out[kB3] = gb3;
            loss_partial[blockIdx.x] = loss;
        }
    }
}

constexpr int kGraphSteps = 16;
constexpr int kUpdateParams = 64;            // parameters per workgroup
constexpr int kUpdateParts = 4;              // wavefronts that share the chunks

// Sum of the chunks' gradients and, with ADAM, the step of Adam (Kingma & Ba
// 2015, bias correction) and the step's loss; the step counter lives in
// device memory so that a captured step can be replayed. Without ADAM the
// gradient goes to grad and the loss to losses[0]. A wavefront adds its part
// of the chunks for 64 parameters, eight loads in flight; the parts are added
// in order. 5.3 us at 125 chunks (8.5 MB); the sum, Adam and the counter were
// three launches of 7.9, 4.8 and 4.2 us.
template <bool ADAM>
__global__ __launch_bounds__(kUpdateParams* kUpdateParts) void mlp_update_kernel(
    const float* __restrict__ partial, const float* __restrict__ loss_partial, int groups,
    int B, float* __restrict__ grad, float* __restrict__ P, float* __restrict__ m1,
    float* __restrict__ m2, const int* __restrict__ step, float lr, float beta1,
    float beta2, float eps, float* __restrict__ losses, int max_steps)
{
    __shared__ float part[kUpdateParts][kUpdateParams];
    const int lane = threadIdx.x % kUpdateParams;
    const int w = threadIdx.x / kUpdateParams;
    const int p = blockIdx.x * kUpdateParams + lane;
    const int q = p < kMlpParams ? p : kMlpParams - 1;
    const int per = (groups + kUpdateParts - 1) / kUpdateParts;
    const int c1 = (w + 1) * per < groups ? (w + 1) * per : groups;
    float s = 0.0f;
#pragma unroll 8
    for (int c = w * per; c < c1; ++c) s += partial[(size_t) c * kMlpParams + q];
    part[w][lane] = s;
    __syncthreads();
    if (w != 0) return;
    float g = part[0][lane];
    for (int i = 1; i < kUpdateParts; ++i) g += part[i][lane];
    if (blockIdx.x == 0)
    {
        float l = 0.0f;
        for (int c = lane; c < groups; c += 64) l += loss_partial[c];
        l = lanes_sum<64>(l) / (float) B;
        const int at = ADAM ? *step - 1 : 0;
        if (lane == 0 && losses && at < max_steps) losses[at] = l;
    }
    if (p >= kMlpParams) return;
    if constexpr (ADAM)
    {
        const float t = (float) *step;
        const float a = beta1 * m1[p] + (1.0f - beta1) * g;
        const float v = beta2 * m2[p] + (1.0f - beta2) * g * g;
        m1[p] = a;
        m2[p] = v;
        const float ah = a / (1.0f - powf(beta1, t));
        const float vh = v / (1.0f - powf(beta2, t));
        P[p] -= lr * ah / (sqrtf(vh) + eps);
    }
    else
        grad[p] = g;
}

__global__ void zero_i32_kernel(int* p) { *p = 0; }

__global__ void zero_f32_kernel(float* p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// ---------------------------------------------------------------- inference

// BF16 matrix-core inference. One wavefront per 16 queries: layer 1 in FP32
// (h1 = silu(W1 x + b1)), layer 2 as 8 x 8 products of 16x16x16 BF16 tiles
// on v_mfma_f32_16x16x16_bf16 with FP32 accumulation, then silu, the dot
// with W3 and b3. Operand layout of the 16x16x16 MFMA (wave64): lane l holds
// A[l % 16][4 (l / 16) + 0..3] and B[4 (l / 16) + 0..3][l % 16]; the result
// lane l holds D[4 (l / 16) + 0..3][l % 16].
typedef short bf16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short to_bf16(float f)
{
    // round to nearest even
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    const uint32_t lsb = (u >> 16) & 1u;
    u += 0x7fffu + lsb;
    return (short) (u >> 16);
}

__global__ __launch_bounds__(256) void mlp_infer_bf16_kernel(const float* __restrict__ P,
                                                             const short* __restrict__ W2b,
                                                             const float* __restrict__ x,
                                                             int Q, float* __restrict__ y)
{
    // per wavefront: h1 tile [16 queries][128] as BF16 in LDS
    __shared__ short h1s[4][16][H];
    __shared__ float part[4][16][16];
    const int lane = threadIdx.x % 64;
    const int w = threadIdx.x / 64;
    const int q0 = (blockIdx.x * 4 + w) * 16;
    // every wavefront reaches both barriers; inactive ones skip the work
    const bool active = q0 < Q;
    if (active)
    {
        // layer 1: lane handles (query r = lane / 4, units (lane % 4) * 32 .. +31)
        const int r = lane / 4;
        const int u0 = (lane % 4) * 32;
        const int q = q0 + r;
        const float x0 = q < Q ? x[2 * q] : 0.0f;
        const float x1 = q < Q ? x[2 * q + 1] : 0.0f;
        for (int u = u0; u < u0 + 32; ++u)
        {
            const float a = P[kW1 + 2 * u] * x0 + P[kW1 + 2 * u + 1] * x1 + P[kB1 + u];
            h1s[w][r][u] = to_bf16(silu(a));
        }
    }
    __syncthreads();
    const int row = lane % 16;        // A row (query) / B,D column
    const int kq = 4 * (lane / 16);   // k offset within the 16-wide slice
    float ysum[4] = {0.f, 0.f, 0.f, 0.f};
    if (active)
    {
        for (int nb = 0; nb < H / 16; ++nb)          // output column block
        {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int kb = 0; kb < H / 16; ++kb)      // reduction block
            {
                bf16x4 a, bm;
                for (int t = 0; t < 4; ++t)
                {
                    a[t] = h1s[w][row][kb * 16 + kq + t];
                    // B[k][n] = W2[n][k]: output unit n = nb*16 + row, input k
                    bm[t] = W2b[(size_t) (nb * 16 + row) * H + kb * 16 + kq + t];
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bm, acc, 0, 0, 0);
            }
            // lane holds z2[query 4*(lane/16)+i][unit nb*16 + row]
            const int unit = nb * 16 + row;
            const float b2 = P[kB2 + unit], w3 = P[kW3 + unit];
            for (int i = 0; i < 4; ++i) ysum[i] += w3 * silu(acc[i] + b2);
        }
        // sum over the 16 columns held by lanes with the same lane / 16
        for (int i = 0; i < 4; ++i) part[w][4 * (lane / 16) + i][row] = ysum[i];
    }
    __syncthreads();
    if (active && lane < 16)
    {
        float s = P[kB3];
        for (int c = 0; c < 16; ++c) s += part[w][lane][c];
        const int q = q0 + lane;
        if (q < Q) y[q] = s;
    }
}

__global__ void to_bf16_kernel(const float* __restrict__ in, short* __restrict__ out, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = to_bf16(in[i]);
}

// FP32 inference: forward pass without storing pre-activations.
__global__ __launch_bounds__(H) void mlp_infer_f32_kernel(const float* __restrict__ P,
                                                          const float* __restrict__ x, int Q,
                                                          float* __restrict__ y)
{
    __shared__ float h1[H];
    __shared__ float red[H];
    const int b = blockIdx.x;
    const int j = threadIdx.x;
    if (b >= Q) return;
    const float x0 = x[2 * b], x1 = x[2 * b + 1];
    h1[j] = silu(P[kW1 + 2 * j] * x0 + P[kW1 + 2 * j + 1] * x1 + P[kB1 + j]);
    __syncthreads();
    float a2 = P[kB2 + j];
    const float* w = P + kW2 + (size_t) j * H;
    for (int k = 0; k < H; ++k) a2 += w[k] * h1[k];
    red[j] = P[kW3 + j] * silu(a2);
    __syncthreads();
    for (int s = H / 2; s > 0; s >>= 1)
    {
        if (j < s) red[j] += red[j + s];
        __syncthreads();
    }
    if (j == 0) y[b] = red[0] + P[kB3];
}

struct DevBuf {
    void* p = nullptr;
    ~DevBuf()
    {
        if (p) (void) hipFree(p);
    }
};

}  // namespace

}  // namespace slq

using namespace slq;

extern "C" {

int slq_mlp_num_params(void) { return kMlpParams; }

int slq_mlp_grad(const float* params, const float* x, const float* target, int32_t B,
                 float* loss, float* grad)
{
    if (!params || !x || !target || B < 1 || !grad)
    {
        set_error("slq_mlp_grad: invalid argument");
        return SLQ_E_ARG;
    }
    DevBuf dp, dx, dt, dg, dl, dpart, dlpart;
    const int C = train_groups(B);
    SLQ_CHECK(hipMalloc(&dpart.p, sizeof(float) * kMlpParams * C));
    SLQ_CHECK(hipMalloc(&dlpart.p, sizeof(float) * C));
    SLQ_CHECK(hipMalloc(&dp.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dx.p, sizeof(float) * 2 * B));
    SLQ_CHECK(hipMalloc(&dt.p, sizeof(float) * B));
    SLQ_CHECK(hipMalloc(&dg.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dl.p, sizeof(float)));
    SLQ_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    SLQ_CHECK(hipMemcpy(dx.p, x, sizeof(float) * 2 * B, hipMemcpyHostToDevice));
    SLQ_CHECK(hipMemcpy(dt.p, target, sizeof(float) * B, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(mlp_train_kernel, dim3(C), dim3(kTrainThreads), 0, 0,
                       (const float*) dp.p, (const float*) dx.p, (const float*) dt.p, B,
                       train_chunk(B), (float*) dpart.p, (float*) dlpart.p, (int*) nullptr);
    hipLaunchKernelGGL(mlp_update_kernel<false>,
                       dim3((kMlpParams + kUpdateParams - 1) / kUpdateParams),
                       dim3(kUpdateParams * kUpdateParts), 0, 0, (const float*) dpart.p,
                       (const float*) dlpart.p, C, B, (float*) dg.p, (float*) nullptr,
                       (float*) nullptr, (float*) nullptr, (const int*) nullptr, 0.f, 0.f,
                       0.f, 0.f, (float*) dl.p, 1);
    SLQ_CHECK(hipGetLastError());
    SLQ_CHECK(hipDeviceSynchronize());
    SLQ_CHECK(hipMemcpy(grad, dg.p, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
    if (loss) SLQ_CHECK(hipMemcpy(loss, dl.p, sizeof(float), hipMemcpyDeviceToHost));
    return SLQ_OK;
}

int slq_mlp_train(float* params, const float* x, const float* target, int32_t B,
                  int32_t steps, float lr, float* losses)
{
    if (!params || !x || !target || B < 1 || steps < 1 || !(lr > 0.f))
    {
        set_error("slq_mlp_train: invalid argument");
        return SLQ_E_ARG;
    }
    DevBuf dp, dx, dt, dm1, dm2, dstep, dlosses, dpart, dlpart;
    const int C = train_groups(B);
    SLQ_CHECK(hipMalloc(&dpart.p, sizeof(float) * kMlpParams * C));
    SLQ_CHECK(hipMalloc(&dlpart.p, sizeof(float) * C));
    SLQ_CHECK(hipMalloc(&dp.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dx.p, sizeof(float) * 2 * B));
    SLQ_CHECK(hipMalloc(&dt.p, sizeof(float) * B));
    SLQ_CHECK(hipMalloc(&dm1.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dm2.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dstep.p, sizeof(int)));
    SLQ_CHECK(hipMalloc(&dlosses.p, sizeof(float) * steps));
    SLQ_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    SLQ_CHECK(hipMemcpy(dx.p, x, sizeof(float) * 2 * B, hipMemcpyHostToDevice));
    SLQ_CHECK(hipMemcpy(dt.p, target, sizeof(float) * B, hipMemcpyHostToDevice));
    hipStream_t s = nullptr;
    SLQ_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    const int pg = (kMlpParams + 255) / 256;
    hipLaunchKernelGGL(zero_f32_kernel, dim3(pg), dim3(256), 0, s, (float*) dm1.p, kMlpParams);
    hipLaunchKernelGGL(zero_f32_kernel, dim3(pg), dim3(256), 0, s, (float*) dm2.p, kMlpParams);
    hipLaunchKernelGGL(zero_i32_kernel, dim3(1), dim3(1), 0, s, (int*) dstep.p);
    const auto one_step = [&] {
        hipLaunchKernelGGL(mlp_train_kernel, dim3(C), dim3(kTrainThreads), 0, s,
                           (const float*) dp.p, (const float*) dx.p, (const float*) dt.p, B,
                           train_chunk(B), (float*) dpart.p, (float*) dlpart.p,
                           (int*) dstep.p);
        hipLaunchKernelGGL(mlp_update_kernel<true>,
                           dim3((kMlpParams + kUpdateParams - 1) / kUpdateParams),
                           dim3(kUpdateParams * kUpdateParts), 0, s, (const float*) dpart.p,
                           (const float*) dlpart.p, C, B, (float*) nullptr, (float*) dp.p,
                           (float*) dm1.p, (float*) dm2.p, (const int*) dstep.p, lr, 0.9f,
                           0.999f, 1e-8f, (float*) dlosses.p, steps);
    };
    // kGraphSteps training steps, captured once and replayed; the steps
    // left over are launched one by one (so are all of a few, where the
    // capture costs more than its launches save)
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int r = SLQ_OK;
    int done = 0;
    hipError_t e = hipSuccess;
    if (steps >= 2 * kGraphSteps)
    {
        e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess)
        {
            for (int i = 0; i < kGraphSteps; ++i) one_step();
            e = hipStreamEndCapture(s, &graph);
        }
        if (e == hipSuccess) e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        for (; e == hipSuccess && steps - done >= kGraphSteps; done += kGraphSteps)
            e = hipGraphLaunch(exec, s);
    }
    for (; e == hipSuccess && done < steps; ++done)
    {
        one_step();
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) r = hip_status(e, "slq_mlp_train", __FILE__, __LINE__);
    if (exec) (void) hipGraphExecDestroy(exec);
    if (graph) (void) hipGraphDestroy(graph);
    (void) hipStreamDestroy(s);
    if (r != SLQ_OK) return r;
    SLQ_CHECK(hipMemcpy(params, dp.p, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
    if (losses)
        SLQ_CHECK(hipMemcpy(losses, dlosses.p, sizeof(float) * steps, hipMemcpyDeviceToHost));
    return SLQ_OK;
}

int slq_mlp_predict(const float* params, const float* x, int32_t Q, int32_t bf16,
                    float* y, double* seconds)
{
    if (!params || !x || Q < 1 || !y)
    {
        set_error("slq_mlp_predict: invalid argument");
        return SLQ_E_ARG;
    }
    DevBuf dp, dx, dy, dw;
    SLQ_CHECK(hipMalloc(&dp.p, sizeof(float) * kMlpParams));
    SLQ_CHECK(hipMalloc(&dx.p, sizeof(float) * 2 * Q));
    SLQ_CHECK(hipMalloc(&dy.p, sizeof(float) * Q));
    SLQ_CHECK(hipMalloc(&dw.p, sizeof(short) * H * H));
    SLQ_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    SLQ_CHECK(hipMemcpy(dx.p, x, sizeof(float) * 2 * Q, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(to_bf16_kernel, dim3((H * H + 255) / 256), dim3(256), 0, 0,
                       (const float*) dp.p + kW2, (short*) dw.p, H * H);
    SLQ_CHECK(hipDeviceSynchronize());
    hipEvent_t e0, e1;
    SLQ_CHECK(hipEventCreate(&e0));
    SLQ_CHECK(hipEventCreate(&e1));
    (void) hipEventRecord(e0, 0);
    if (bf16)
    {
        const int waves = (Q + 15) / 16;
        hipLaunchKernelGGL(mlp_infer_bf16_kernel, dim3((waves + 3) / 4), dim3(256), 0, 0,
                           (const float*) dp.p, (const short*) dw.p, (const float*) dx.p, Q,
                           (float*) dy.p);
    }
    else
        hipLaunchKernelGGL(mlp_infer_f32_kernel, dim3(Q), dim3(H), 0, 0, (const float*) dp.p,
                           (const float*) dx.p, Q, (float*) dy.p);
    (void) hipEventRecord(e1, 0);
    SLQ_CHECK(hipGetLastError());
    SLQ_CHECK(hipEventSynchronize(e1));
    float ms = 0.f;
    (void) hipEventElapsedTime(&ms, e0, e1);
    if (seconds) *seconds = ms * 1e-3;
    (void) hipEventDestroy(e0);
    (void) hipEventDestroy(e1);
    SLQ_CHECK(hipMemcpy(y, dy.p, sizeof(float) * Q, hipMemcpyDeviceToHost));
    return SLQ_OK;
}

}  // extern "C"
