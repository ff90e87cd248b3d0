// rast_mlp.hip -- learned bin-capacity model for gfx950.
//
// A per-tile MLP in -> H -> H -> 1 (ReLU, fp32 weights and accumulation)
// predicts log(1 + queue length) of each screen tile from features available
// before binning: the previous frame's exact queue lengths (the tile and its
// 3x3 and 5x5 neighbourhoods), the previous frame's min depth and the tile
// position: all known before this frame's vertex pass, in whose launch the
// frame-time inference runs (rast_capacity.h).  Capacities
// ceil(expm1(pred) * margin) + slack let binning run in one pass; entries
// beyond a tile's capacity are re-binned exactly (rast_kernels.hip), so the
// prediction never changes the frame.  The reference has no counterpart: it
// sizes every queue to a compile-time constant (CCR/DEFINES.h:21-23).
//
// Training runs on the GPU with the kernels below: forward, backward and the
// weight gradients on the matrix cores, the gradients summed over the batch in
// a fixed order (deterministic), and Adam.  Loss: pinball (quantile tau) on
// target - pred, averaged over the batch; its gradient is checked against
// the CPU oracle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "rast_capacity.h"
#include "rast_launch.h"
#include "rast_model.h"
#include "rast_state.h"

using namespace rast;

namespace {

constexpr int F = kNumFeatures;

__host__ __device__ inline size_t num_params(int H) { return (size_t)H * F + H + (size_t)H * H + H + H + 1; }

// ---------------------------------------------------------------- features

// Training-set features of a rendered frame (tile_features: rast_capacity.h).
__global__ __launch_bounds__(256) void k_features(FrameParams fp, const uint32_t *__restrict__ prev,
                                                  const float *__restrict__ prev_depth, float *__restrict__ out)
{
    const uint32_t n = fp.tiles_x * fp.tiles_y;
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n) return;
    float f[F];
    tile_features(fp, t, prev, prev_depth, f);
    for (int q = 0; q < F; ++q) out[(size_t)t * F + q] = f[q];
}

__global__ __launch_bounds__(256) void k_targets(uint32_t n, const uint32_t *__restrict__ count,
                                                 float *__restrict__ y)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t < n) y[t] = log1pf((float)count[t]);
}

// ----------------------------------------------------------- matrix cores
//
// The kernels below run on v_mfma_f32_16x16x4f32 (fp32 in and out; A 16x4:
// lane l holds row l % 16, k = l / 16; B 4x16: lane l holds k = l / 16, column
// l % 16; D 16x16: lane l holds column l % 16, rows 4 (l / 16) + r in register
// r).  With m = l % 16 and q = l / 16, a sum over H inputs is taken in the
// steps (jc, r), each over the four inputs 16 jc + 4 q + r: both operands of
// four steps are then one 16-byte read per lane.

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma4(const float4 a, const float4 b, v4f c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

__device__ __forceinline__ float relu(float a) { return a > 0.f ? a : 0.f; }

__device__ __forceinline__ const float4 *f4(const float *p) { return reinterpret_cast<const float4 *>(p); }

// ----------------------------------------------------------------- forward

// Predictions of n samples, one wave per 16 of them (units x samples, as the
// frame-time model: layer 1's result is layer 2's B operand as it stands, so
// no activation passes through memory).  A frame's 8,160 tiles are 510 waves:
// one sample per lane left most of the chip idle behind a serial chain of
// 4.7 K multiply-adds (8,160 samples, H = 64: 51.7 -> 7.5 us).
template <int H>
__global__ __launch_bounds__(256) void k_mlp_infer(uint32_t n, const float *__restrict__ x, const float *__restrict__ p,
                                                   float *__restrict__ pred)
{
    constexpr int NJ = H / 16;
    const float *W1 = p, *b1 = W1 + H * F, *W2 = b1 + H, *b2 = W2 + H * H, *W3 = b2 + H, *b3 = W3 + H;
    const uint32_t lane = threadIdx.x & 63u, m = lane & 15u, q = lane >> 4;
    const uint32_t s0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 16u;
    if (s0 >= n) return;  // the same for the whole wave
    // the last wave's missing samples repeat the last one
    const uint32_t s = s0 + m < n ? s0 + m : n - 1u;
    const float2 xb = *reinterpret_cast<const float2 *>(x + (size_t)s * F + 2u * q);  // inputs 2q, 2q + 1
    float4 h1[NJ];
#pragma unroll
    for (int jc = 0; jc < NJ; ++jc) {
        const float2 a = *reinterpret_cast<const float2 *>(W1 + (jc * 16 + m) * F + 2u * q);
        v4f acc = { 0.f, 0.f, 0.f, 0.f };
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, xb.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, xb.y, acc, 0, 0, 0);
        const float4 b = f4(b1)[jc * 4 + q];  // units 16 jc + 4 q + r
        h1[jc] = make_float4(relu(acc[0] + b.x), relu(acc[1] + b.y), relu(acc[2] + b.z), relu(acc[3] + b.w));
    }
    float o = 0.f;
#pragma unroll
    for (int jo = 0; jo < NJ; ++jo) {
        v4f acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int jc = 0; jc < NJ; ++jc) acc = mfma4(f4(W2 + (jo * 16 + m) * H)[jc * 4 + q], h1[jc], acc);
        const float4 b = f4(b2)[jo * 4 + q], w = f4(W3)[jo * 4 + q];
        o += w.x * relu(acc[0] + b.x);
        o += w.y * relu(acc[1] + b.y);
        o += w.z * relu(acc[2] + b.z);
        o += w.w * relu(acc[3] + b.w);
    }
    // the sample's other units sit in the other three lane groups
    o += __shfl_xor(o, 16);
    o += __shfl_xor(o, 32);
    if (q == 0 && s0 + m < n) pred[s0 + m] = o + b3[0];
}

// ----------------------------------------------------------------- training

constexpr uint32_t kTrainSamples = 32;  // samples of a workgroup's round
constexpr uint32_t kTrainBlocks = 256;  // workgroups of a step at most: one per CU

// Training sample s of the step with this seed: a hash of (seed, s), in [0, N).
__device__ __forceinline__ uint32_t batch_sample(uint32_t seed, uint32_t s, uint32_t N)
{
    uint32_t x = seed ^ (s * 0x9E3779B9u);
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return (uint32_t)(((uint64_t)x * N) >> 32);
}

// Forward and backward of a step's samples: one workgroup of H / 16 waves
// takes rounds of 32 samples (workgroup b rounds b, b + gridDim.x, ...) and
// keeps its weight gradients in registers over all of them, so a step leaves
// at most kTrainBlocks partial gradients, summed in a fixed order by
// k_reduce_grad: deterministic.  Wave w owns the 16 units 16 w ..: of layer 1,
// of layer 2, of the back-propagated d1 and of the rows of both weight
// gradients; activations and deltas pass between the waves through LDS rows
// of H + 4 floats (16-byte reads of 16 rows then fall on distinct banks).
//
// kRandom: sample s is batch_sample(seed, s); else sample s itself.
// At 8,192 samples and H = 64 a step is 108 MFMAs per wave and a chain of
// loads, barriers and LDS round trips: 9.2 us.  One sample per lane of a
// 64-sample workgroup took 73 us (one wave on half of the CUs did the network,
// and 93% of the LDS accesses met bank conflicts).
template <int H, bool kRandom>
__global__ __launch_bounds__(4 * H) void k_train_partial(uint32_t B, uint32_t N, const float *__restrict__ X,
                                                         const float *__restrict__ Y, uint32_t seed,
                                                         const float *__restrict__ p, float tau,
                                                         float *__restrict__ partial)
{
    constexpr int NJ = H / 16, S = (int)kTrainSamples, NB = S / 16, LD = H + 4, NP = H * F + H + H * H + H + H + 1;
    static_assert(F == 8, "two 16-byte words of features; column 8 of the padded rows counts the samples");
    __shared__ __align__(16) float sx[S][20];  // features, 1 (0 for a missing sample), zeros
    __shared__ __align__(16) float sh1[S][LD], sd1[S][LD], sd2[S][LD];
    __shared__ float sout[NJ][S], sy[S];
    const float *W1 = p, *b1 = W1 + H * F, *W2 = b1 + H, *b2 = W2 + H * H, *W3 = b2 + H, *b3 = W3 + H;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, m = lane & 15u, q = lane >> 4;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t u0 = 16u * w + 4u * q;  // the lane's four units (register r: unit u0 + r)
    // the wave's weights in operand order: rows of W1 and W2, and columns of W2 for the way back
    const float2 w1a = *reinterpret_cast<const float2 *>(W1 + (16u * w + m) * F + 2u * q);
    float4 w2a[NJ], w2t[NJ];
#pragma unroll
    for (int jc = 0; jc < NJ; ++jc) {
        w2a[jc] = f4(W2 + (16u * w + m) * H)[jc * 4 + q];
        const float *c = W2 + (size_t)(16 * jc + 4 * q) * H + 16u * w + m;
        w2t[jc] = make_float4(c[0], c[H], c[2 * H], c[3 * H]);
    }
    const float4 b1v = f4(b1)[u0 / 4], b2v = f4(b2)[u0 / 4], w3v = f4(W3)[u0 / 4];
    const float bias1[4] = { b1v.x, b1v.y, b1v.z, b1v.w }, bias2[4] = { b2v.x, b2v.y, b2v.z, b2v.w };
    const float w3[4] = { w3v.x, w3v.y, w3v.z, w3v.w };
    const float b3v = b3[0];

    v4f gW2[NJ], gW1 = { 0.f, 0.f, 0.f, 0.f };
    float gW3[4] = {}, gb2[4] = {}, gb3 = 0.f, loss = 0.f;
#pragma unroll
    for (int k = 0; k < NJ; ++k) gW2[k] = v4f{ 0.f, 0.f, 0.f, 0.f };

    for (uint32_t base = blockIdx.x * (uint32_t)S; base < B; base += gridDim.x * (uint32_t)S) {
        __syncthreads();  // the previous round's rows are read
        if (tid < 2u * S) {
            const uint32_t r = tid >> 1, half = tid & 1u, s = base + r;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            float y = 0.f;
            if (s < B) {
                const uint32_t src = kRandom ? batch_sample(seed, s, N) : s;
                v = f4(X + (size_t)src * F)[half];
                if (half == 0) y = Y[src];
            }
            *reinterpret_cast<float4 *>(&sx[r][4 * half]) = v;
            *reinterpret_cast<float4 *>(&sx[r][8 + 4 * half]) = make_float4(half == 0 && s < B ? 1.f : 0.f, 0.f, 0.f, 0.f);
            if (half == 0) sy[r] = y;
        }
        __syncthreads();
        float h1[NB][4], h2[NB][4];
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
            const float2 xb = *reinterpret_cast<const float2 *>(&sx[16 * sb + m][2u * q]);
            v4f acc = { 0.f, 0.f, 0.f, 0.f };
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w1a.x, xb.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w1a.y, xb.y, acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) h1[sb][r] = relu(acc[r] + bias1[r]);
            *reinterpret_cast<float4 *>(&sh1[16 * sb + m][u0]) = make_float4(h1[sb][0], h1[sb][1], h1[sb][2], h1[sb][3]);
        }
        __syncthreads();
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
            v4f acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int jc = 0; jc < NJ; ++jc) acc = mfma4(w2a[jc], f4(&sh1[16 * sb + m][0])[jc * 4 + q], acc);
            float o = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h2[sb][r] = relu(acc[r] + bias2[r]);
                o += w3[r] * h2[sb][r];
            }
            o += __shfl_xor(o, 16);
            o += __shfl_xor(o, 32);
            if (q == 0) sout[w][16 * sb + m] = o;
        }
        __syncthreads();
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
            const uint32_t r0 = 16 * sb + m;
            float out = b3v;
#pragma unroll
            for (int k = 0; k < NJ; ++k) out += sout[k][r0];
            const float r = sy[r0] - out;
            const bool live = base + r0 < B;
            const float g = live ? (r > 0.f ? -tau : 1.f - tau) / (float)B : 0.f;
            float d2[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                d2[k] = h2[sb][k] > 0.f ? g * w3[k] : 0.f;
                gW3[k] += g * h2[sb][k];
                gb2[k] += d2[k];
            }
            gb3 += g;
            loss += live ? (r > 0.f ? tau * r : (tau - 1.f) * r) : 0.f;
            *reinterpret_cast<float4 *>(&sd2[r0][u0]) = make_float4(d2[0], d2[1], d2[2], d2[3]);
        }
        __syncthreads();
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
            v4f acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int jc = 0; jc < NJ; ++jc) acc = mfma4(w2t[jc], f4(&sd2[16 * sb + m][0])[jc * 4 + q], acc);
            float d1[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) d1[r] = h1[sb][r] > 0.f ? acc[r] : 0.f;
            *reinterpret_cast<float4 *>(&sd1[16 * sb + m][u0]) = make_float4(d1[0], d1[1], d1[2], d1[3]);
        }
        __syncthreads();
        // weight gradients: sums over the samples, four (4 t + q) a step; column 8 of sx gives gb1
#pragma unroll
        for (int t = 0; t < S / 4; ++t) {
            const float a2 = sd2[4 * t + q][16u * w + m], a1 = sd1[4 * t + q][16u * w + m];
#pragma unroll
            for (int k = 0; k < NJ; ++k)
                gW2[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, sh1[4 * t + q][16 * k + m], gW2[k], 0, 0, 0);
            gW1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, sx[4 * t + q][m], gW1, 0, 0, 0);
        }
    }

    float *out = partial + (size_t)blockIdx.x * (NP + 1);
    float *oW1 = out, *ob1 = oW1 + H * F, *oW2 = ob1 + H, *ob2 = oW2 + H * H, *oW3 = ob2 + H, *ob3 = oW3 + H;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int k = 0; k < NJ; ++k) oW2[(u0 + r) * H + 16 * k + m] = gW2[k][r];
        if (m < (uint32_t)F) oW1[(u0 + r) * F + m] = gW1[r];
        if (m == (uint32_t)F) ob1[u0 + r] = gW1[r];
    }
    // over the 16 samples of a lane group
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            gb2[r] += __shfl_xor(gb2[r], o);
            gW3[r] += __shfl_xor(gW3[r], o);
        }
        gb3 += __shfl_xor(gb3, o);
        loss += __shfl_xor(loss, o);
    }
    if (m == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ob2[u0 + r] = gb2[r];
            oW3[u0 + r] = gW3[r];
        }
    }
    if (tid == 0) {
        ob3[0] = gb3;
        out[NP] = loss;
    }
}

// grad[i] = the sum of partial[b][i] over the workgroups b, in a fixed order;
// loss = mean.  A workgroup takes 64 parameters (one per lane), its 16 waves
// every 16th partial each: the loads of a wave are independent of each other.
// 256 partials of 4,801 parameters: 3.8 us with the Adam step (one thread per
// parameter over 128 of them took 29.6 us, Adam 4.7 us in a launch of its own).
// kAdam: the parameters' Adam step with that gradient, in the same launch.
template <bool kAdam>
__global__ __launch_bounds__(1024) void k_reduce_grad(uint32_t nblocks, uint32_t np, uint32_t B,
                                                      const float *__restrict__ partial, float *__restrict__ grad,
                                                      float *__restrict__ loss, float *__restrict__ p,
                                                      float *__restrict__ m, float *__restrict__ v, float lr, float b1c,
                                                      float b2c)
{
    __shared__ float red[16][64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, i = blockIdx.x * 64u + lane;
    float a = 0.f;
    if (i <= np) {
#pragma unroll 8
        for (uint32_t b = wave; b < nblocks; b += 16u) a += partial[(size_t)b * (np + 1) + i];
    }
    red[wave][lane] = a;
    __syncthreads();
    if (wave != 0 || i > np) return;
    a = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) a += red[k][lane];
    if (i == np) {
        loss[0] = a / (float)B;
        return;
    }
    if constexpr (kAdam) {
        const float mi = 0.9f * m[i] + 0.1f * a;
        const float vi = 0.999f * v[i] + 0.001f * a * a;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / b1c) / (sqrtf(vi / b2c) + 1e-8f);
    } else {
        grad[i] = a;
    }
}

uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

}  // namespace

// ------------------------------------------------------------------ object

struct rast_binmodel {
    int device = 0;
    int H = 64;
    hipStream_t stream = nullptr;    // home's; the model's own once that renderer is gone
    rast_renderer *home = nullptr;   // the renderer it was created on, while that exists
    DBuf params, grad, adam_m, adam_v;
    DBuf X, Y;            // recorded training set
    uint32_t n = 0, cap = 0;
    DBuf partial, loss, io_x, io_y, io_p;  // partial: per workgroup gradients + loss
    uint32_t batch_cap = 0;
    uint64_t adam_t = 0;
    std::vector<rast_renderer *> users;  // the renderers it is attached to
};

// Guards every model's users and home, and every renderer's models: a model
// serves renderers that different threads may attach and destroy.
static std::mutex g_models_mutex;

namespace rast_detail {

int ensure(DBuf &b, size_t bytes)
{
    if (b.p && b.n >= bytes) return RAST_OK;
    dfree(b);
    HIP_TRY(rast_dev_malloc(&b.p, bytes < 256 ? 256 : bytes));
    b.n = bytes < 256 ? 256 : bytes;
    return RAST_OK;
}

int launch_infer(int H, uint32_t n, const float *x, const float *p, float *pred, hipStream_t s)
{
    const dim3 g(cdiv(n, 64)), b(256);
    switch (H) {
    case 16: hipLaunchKernelGGL(k_mlp_infer<16>, g, b, 0, s, n, x, p, pred); break;
    case 32: hipLaunchKernelGGL(k_mlp_infer<32>, g, b, 0, s, n, x, p, pred); break;
    case 64: hipLaunchKernelGGL(k_mlp_infer<64>, g, b, 0, s, n, x, p, pred); break;
    default: return rast_set_error(RAST_E_INVALID_ARG, "hidden size %d not in {16, 32, 64}", H);
    }
    HIP_TRY(hipGetLastError());
    return RAST_OK;
}

constexpr uint32_t kMaxBatch = 1u << 16;

uint32_t train_blocks(uint32_t B) { return std::min(cdiv(B, kTrainSamples), kTrainBlocks); }

int ensure_batch(rast_binmodel *m, uint32_t B)
{
    if (B <= m->batch_cap) return RAST_OK;
    RAST_TRY(ensure(m->partial, train_blocks(B) * (num_params(m->H) + 1) * 4));
    RAST_TRY(ensure(m->loss, 64));
    m->batch_cap = B;
    return RAST_OK;
}

// One forward/backward over B samples of (X, Y): the partial gradients of
// train_blocks(B) workgroups.  kRandom: B samples drawn from the N by seed.
template <bool kRandom>
int train_partial(rast_binmodel *m, uint32_t B, uint32_t N, const float *X, const float *Y, uint32_t seed, float tau)
{
    if (B == 0 || B > kMaxBatch) return rast_set_error(RAST_E_INVALID_ARG, "batch %u not in [1, %u]", B, kMaxBatch);
    RAST_TRY(ensure_batch(m, B));
    const dim3 g(train_blocks(B)), b(4 * m->H);
    const float *p = (const float *)m->params.p;
    float *part = (float *)m->partial.p;
    switch (m->H) {
    case 16: hipLaunchKernelGGL((k_train_partial<16, kRandom>), g, b, 0, m->stream, B, N, X, Y, seed, p, tau, part); break;
    case 32: hipLaunchKernelGGL((k_train_partial<32, kRandom>), g, b, 0, m->stream, B, N, X, Y, seed, p, tau, part); break;
    default: hipLaunchKernelGGL((k_train_partial<64, kRandom>), g, b, 0, m->stream, B, N, X, Y, seed, p, tau, part); break;
    }
    HIP_TRY(hipGetLastError());
    return RAST_OK;
}

// Sums the partial gradients of a B-sample step into grad and loss.
int reduce_grad(rast_binmodel *m, uint32_t B)
{
    const uint32_t np = (uint32_t)num_params(m->H);
    hipLaunchKernelGGL(k_reduce_grad<false>, dim3(cdiv(np + 1, 64)), dim3(1024), 0, m->stream, train_blocks(B), np, B,
                       (const float *)m->partial.p, (float *)m->grad.p, (float *)m->loss.p, (float *)nullptr,
                       (float *)nullptr, (float *)nullptr, 0.f, 1.f, 1.f);
    HIP_TRY(hipGetLastError());
    return RAST_OK;
}

// The same sum and the Adam step with it.
int reduce_adam(rast_binmodel *m, uint32_t B, float lr, float b1c, float b2c)
{
    const uint32_t np = (uint32_t)num_params(m->H);
    hipLaunchKernelGGL(k_reduce_grad<true>, dim3(cdiv(np + 1, 64)), dim3(1024), 0, m->stream, train_blocks(B), np, B,
                       (const float *)m->partial.p, (float *)m->grad.p, (float *)m->loss.p, (float *)m->params.p,
                       (float *)m->adam_m.p, (float *)m->adam_v.p, lr, b1c, b2c);
    HIP_TRY(hipGetLastError());
    return RAST_OK;
}

}  // namespace rast_detail

using namespace rast_detail;

namespace rast {
hipError_t launch_tile_features(const FrameParams &fp, const uint32_t *prev_count, const float *prev_depth,
                                float *features, hipStream_t s)
{
    const uint32_t n = fp.tiles_x * fp.tiles_y;
    hipLaunchKernelGGL(k_features, dim3(cdiv(n, 256)), dim3(256), 0, s, fp, prev_count, prev_depth, features);
    return hipGetLastError();
}
}  // namespace rast


// r is no longer one of its model's users (g_models_mutex is held).
static void forget_user(rast_renderer *r)
{
    if (!r->model) return;
    auto &u = r->model->users;
    u.erase(std::remove(u.begin(), u.end(), r), u.end());
    r->model = nullptr;
}

int rast_model_attach(rast_renderer *r, rast_binmodel *m)
{
    if (r->model == m) return RAST_OK;
    if (r->model) {  // frames still queued read it, and it may be destroyed from here on
        HIP_TRY(hipSetDevice(r->device));
        RAST_TRY(rast_settle(r));
    }
    std::lock_guard<std::mutex> lock(g_models_mutex);
    try {
        if (m) m->users.push_back(r);
    } catch (const std::bad_alloc &) {
        return rast_set_error(RAST_E_OUT_OF_MEMORY, "host allocation failed");
    }
    forget_user(r);
    r->model = m;
    return RAST_OK;
}

void rast_model_renderer_gone(rast_renderer *r)
{
    std::lock_guard<std::mutex> lock(g_models_mutex);
    forget_user(r);
    for (rast_binmodel *m : r->models) {
        m->home = nullptr;
        m->stream = nullptr;  // made by its next use (model_ready)
    }
    r->models.clear();
}

// Makes the model's device current and sees that it has a stream.
static int model_ready(rast_binmodel *m)
{
    HIP_TRY(hipSetDevice(m->device));
    if (!m->stream) HIP_TRY(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    return RAST_OK;
}

// --------------------------------------------------------------------- ABI

extern "C" int rast_binmodel_num_features(void) { return F; }

static void init_params(std::vector<float> &p, int H, uint32_t seed)
{
    uint32_t state = seed * 2654435761u + 12345u;
    auto next = [&]() {
        state ^= state << 13; state ^= state >> 17; state ^= state << 5;
        return (float)(state >> 8) * (1.0f / 16777216.0f);
    };
    size_t o = 0;
    const float a1 = std::sqrt(6.0f / F), a2 = std::sqrt(6.0f / H), a3 = std::sqrt(3.0f / H);
    for (int i = 0; i < H * F; ++i) p[o++] = (2.f * next() - 1.f) * a1;
    for (int i = 0; i < H; ++i) p[o++] = 0.01f;
    for (int i = 0; i < H * H; ++i) p[o++] = (2.f * next() - 1.f) * a2;
    for (int i = 0; i < H; ++i) p[o++] = 0.01f;
    for (int i = 0; i < H; ++i) p[o++] = (2.f * next() - 1.f) * a3;
    p[o++] = 1.0f;
}

extern "C" int rast_binmodel_create(rast_renderer *r, uint32_t hidden, uint32_t seed, rast_binmodel **out)
try {
    if (!out) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_create: null output");
    *out = nullptr;
    if (!r) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_create: null renderer");
    if (hidden != 16 && hidden != 32 && hidden != 64)
        return rast_set_error(RAST_E_INVALID_ARG, "hidden size %u not in {16, 32, 64}", hidden);
    HIP_TRY(hipSetDevice(r->device));
    const size_t np = num_params((int)hidden);
    std::vector<float> p(np);
    init_params(p, (int)hidden, seed);
    rast_binmodel *m = new (std::nothrow) rast_binmodel();
    if (!m) return rast_set_error(RAST_E_OUT_OF_MEMORY, "host allocation failed");
    m->device = r->device;
    m->H = (int)hidden;
    try {
        std::lock_guard<std::mutex> lock(g_models_mutex);
        r->models.push_back(m);
    } catch (const std::bad_alloc &) {
        delete m;
        return rast_set_error(RAST_E_OUT_OF_MEMORY, "host allocation failed");
    }
    m->home = r;
    m->stream = r->stream;
    int rc = ensure(m->params, np * 4);
    if (rc == RAST_OK) rc = ensure(m->grad, np * 4);
    if (rc == RAST_OK) rc = ensure(m->adam_m, np * 4);
    if (rc == RAST_OK) rc = ensure(m->adam_v, np * 4);
    if (rc == RAST_OK && hipMemcpy(m->params.p, p.data(), np * 4, hipMemcpyHostToDevice) != hipSuccess) rc = RAST_E_HIP;
    if (rc == RAST_OK && hipMemset(m->adam_m.p, 0, np * 4) != hipSuccess) rc = RAST_E_HIP;
    if (rc == RAST_OK && hipMemset(m->adam_v.p, 0, np * 4) != hipSuccess) rc = RAST_E_HIP;
    if (rc != RAST_OK) {
        (void)hipGetLastError();
        rast_binmodel_destroy(m);
        return rast_set_error(rc, "rast_binmodel_create: allocation failed");
    }
    *out = m;
    return RAST_OK;
} RAST_CATCH

extern "C" int rast_binmodel_destroy(rast_binmodel *m)
{
    if (!m) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_destroy: null model");
    (void)hipSetDevice(m->device);
    {
        std::lock_guard<std::mutex> lock(g_models_mutex);
        for (rast_renderer *r : m->users) {
            (void)rast_settle(r);
            r->model = nullptr;
        }
        if (m->home) {
            (void)rast_settle(m->home);
            auto &v = m->home->models;
            v.erase(std::remove(v.begin(), v.end(), m), v.end());
        }
    }
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    if (m->stream && !m->home) (void)hipStreamDestroy(m->stream);
    DBuf *bufs[] = { &m->params, &m->grad, &m->adam_m, &m->adam_v, &m->X, &m->Y, &m->partial, &m->loss,
                     &m->io_x, &m->io_y, &m->io_p };
    for (DBuf *b : bufs) dfree(*b);
    delete m;
    return RAST_OK;
}

extern "C" int rast_binmodel_num_params(rast_binmodel *m, size_t *out)
{
    if (!m || !out) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_num_params: null argument");
    *out = num_params(m->H);
    return RAST_OK;
}

extern "C" int rast_binmodel_get_params(rast_binmodel *m, float *dst, size_t count)
{
    if (!m || !dst || count != num_params(m->H))
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_get_params: bad arguments");
    RAST_TRY(model_ready(m));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(dst, m->params.p, count * 4, hipMemcpyDeviceToHost));
    return RAST_OK;
}

extern "C" int rast_binmodel_set_params(rast_binmodel *m, const float *src, size_t count)
try {
    if (!m || !src || count != num_params(m->H))
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_set_params: bad arguments");
    RAST_TRY(model_ready(m));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(m->params.p, src, count * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(m->adam_m.p, 0, count * 4));
    HIP_TRY(hipMemset(m->adam_v.p, 0, count * 4));
    m->adam_t = 0;
    return RAST_OK;
} RAST_CATCH

extern "C" int rast_binmodel_clear_data(rast_binmodel *m)
{
    if (!m) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_clear_data: null model");
    m->n = 0;
    return RAST_OK;
}

extern "C" int rast_binmodel_record(rast_binmodel *m, rast_renderer *r)
try {
    if (!m || !r) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_record: null argument");
    RAST_TRY(rast_sync(r));
    if (!r->frame_valid || !r->frame_had_prev || r->model != m)
        return rast_set_error(RAST_E_STATE,
                              "rast_binmodel_record: needs two consecutive frames rendered with this model attached");
    RAST_TRY(model_ready(m));
    const uint32_t tx = (r->W + r->tile - 1) / r->tile, ty = (r->H + r->tile - 1) / r->tile, nt = tx * ty;
    if ((uint64_t)m->n + nt > 0x7FFFFFFFull) return rast_set_error(RAST_E_STATE, "training set full");
    if (m->n + nt > m->cap) {
        const uint32_t ncap = std::max<uint32_t>(m->cap * 2, m->n + nt);
        DBuf nx, ny;
        if (rast_dev_malloc(&nx.p, (size_t)ncap * F * 4) != hipSuccess) return rast_set_error(RAST_E_OUT_OF_MEMORY, "training set");
        nx.n = (size_t)ncap * F * 4;
        if (rast_dev_malloc(&ny.p, (size_t)ncap * 4) != hipSuccess) {
            dfree(nx);
            return rast_set_error(RAST_E_OUT_OF_MEMORY, "training set");
        }
        ny.n = (size_t)ncap * 4;
        if (m->n) {
            HIP_TRY(hipMemcpy(nx.p, m->X.p, (size_t)m->n * F * 4, hipMemcpyDeviceToDevice));
            HIP_TRY(hipMemcpy(ny.p, m->Y.p, (size_t)m->n * 4, hipMemcpyDeviceToDevice));
        }
        dfree(m->X);
        dfree(m->Y);
        m->X = nx;
        m->Y = ny;
        m->cap = ncap;
    }
    // features of the frame just rendered (the previous frame's counts and
    // depths); target: this frame's exact counts
    FrameParams fp{};
    fp.tiles_x = tx;
    fp.tiles_y = ty;
    const int last = r->cur ^ 1, before = r->cur;
    float *xdst = (float *)m->X.p + (size_t)m->n * F;
    float *ydst = (float *)m->Y.p + (size_t)m->n;
    HIP_TRY(launch_tile_features(fp, (const uint32_t *)r->tile_count[before].p, (const float *)r->tile_min_depth[before].p, xdst,
                                 r->stream));
    hipLaunchKernelGGL(k_targets, dim3(cdiv(nt, 256)), dim3(256), 0, r->stream, nt,
                       (const uint32_t *)r->tile_count[last].p, ydst);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(r->stream));
    m->n += nt;
    return RAST_OK;
} RAST_CATCH

extern "C" int rast_binmodel_train(rast_binmodel *m, uint32_t epochs, uint32_t batch, float lr, float tau,
                                   float *final_loss)
try {
    if (!m || batch == 0 || batch > kMaxBatch || !(lr > 0.f) || !(tau > 0.f && tau < 1.f))
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_train: bad arguments");
    if (m->n == 0) return rast_set_error(RAST_E_STATE, "rast_binmodel_train: no recorded data");
    RAST_TRY(model_ready(m));
    RAST_TRY(ensure_batch(m, batch));
    const uint32_t steps = std::max<uint32_t>(1, (uint32_t)(((uint64_t)m->n * epochs + batch - 1) / batch));
    for (uint32_t st = 0; st < steps; ++st) {
        const uint32_t seed = (uint32_t)(m->adam_t * 0x9E3779B1ull + 7u);
        RAST_TRY(train_partial<true>(m, batch, m->n, (const float *)m->X.p, (const float *)m->Y.p, seed, tau));
        ++m->adam_t;
        const float b1c = 1.f - std::pow(0.9f, (float)m->adam_t), b2c = 1.f - std::pow(0.999f, (float)m->adam_t);
        RAST_TRY(reduce_adam(m, batch, lr, b1c, b2c));
    }
    HIP_TRY(hipStreamSynchronize(m->stream));
    if (final_loss) HIP_TRY(hipMemcpy(final_loss, m->loss.p, 4, hipMemcpyDeviceToHost));
    return RAST_OK;
} RAST_CATCH

extern "C" int rast_binmodel_forward(rast_binmodel *m, const float *x, uint32_t n, float *pred)
try {
    if (!m || !x || !pred || n == 0) return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_forward: bad arguments");
    RAST_TRY(model_ready(m));
    RAST_TRY(ensure(m->io_x, (size_t)n * F * 4));
    RAST_TRY(ensure(m->io_p, (size_t)n * 4));
    HIP_TRY(hipMemcpy(m->io_x.p, x, (size_t)n * F * 4, hipMemcpyHostToDevice));
    RAST_TRY(launch_infer(m->H, n, (const float *)m->io_x.p, (const float *)m->params.p,
                          (float *)m->io_p.p, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(pred, m->io_p.p, (size_t)n * 4, hipMemcpyDeviceToHost));
    return RAST_OK;
} RAST_CATCH

// ------------------------------------------------ allocation-free forward

// Device staging of rast_binmodel_forward_noalloc: at most
// kNoAllocMaxSamples samples (F floats each) and their predictions, 2.25 MiB
// on every GPU the library runs on, held until the process ends.  In host
// code this name is not a device address: the array's address on a device is
// read once with hipGetSymbolAddress (that device current) and used instead.
constexpr uint32_t kNoAllocMaxSamples = 1u << 16;
static __device__ __align__(256) float scratch[(size_t)kNoAllocMaxSamples * (kNumFeatures + 1)];

namespace {

constexpr int kNoAllocDevices = 64;

// Per-device address of `scratch`, and the lock that keeps calls on one GPU
// from overlapping (they share that GPU's array).
struct NoAllocState {
    std::mutex mu;
    float *ptr[kNoAllocDevices] = {};
};
NoAllocState g_noalloc;

// The calling thread holds g_noalloc.mu and has made `device` current.
int noalloc_scratch(int device, float **out)
{
    if (device < 0 || device >= kNoAllocDevices)
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_forward_noalloc: device %d above %d", device,
                              kNoAllocDevices - 1);
    if (!g_noalloc.ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return rast_set_error(RAST_E_HIP, "rast_binmodel_forward_noalloc: hipGetSymbolAddress(scratch): %s",
                                  hipGetErrorString(e));
        g_noalloc.ptr[device] = (float *)p;
    }
    *out = g_noalloc.ptr[device];
    return RAST_OK;
}

}  // namespace

extern "C" int rast_binmodel_forward_noalloc(rast_binmodel *m, const float *x, uint32_t n, float *pred)
try {
    if (!m || !x || !pred || n == 0)
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_forward_noalloc: bad arguments");
    if (n > kNoAllocMaxSamples)
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_forward_noalloc: %u samples above the maximum %u", n,
                              kNoAllocMaxSamples);
    std::lock_guard<std::mutex> lock(g_noalloc.mu);
    RAST_TRY(model_ready(m));
    float *base = nullptr;
    RAST_TRY(noalloc_scratch(m->device, &base));
    float *sx = base, *sp = base + (size_t)kNoAllocMaxSamples * F;
    // every word the kernel reads is written first: nothing to clear
    HIP_TRY(hipMemcpyAsync(sx, x, (size_t)n * F * 4, hipMemcpyHostToDevice, m->stream));
    RAST_TRY(launch_infer(m->H, n, sx, (const float *)m->params.p, sp, m->stream));
    HIP_TRY(hipMemcpyAsync(pred, sp, (size_t)n * 4, hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    return RAST_OK;
} RAST_CATCH

extern "C" int rast_binmodel_loss_grad(rast_binmodel *m, const float *x, const float *target, uint32_t n, float tau,
                                       float *loss, float *grad)
try {
    if (!m || !x || !target || !grad || n == 0 || n > kMaxBatch)
        return rast_set_error(RAST_E_INVALID_ARG, "rast_binmodel_loss_grad: bad arguments");
    RAST_TRY(model_ready(m));
    RAST_TRY(ensure(m->io_x, (size_t)n * F * 4));
    RAST_TRY(ensure(m->io_y, (size_t)n * 4));
    HIP_TRY(hipMemcpy(m->io_x.p, x, (size_t)n * F * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(m->io_y.p, target, (size_t)n * 4, hipMemcpyHostToDevice));
    RAST_TRY(train_partial<false>(m, n, n, (const float *)m->io_x.p, (const float *)m->io_y.p, 0u, tau));
    RAST_TRY(reduce_grad(m, n));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(grad, m->grad.p, num_params(m->H) * 4, hipMemcpyDeviceToHost));
    if (loss) HIP_TRY(hipMemcpy(loss, m->loss.p, 4, hipMemcpyDeviceToHost));
    return RAST_OK;
} RAST_CATCH

int rast_model_hidden(const rast_binmodel *m) { return m ? m->H : 0; }
const float *rast_model_params(const rast_binmodel *m) { return m ? (const float *)m->params.p : nullptr; }
