// Training and evaluation kernels of the warm-start surrogate, and the
// library's resident copy of the loaded network.
//
// Training step (all FP32 accumulation; BF16 rounding where the inference
// kernel rounds, so the trained network is the one the ascent evaluates):
//   mlp_train       64 samples at a time through the whole step in LDS --
//                   z1 = W1 u + b1, h1 = bf16(gelu(z1)), z2 = W2 h1 + b2,
//                   h2 = gelu(z2), y = w3 . h2 + b3, dy = 2 (y - t) / n,
//                   dz2 = dy w3 gelu'(z2), dz1 = (W2^T dz2) gelu'(z1) -- and
//                   the block's sums of the weight gradients
//   mlp_grad_sum    the blocks' sums added up (fixed order: deterministic)
//   mlp_adam        Adam on the FP32 master vector
// The gradient is the straight-through one: the BF16 rounding is treated as
// the identity in the backward pass.
#include <hip/hip_runtime.h>
#include <math.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "../../include/xcape_hip.h"
#include "capi_common.h"
#include "mlp_device.h"

using namespace xcape;

namespace {

constexpr int H = MLP_H;

// weights as the forward uses them: BF16-rounded W1, W2, w3; FP32 biases
struct alignas(16) FwdWeights {
    float w1[H * 3], b1[H], w2[H * H], b2[H], w3[H], b3;
};

__device__ __forceinline__ void load_weights(const float *theta, FwdWeights &w)
{
    for (int i = threadIdx.x; i < H * 3; i += blockDim.x) w.w1[i] = bf16_round(theta[MLP_OFF_W1 + i]);
    for (int i = threadIdx.x; i < H * H; i += blockDim.x) w.w2[i] = bf16_round(theta[MLP_OFF_W2 + i]);
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
        w.b1[i] = theta[MLP_OFF_B1 + i];
        w.b2[i] = theta[MLP_OFF_B2 + i];
        w.w3[i] = bf16_round(theta[MLP_OFF_W3 + i]);
    }
    if (threadIdx.x == 0) w.b3 = theta[MLP_OFF_B3];
    __syncthreads();
}

// forward for one sample
__device__ __forceinline__ float forward_one(const FwdWeights &w, const float *u)
{
    float h1[H];
#pragma unroll
    for (int j = 0; j < H; ++j) {
        const float z = w.b1[j] + w.w1[3 * j] * u[0] + w.w1[3 * j + 1] * u[1] + w.w1[3 * j + 2] * u[2];
        h1[j] = bf16_round(gelu_f(z));
    }
    float y = w.b3;
    for (int i = 0; i < H; ++i) {
        float z = w.b2[i];
#pragma unroll
        for (int j = 0; j < H; ++j) z += w.w2[i * H + j] * h1[j];
        y += w.w3[i] * gelu_f(z);
    }
    return y;
}

__global__ void __launch_bounds__(256) mlp_forward(const float *x, int64_t n, const float *theta,
                                                   float *y)
{
    __shared__ FwdWeights w;
    load_weights(theta, w);
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const float u[3] = {x[3 * s], x[3 * s + 1], x[3 * s + 2]};
    y[s] = forward_one(w, u);
}

// ---- the training step's gradients ------------------------------------------
//
// A block takes tiles of 64 samples in turn and keeps everything of a tile in
// LDS and registers; with one pass per layer over global memory instead, the
// activations and their gradients (6 arrays of 64 floats per sample) went
// through HBM between three launches, and the weight gradients' sums ran on 65
// blocks.  A step at 16 384 samples (gradients and Adam) took 334 us so and
// takes 43 us here; what is left is its three launches.
//
// The products over 64 units or 64 samples run on the matrix cores: the
// forward's W2 h1 in BF16 (both operands are BF16 values: exact products, FP32
// sums), the backward's W2^T dz2 and dz2 h1^T in FP32, since dz2 is FP32.
// Wave (tm, tn) = (wave / 2, wave % 2) owns one 32 x 32 tile of each product,
// in the layout of v_mfma_f32_32x32x*: register r of lane (half, col) is
// element [32 tm + 8 (r / 4) + 4 half + r % 4][32 tn + col].  Layer 1 is
// computed in that layout too ([sample][unit]), so its slopes stay in the
// registers where the backward product delivers dz1.
constexpr int TT = 64;                 // samples per tile
constexpr int TP = 65;                 // row pitch of the FP32 tiles in LDS (distinct banks)
constexpr int TPB = 36;                // row pitch of the BF16 tiles, words (16-byte rows)
constexpr int GRAD_ROW = MLP_NPARAMS + 1;   // a block's sums: the gradient, then the loss
constexpr int TRAIN_BLOCKS = 256;      // one per CU (the tiles take 88 KB of its LDS)

struct TrainLds {
    float w2[H * H];                   // BF16-rounded, [i][j]
    float h1[TT * TP];                 // [sample][j]
    float dz2[H * TP];                 // [i][sample]
    float h2[H * TP];                  // [i][sample]
    uint32_t w2b[H * TPB];             // BF16 pairs, [i][j]
    uint32_t h1b[TT * TPB];            // BF16 pairs, [sample][j]
    float x[TT * 3], t[TT], y[2][TT], dy[TT];
    float b2[H], w3[H], red[4][H];
};

// gelu_f of one argument, and its derivative
__device__ __forceinline__ void gelu_both(float z, float &h, float &slope)
{
    const float c = 0.7978845608028654f, a = 0.044715f;
    const float u = c * (z + a * z * z * z);
    const float e = __expf(2.0f * u);
    const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e);
    h = 0.5f * z * (1.0f + t);
    slope = 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * c * (1.0f + 3.0f * a * z * z);
}

// grid: at most TRAIN_BLOCKS blocks, block b takes tiles b, b + grid, ...;
// part: GRAD_ROW floats per block
__global__ void __launch_bounds__(256) mlp_train(const float *x, const float *t, int64_t n,
                                                 const float *theta, float *part)
{
    __shared__ TrainLds L;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int half = lane >> 5, col = lane & 31, tm = wave >> 1, tn = wave & 1;
    const int row0 = 32 * tm + 4 * half;           // row of register r: row0 + 8 (r / 4) + r % 4
    const int j = 32 * tn + col;
    for (int i = tid; i < H * H; i += 256) {
        const uint16_t b = bf16_bits(theta[MLP_OFF_W2 + i]);
        L.w2[i] = __uint_as_float((uint32_t)b << 16);
        reinterpret_cast<uint16_t *>(L.w2b)[(i / H) * 2 * TPB + i % H] = b;
    }
    if (tid < H) {
        L.b2[tid] = theta[MLP_OFF_B2 + tid];
        L.w3[tid] = bf16_round(theta[MLP_OFF_W3 + tid]);
    }
    const float b3 = theta[MLP_OFF_B3];
    const float b1 = theta[MLP_OFF_B1 + j];
    const float w10 = bf16_round(theta[MLP_OFF_W1 + 3 * j]),
                w11 = bf16_round(theta[MLP_OFF_W1 + 3 * j + 1]),
                w12 = bf16_round(theta[MLP_OFF_W1 + 3 * j + 2]);
    xc_f32x16 gw2 = {};
    float gw10 = 0.0f, gw11 = 0.0f, gw12 = 0.0f, gb1 = 0.0f;   // unit j, this lane's samples
    float gvec = 0.0f;            // threads 0 .. 63: dw3[tid]; 64 .. 127: db2[tid - 64]
    float gb3 = 0.0f, loss = 0.0f;                             // threads 0 .. 63
    const int64_t tiles = (n + TT - 1) / TT;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t s0 = tile * TT;
        const int ns = n - s0 < TT ? (int)(n - s0) : TT;
        // samples past n: zero inputs, and dy = 0 below
        if (tid < 3 * TT) L.x[tid] = tid < 3 * ns ? x[3 * s0 + tid] : 0.0f;
        else if (tid - 3 * TT < TT) L.t[tid - 3 * TT] = tid - 3 * TT < ns ? t[s0 + tid - 3 * TT] : 0.0f;
        __syncthreads();
        // layer 1: samples row0 + .., unit j
        float slope1[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int s = row0 + 8 * (r >> 2) + (r & 3);
            const float z = b1 + w10 * L.x[3 * s] + w11 * L.x[3 * s + 1] + w12 * L.x[3 * s + 2];
            float h;
            gelu_both(z, h, slope1[r]);
            const uint16_t b = bf16_bits(h);
            L.h1[s * TP + j] = __uint_as_float((uint32_t)b << 16);
            reinterpret_cast<uint16_t *>(L.h1b)[s * 2 * TPB + j] = b;
        }
        __syncthreads();
        // layer 2: units row0 + .., sample j; layer 3's partial sums
        xc_f32x16 z2 = {};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const int k0 = 8 * kb + 4 * half;      // words
            xc_bf16x8 a, b;
            __builtin_memcpy(&a, &L.w2b[(32 * tm + col) * TPB + k0], 16);
            __builtin_memcpy(&b, &L.h1b[j * TPB + k0], 16);
            z2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, z2, 0, 0, 0);
        }
        float slope2[16], part3 = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = row0 + 8 * (r >> 2) + (r & 3);
            float h;
            gelu_both(z2[r] + L.b2[i], h, slope2[r]);
            L.h2[i * TP + j] = h;
            part3 += L.w3[i] * h;
        }
        part3 += __shfl_xor(part3, 32, 64);
        if (half == 0) L.y[tm][j] = part3;
        __syncthreads();
        if (tid < TT) {
            const float r = tid < ns ? (b3 + L.y[0][tid] + L.y[1][tid]) - L.t[tid] : 0.0f;
            const float g = 2.0f * r / (float)n;
            L.dy[tid] = g;
            gb3 += g;
            loss += r * r;
        }
        __syncthreads();
        const float dyj = L.dy[j];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = row0 + 8 * (r >> 2) + (r & 3);
            L.dz2[i * TP + j] = dyj * L.w3[i] * slope2[r];
        }
        __syncthreads();
        // dz1^T W2 (samples x units) and dz2 h1 (units x units)
        xc_f32x16 d1 = {};
#pragma unroll 8
        for (int kk = 0; kk < 32; ++kk) {
            const int k = 2 * kk + half;
            d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(L.dz2[k * TP + 32 * tm + col],
                                                      L.w2[k * H + j], d1, 0, 0, 0);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(L.dz2[(32 * tm + col) * TP + k],
                                                       L.h1[k * TP + j], gw2, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int s = row0 + 8 * (r >> 2) + (r & 3);
            const float d = d1[r] * slope1[r];
            gw10 += d * L.x[3 * s];
            gw11 += d * L.x[3 * s + 1];
            gw12 += d * L.x[3 * s + 2];
            gb1 += d;
        }
        if (tid < 2 * H) {
            const float *v = tid < H ? L.h2 + tid * TP : L.dz2 + (tid - H) * TP;
#pragma unroll 8
            for (int s = 0; s < TT; ++s) gvec += tid < H ? L.dy[s] * v[s] : v[s];
        }
        __syncthreads();   // the tile's arrays are rewritten by the next one
    }
    // the block's sums
    float *p = part + (size_t)blockIdx.x * GRAD_ROW;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        p[MLP_OFF_W2 + (row0 + 8 * (r >> 2) + (r & 3)) * H + j] = gw2[r];
    if (tid < H) p[MLP_OFF_W3 + tid] = gvec;
    else if (tid < 2 * H) p[MLP_OFF_B2 + tid - H] = gvec;
    // unit j's sums: this lane's, its other half's, the other row tile's
    gw10 += __shfl_xor(gw10, 32, 64);
    gw11 += __shfl_xor(gw11, 32, 64);
    gw12 += __shfl_xor(gw12, 32, 64);
    gb1 += __shfl_xor(gb1, 32, 64);
    if (tm == 1 && half == 0) {
        L.red[0][j] = gw10;
        L.red[1][j] = gw11;
        L.red[2][j] = gw12;
        L.red[3][j] = gb1;
    }
    __syncthreads();
    if (tm == 0 && half == 0) {
        p[MLP_OFF_W1 + 3 * j] = gw10 + L.red[0][j];
        p[MLP_OFF_W1 + 3 * j + 1] = gw11 + L.red[1][j];
        p[MLP_OFF_W1 + 3 * j + 2] = gw12 + L.red[2][j];
        p[MLP_OFF_B1 + j] = gb1 + L.red[3][j];
    }
    if (wave == 0) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            gb3 += __shfl_xor(gb3, off, 64);
            loss += __shfl_xor(loss, off, 64);
        }
        if (lane == 0) {
            p[MLP_OFF_B3] = gb3;
            p[MLP_NPARAMS] = loss;
        }
    }
}

// The blocks' sums of one parameter per lane: 16 rows of 64 lanes take every
// 16th block's, and are added in order.
__global__ void __launch_bounds__(1024) mlp_grad_sum(const float *part, int nblk, int64_t n,
                                                     float *grad, float *loss)
{
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    float v = 0.0f;
    if (c < GRAD_ROW) {
#pragma unroll 4
        for (int b = w; b < nblk; b += 16) v += part[(size_t)b * GRAD_ROW + c];
    }
    red[w][lane] = v;
    __syncthreads();
    if (w == 0 && c < GRAD_ROW) {
        v = red[0][lane];
#pragma unroll
        for (int k = 1; k < 16; ++k) v += red[k][lane];
        if (c < MLP_NPARAMS) grad[c] = v;
        else if (loss) *loss = v / (float)n;
    }
}

__global__ void mlp_adam(float *theta, const float *grad, float *m, float *v, int64_t step,
                         float lr, float b1, float b2, float eps, float wd)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MLP_NPARAMS) return;
    const float g = grad[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / (1.0f - powf(b1, (float)step));
    const float vh = vi / (1.0f - powf(b2, (float)step));
    theta[i] -= lr * (mh / (sqrtf(vh) + eps) + wd * theta[i]);
}

// Pack the FP32 master vector and normalisation into the device layout the
// ascent kernels read.
__global__ void pack_surrogate(const float *theta, const float *norm, SurrogateDev *S)
{
    for (int i = threadIdx.x; i < H * H; i += blockDim.x) S->w2[i] = bf16_bits(theta[MLP_OFF_W2 + i]);
    for (int i = threadIdx.x; i < H * 3; i += blockDim.x) S->w1[i] = bf16_round(theta[MLP_OFF_W1 + i]);
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
        S->b1[i] = theta[MLP_OFF_B1 + i];
        S->b2[i] = theta[MLP_OFF_B2 + i];
        S->w3[i] = bf16_round(theta[MLP_OFF_W3 + i]);
    }
    if (threadIdx.x == 0) {
        S->b3 = theta[MLP_OFF_B3];
        for (int k = 0; k < 3; ++k) {
            S->in_mean[k] = norm[k];
            S->in_scale[k] = norm[3 + k];
        }
        S->out_scale = norm[6];
        S->out_offset = norm[7];
    }
}

// Batch evaluation through the in-kernel (MFMA) path: each wave evaluates 64
// samples with surrogate_eval_wave.  Lanes past n evaluate a dummy sample.
__global__ void __launch_bounds__(256) surrogate_eval_kernel(const SurrogateDev *S,
                                                             const float *x, int64_t n,
                                                             float *y)
{
    __shared__ uint32_t lds[4 * MLP_LDS_WORDS_PER_WAVE];
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool ok = s < n;
    const float x0 = ok ? x[3 * s] : 0.0f, x1 = ok ? x[3 * s + 1] : 0.0f,
                x2 = ok ? x[3 * s + 2] : 0.0f;
    const float r = surrogate_eval_wave(S, x0, x1, x2,
                                        lds + (threadIdx.x >> 6) * MLP_LDS_WORDS_PER_WAVE);
    if (ok) y[s] = r;
}

int check_n(int64_t n)
{
    if (n < 1 || n > (int64_t)1 << 31) return fail(XCAPE_EINVAL, "n=%lld out of range", (long long)n);
    return XCAPE_OK;
}

}  // namespace

namespace xcape {

// The loaded network (device memory, one per process); nullptr until
// xcape_surrogate_load.  A load packs the new weights into a buffer of its
// own, waits for the packing to finish and only then publishes the pointer,
// so a kernel launched by another thread sees either the old network or the
// new one, whole.  Replaced buffers are kept (13.6 KB each) until the process
// ends: kernels already queued, and ragged plans (which keep the pointer
// they were created with), may still read them.
std::atomic<SurrogateDev *> g_surrogate{nullptr};
std::mutex g_surrogate_mu;                   // serialises loads
std::vector<SurrogateDev *> g_surrogate_old;  // replaced buffers, kept alive

const void *surrogate_device() { return g_surrogate.load(std::memory_order_acquire); }

}  // namespace xcape

extern "C" {

int xcape_mlp_nparams(void) { return MLP_NPARAMS; }

int xcape_mlp_forward(const float *x, int64_t n, const float *theta, float *y, void *stream)
{
    int rc = check_n(n);
    if (rc || (rc = ensure_device())) return rc;
    if (!x || !theta || !y) return fail(XCAPE_EINVAL, "NULL argument");
    hipStream_t s = (hipStream_t)stream;
    const unsigned blocks = (unsigned)((n + 255) / 256);
    mlp_forward<<<blocks, 256, 0, s>>>(x, n, theta, y);
    hipError_t e = hipGetLastError();
    return e ? hip_fail(e, "mlp_forward") : XCAPE_OK;
}

int xcape_mlp_loss_grad(const float *x, const float *t, int64_t n, const float *theta,
                        float *grad, float *loss, void *stream)
{
    int rc = check_n(n);
    if (rc || (rc = ensure_device())) return rc;
    if (!x || !t || !theta || !grad) return fail(XCAPE_EINVAL, "NULL argument");
    hipStream_t s = (hipStream_t)stream;
    const int64_t tiles = (n + TT - 1) / TT;
    const int blocks = tiles < TRAIN_BLOCKS ? (int)tiles : TRAIN_BLOCKS;
    DevBuf<float> part;
    hipError_t e;
    if ((e = part.alloc((size_t)blocks * GRAD_ROW, s))) return hip_fail(e, "mlp workspace");
    mlp_train<<<blocks, 256, 0, s>>>(x, t, n, theta, part.ptr);
    mlp_grad_sum<<<(GRAD_ROW + 63) / 64, 1024, 0, s>>>(part.ptr, blocks, n, grad, loss);
    e = hipGetLastError();
    return e ? hip_fail(e, "mlp_loss_grad") : XCAPE_OK;
}

int xcape_mlp_adam(float *theta, const float *grad, float *m, float *v, int64_t step, float lr,
                   float beta1, float beta2, float eps, float weight_decay, void *stream)
{
    if (!theta || !grad || !m || !v) return fail(XCAPE_EINVAL, "NULL argument");
    if (step < 1) return fail(XCAPE_EINVAL, "step must be >= 1");
    int rc = ensure_device();
    if (rc) return rc;
    mlp_adam<<<(MLP_NPARAMS + 255) / 256, 256, 0, (hipStream_t)stream>>>(
        theta, grad, m, v, step, lr, beta1, beta2, eps, weight_decay);
    hipError_t e = hipGetLastError();
    return e ? hip_fail(e, "mlp_adam") : XCAPE_OK;
}

int xcape_surrogate_load(const float *theta, const float *norm, void *stream)
{
    if (!theta || !norm) return fail(XCAPE_EINVAL, "NULL argument");
    int rc = ensure_device();
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    hipError_t e;
    std::lock_guard<std::mutex> lk(g_surrogate_mu);
    SurrogateDev *fresh = nullptr;
    if ((e = hipMalloc((void **)&fresh, sizeof(SurrogateDev))))
        return hip_fail(e, "surrogate allocation");
    pack_surrogate<<<1, 256, 0, s>>>(theta, norm, fresh);
    if ((e = hipGetLastError()) || (e = hipStreamSynchronize(s))) {
        (void)hipFree(fresh);
        return hip_fail(e, "surrogate load");
    }
    SurrogateDev *old = g_surrogate.exchange(fresh, std::memory_order_acq_rel);
    if (old) g_surrogate_old.push_back(old);
    return XCAPE_OK;
}

int xcape_surrogate_loaded(void) { return surrogate_device() != nullptr; }

int xcape_surrogate_eval(const float *x, int64_t n, float *y, void *stream)
{
    int rc = check_n(n);
    if (rc || (rc = ensure_device())) return rc;
    const SurrogateDev *sur = static_cast<const SurrogateDev *>(surrogate_device());
    if (!sur) return fail(XCAPE_ESTATE, "no surrogate loaded");
    if (!x || !y) return fail(XCAPE_EINVAL, "NULL argument");
    hipStream_t s = (hipStream_t)stream;
    surrogate_eval_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(sur, x, n, y);
    hipError_t e = hipGetLastError();
    return e ? hip_fail(e, "surrogate_eval") : XCAPE_OK;
}

}  // extern "C"
