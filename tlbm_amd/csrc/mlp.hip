// mlp.hip -- training and stand-alone inference of the closure network
// (mlp.h), and their C-ABI (include/tlbm_gpu.h, tlbm_mlp_*).
//
// Training: each step draws `batch` samples (a counter-based hash of seed,
// step and position picks each index).  A wavefront takes 32 samples at a
// time through the forward and the backward pass and their weight gradient
// with FP32 MFMA and keeps the gradient in registers; per-workgroup partial
// gradients are folded in a fixed order by a second kernel, which applies Adam.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "mlp.h"
#include "tlbm_gpu.h"

namespace tlbm {

constexpr int kUnit = 32;           // samples a wavefront takes at a time
constexpr int kGradWaves = 4;       // wavefronts of a training workgroup
constexpr int kGradBlocks = 256;    // at most one training workgroup per CU
// offsets of the flat parameters
constexpr int kB1 = kMlpH * kMlpIn, kW2 = kB1 + kMlpH, kB2 = kW2 + kMlpH * kMlpH, kW3 = kB2 + kMlpH,
              kB3 = kW3 + kMlpH;

__device__ inline uint64_t mix64(uint64_t x) {  // splitmix64 finaliser
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// Partial gradient and loss of one workgroup's samples.  mode 0: sample i of the
// batch is index first + i; mode 1: a hashed index.
//
// All five products are v_mfma_f32_32x32x2_f32 (lane l supplies A[l%32][g] and
// B[g][l%32], g = l/32; lane l holds, in register 4q + r, row 8q + 4g + r of
// column l%32).  With the samples as columns a layer's output registers are
// the next product's B operand: K step (q, r) takes units 8q + r and
// 8q + 4 + r, and the weights are held per lane in that order, W2 both as it
// is (forward) and transposed (backward).  The weight gradients contract over
// the samples, so activations and deltas pass through LDS, written by rows of
// a sample and read by columns, within the wavefront.  b1 is the weight of an
// eighth input 1, so its gradient is that of W1.
//
// 65536 samples take 20 us.  The 68 products of 64 cycles per 32 samples are
// 3.6 us of that; the rest is what a wavefront's two units do not hide: the
// operands' loads, the samples' hashed indexes and gathers, the LDS passes and
// the wavefronts' sums.  One thread per sample with the weights in LDS took
// 46 us (an LDS read per multiply-add), and a fold by one thread per parameter
// 159 us (512 dependent loads).
__global__ void __launch_bounds__(kGradWaves * 64)
k_mlp_grad(const float *__restrict__ X, const float *__restrict__ Tg, int64_t M, int64_t first,
           int mode, uint64_t seed, int64_t step, int64_t batch, const float *__restrict__ params,
           float *__restrict__ partial, double *__restrict__ losses) {
    constexpr int S = kMlpH + 4;  // row of a sample in LDS: 16-byte aligned, banks spread
    struct Wave {
        float d[kUnit * S];   // deltas by sample (d2, then d1)
        float h[kUnit * S];   // h1 by sample
        float x[kUnit * 12];  // inputs by sample
    };
    __shared__ alignas(16) Wave sw[kGradWaves];
    __shared__ float sum[kMlpParams];
    __shared__ double loss_sum;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, c = l & 31, g = l >> 5;
    Wave &W = sw[wave];
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // operands that stay: W1 with b1 as input 7, W2, its transpose, b2 and w3
    float a1[4], a2[16], a2t[16], w3[16];
    f32x16 b2;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int k = 2 * t + g;
        a1[t] = k < kMlpIn ? params[c * kMlpIn + k] : params[kB1 + c];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int u = 8 * (k >> 2) + 4 * g + (k & 3);
        a2[k] = params[kW2 + c * kMlpH + u];
        a2t[k] = params[kW2 + u * kMlpH + c];
        b2[k] = params[kB2 + u];
        w3[k] = params[kW3 + u];
    }
    const float b3 = params[kB3];
    f32x16 gW2 = zero, gW1 = zero, gb2 = zero, gw3 = zero;
    float gb3 = 0.f;
    double loss = 0.0;
    const int64_t units = (batch + kUnit - 1) / kUnit, stride = int64_t(gridDim.x) * kGradWaves;
    for (int64_t un = int64_t(blockIdx.x) * kGradWaves + wave; un < units; un += stride) {
        const int64_t pos = un * kUnit + c;
        const bool live = pos < batch;
        int64_t idx = 0;
        if (live)
            idx = mode == 0 ? first + pos
                            : int64_t(mix64(seed ^ mix64(uint64_t(step) * 0x100000001ull + uint64_t(pos))) % uint64_t(M));
        float x[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = 2 * t + g;
            x[t] = k == kMlpIn ? 1.f : live ? X[idx * kMlpIn + k] : 0.f;
        }
        const float target = live ? Tg[idx] : 0.f;
        f32x16 h1 = zero;
#pragma unroll
        for (int t = 0; t < 4; ++t) h1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[t], x[t], h1, 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 16; ++k) h1[k] = fmaxf(h1[k], 0.f);
        f32x16 h2 = b2;
#pragma unroll
        for (int k = 0; k < 16; ++k) h2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[k], h1[k], h2, 0, 0, 0);
        float z = 0.f;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            h2[k] = fmaxf(h2[k], 0.f);
            z += w3[k] * h2[k];
        }
        z = (z + __shfl_xor(z, 32, 64)) + b3;
        const float y = z > 20.f ? z : log1pf(expf(z));
        const float r = live ? y - target : 0.f;
        const float dz = r / (1.f + expf(-z)) / float(batch);
        if (g == 0) {
            loss += double(0.5f * r * r);
            gb3 += dz;
        }
        f32x16 d2;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            d2[k] = h2[k] > 0.f ? dz * w3[k] : 0.f;
            gb2[k] += d2[k];
            gw3[k] += dz * h2[k];
        }
        f32x16 d1 = zero;
#pragma unroll
        for (int k = 0; k < 16; ++k) d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2t[k], d2[k], d1, 0, 0, 0);
        // dW2 = sum_s d2 h1^T
        typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            *reinterpret_cast<f32x4 *>(&W.d[c * S + 8 * q + 4 * g]) = f32x4{d2[4 * q], d2[4 * q + 1], d2[4 * q + 2], d2[4 * q + 3]};
            *reinterpret_cast<f32x4 *>(&W.h[c * S + 8 * q + 4 * g]) = f32x4{h1[4 * q], h1[4 * q + 1], h1[4 * q + 2], h1[4 * q + 3]};
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) W.x[c * 12 + 2 * t + g] = x[t];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int k = 0; k < 16; ++k)
            gW2 = __builtin_amdgcn_mfma_f32_32x32x2f32(W.d[(2 * k + g) * S + c], W.h[(2 * k + g) * S + c], gW2, 0, 0, 0);
        // dW1 = sum_s d1 x^T
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = h1[4 * q + e] > 0.f ? d1[4 * q + e] : 0.f;
            *reinterpret_cast<f32x4 *>(&W.d[c * S + 8 * q + 4 * g]) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const float xv = c < 8 ? W.x[(2 * k + g) * 12 + (c & 7)] : 0.f;
            gW1 = __builtin_amdgcn_mfma_f32_32x32x2f32(W.d[(2 * k + g) * S + c], xv, gW1, 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // sums over the samples' lanes: db2 and dw3 unit by unit through LDS
    // (row k of 64 lanes in W.d and W.h), db3 and the loss by exchange
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        W.d[k * 64 + l] = gb2[k];
        W.h[k * 64 + l] = gw3[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {  // lanes 32-63 hold none
        gb3 += __shfl_xor(gb3, off, 64);
        loss += __shfl_xor(loss, off, 64);
    }
    float unit = 0.f;  // lanes 0-31: db2 of unit c; lanes 32-63: dw3
    {
        const float *src = (g == 0 ? W.d : W.h) + (4 * (c >> 3) + (c & 3)) * 64 + 32 * ((c >> 2) & 1);
        for (int k = 0; k < 32; ++k) unit += src[(k + c) & 31];
    }
    // the wavefronts' sums, in order
    for (int v = 0; v < kGradWaves; ++v) {
        if (wave == v) {
            auto add = [&](int at, float val) { sum[at] = v == 0 ? val : sum[at] + val; };
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int u = 8 * (k >> 2) + 4 * g + (k & 3);
                add(kW2 + u * kMlpH + c, gW2[k]);
                if (c < kMlpIn) add(u * kMlpIn + c, gW1[k]);
                if (c == kMlpIn) add(kB1 + u, gW1[k]);
            }
            add((g == 0 ? kB2 : kW3) + c, unit);
            if (l == 0) add(kB3, gb3);
            if (l == 1) loss_sum = v == 0 ? loss : loss_sum + loss;
        }
        __syncthreads();
    }
    float *out = partial + size_t(blockIdx.x) * kMlpParams;
    for (int k = threadIdx.x; k < kMlpParams; k += kGradWaves * 64) out[k] = sum[k];
    if (threadIdx.x == 0) losses[blockIdx.x] = loss_sum;
}

// Fold the partial gradients in double; with adam != 0 apply Adam.  grad_out
// (may be null) receives the folded gradient, loss_out the mean loss.  A
// workgroup folds 16 parameters, the last one the loss: slice i of its 16
// slices of 16 threads adds partials i, i + 16, ..., then the slices' sums are
// added in order.
constexpr int kFoldBlocks = (kMlpParams + 15) / 16 + 1;
__global__ void __launch_bounds__(256)
k_mlp_fold_adam(const float *__restrict__ partial, const double *__restrict__ losses, int nblocks, int64_t batch,
                int adam, float *__restrict__ params, float *__restrict__ mom, float *__restrict__ vel,
                float lr, float c1, float c2, float *__restrict__ grad_out,
                double *__restrict__ loss_out) {
    __shared__ double part[16][17];
    const int p = threadIdx.x & 15, slice = threadIdx.x >> 4;
    const int k = blockIdx.x * 16 + p;
    const bool mean = blockIdx.x == kFoldBlocks - 1 && p == 0;
    double acc = 0.0;
    if (k < kMlpParams) {
#pragma unroll 4
        for (int b = slice; b < nblocks; b += 16) acc += double(partial[size_t(b) * kMlpParams + k]);
    } else if (mean) {
#pragma unroll 4
        for (int b = slice; b < nblocks; b += 16) acc += losses[b];
    }
    part[slice][p] = acc;
    __syncthreads();
    if (slice != 0 || (k >= kMlpParams && !mean)) return;
    double total = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) total += part[i][p];
    if (mean) {
        *loss_out = total / double(batch);
        return;
    }
    const float g = float(total);
    if (grad_out) grad_out[k] = g;
    if (adam) {
        const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
        const float m = beta1 * mom[k] + (1.f - beta1) * g;
        const float v = beta2 * vel[k] + (1.f - beta2) * g * g;
        mom[k] = m;
        vel[k] = v;
        params[k] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
    }
}

__global__ void __launch_bounds__(256)
k_mlp_infer(const float *__restrict__ X, int64_t n, const MlpPacked *__restrict__ m,
            float *__restrict__ z) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int64_t src = i < n ? i : n - 1;  // whole wavefronts take part
    float x[kMlpIn];
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) x[k] = X[src * kMlpIn + k];
    const float r = mlp_wave(x, m);
    if (i < n) z[i] = r;
}

}  // namespace tlbm

namespace tlbm {
void set_last_error(const std::string &msg);  // tlbm_gpu.cpp
}

namespace {

int mfail(int code, const std::string &msg) {
    tlbm::set_last_error(msg);
    return code;
}

#define MLP_HIP(call)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess)                                                               \
            return mfail(TLBM_EHIP, std::string(#call) + ": " + hipGetErrorString(e_));     \
    } while (0)

}  // namespace

// Training workgroups of a batch: a unit per wavefront while CUs are free.
static int grad_blocks(int64_t batch) {
    const int64_t units = (batch + tlbm::kUnit - 1) / tlbm::kUnit;
    const int64_t blocks = (units + tlbm::kGradWaves - 1) / tlbm::kGradWaves;
    return int(blocks < tlbm::kGradBlocks ? blocks : tlbm::kGradBlocks);
}

struct tlbm_mlp_trainer {
    int64_t n = 0;
    float *X = nullptr, *T = nullptr, *params = nullptr, *mom = nullptr, *vel = nullptr;
    float *partial = nullptr, *grad = nullptr;
    double *loss = nullptr, *losses = nullptr;  // of the batch; of the training workgroups
    int max_batch = 0, max_blocks = 0;
    int64_t steps = 0;
    uint64_t seed = 0;
    hipStream_t stream = nullptr;
};

extern "C" {

int tlbm_mlp_trainer_create(const float *x, const float *t, int64_t n, const float *init,
                            uint64_t seed, int max_batch, tlbm_mlp_trainer **out) {
    if (!x || !t || !init || !out || n <= 0 || max_batch <= 0)
        return mfail(TLBM_EINVAL, "bad trainer arguments");
    *out = nullptr;
    tlbm_mlp_trainer *tr = new (std::nothrow) tlbm_mlp_trainer;
    if (!tr) return mfail(TLBM_ENOMEM, "host allocation failed");
    tr->n = n;
    tr->seed = seed;
    tr->max_batch = max_batch;
    tr->max_blocks = grad_blocks((int64_t(max_batch) + 127) / 128 * 128);
    auto bail = [&](int rc) {
        tlbm_mlp_trainer_destroy(tr);
        return rc;
    };
    const size_t P = tlbm::kMlpParams;
    if (hipStreamCreateWithFlags(&tr->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&tr->X, sizeof(float) * size_t(n) * tlbm::kMlpIn) != hipSuccess ||
        hipMalloc(&tr->T, sizeof(float) * size_t(n)) != hipSuccess ||
        hipMalloc(&tr->params, sizeof(float) * P) != hipSuccess ||
        hipMalloc(&tr->mom, sizeof(float) * P) != hipSuccess ||
        hipMalloc(&tr->vel, sizeof(float) * P) != hipSuccess ||
        hipMalloc(&tr->grad, sizeof(float) * P) != hipSuccess ||
        hipMalloc(&tr->loss, sizeof(double)) != hipSuccess ||
        hipMalloc(&tr->partial, sizeof(float) * size_t(tr->max_blocks) * P) != hipSuccess ||
        hipMalloc(&tr->losses, sizeof(double) * size_t(tr->max_blocks)) != hipSuccess)
        return bail(mfail(TLBM_ENOMEM, "device allocation failed"));
    if (hipMemcpy(tr->X, x, sizeof(float) * size_t(n) * tlbm::kMlpIn, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(tr->T, t, sizeof(float) * size_t(n), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(tr->params, init, sizeof(float) * P, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(tr->mom, 0, sizeof(float) * P) != hipSuccess ||
        hipMemset(tr->vel, 0, sizeof(float) * P) != hipSuccess)
        return bail(mfail(TLBM_EHIP, "upload failed"));
    *out = tr;
    return TLBM_OK;
}

int tlbm_mlp_trainer_destroy(tlbm_mlp_trainer *tr) {
    if (!tr) return TLBM_OK;
    if (tr->stream) (void)hipStreamSynchronize(tr->stream);
    for (void *p : {(void *)tr->X, (void *)tr->T, (void *)tr->params, (void *)tr->mom,
                    (void *)tr->vel, (void *)tr->partial, (void *)tr->grad, (void *)tr->loss,
                    (void *)tr->losses})
        if (p) (void)hipFree(p);
    if (tr->stream) (void)hipStreamDestroy(tr->stream);
    delete tr;
    return TLBM_OK;
}

int tlbm_mlp_trainer_step(tlbm_mlp_trainer *tr, int steps, int batch, float lr, double *last_loss) {
    if (!tr || steps < 0 || batch <= 0) return mfail(TLBM_EINVAL, "bad step arguments");
    // (whole units of 128 samples, as max_batch has always been rounded)
    if ((int64_t(batch) + 127) / 128 > (int64_t(tr->max_batch) + 127) / 128)
        return mfail(TLBM_EINVAL, "batch larger than the trainer's max_batch");
    const int nb = grad_blocks(batch);
    for (int k = 0; k < steps; ++k) {
        ++tr->steps;
        hipLaunchKernelGGL(tlbm::k_mlp_grad, dim3(nb), dim3(tlbm::kGradWaves * 64), 0, tr->stream, tr->X, tr->T,
                           tr->n, int64_t(0), 1, tr->seed, tr->steps, int64_t(batch), tr->params,
                           tr->partial, tr->losses);
        MLP_HIP(hipGetLastError());
        const float c1 = 1.f - std::pow(0.9f, float(tr->steps));
        const float c2 = 1.f - std::pow(0.999f, float(tr->steps));
        hipLaunchKernelGGL(tlbm::k_mlp_fold_adam, dim3(tlbm::kFoldBlocks), dim3(256),
                           0, tr->stream, tr->partial, tr->losses, nb, int64_t(batch), 1, tr->params, tr->mom,
                           tr->vel, lr, c1, c2, (float *)nullptr, tr->loss);
        MLP_HIP(hipGetLastError());
    }
    if (last_loss) {
        MLP_HIP(hipMemcpyAsync(last_loss, tr->loss, sizeof(double), hipMemcpyDeviceToHost, tr->stream));
    }
    MLP_HIP(hipStreamSynchronize(tr->stream));
    return TLBM_OK;
}

int tlbm_mlp_trainer_loss_grad(tlbm_mlp_trainer *tr, int64_t first, int64_t count, double *loss,
                               float *grad) {
    if (!tr || first < 0 || count <= 0 || first + count > tr->n || !loss || !grad)
        return mfail(TLBM_EINVAL, "bad loss_grad arguments");
    if ((count + 127) / 128 > (int64_t(tr->max_batch) + 127) / 128)
        return mfail(TLBM_EINVAL, "count larger than the trainer's max_batch");
    const int nb = grad_blocks(count);
    hipLaunchKernelGGL(tlbm::k_mlp_grad, dim3(nb), dim3(tlbm::kGradWaves * 64), 0, tr->stream, tr->X, tr->T, tr->n,
                       first, 0, tr->seed, int64_t(0), count, tr->params, tr->partial, tr->losses);
    MLP_HIP(hipGetLastError());
    hipLaunchKernelGGL(tlbm::k_mlp_fold_adam, dim3(tlbm::kFoldBlocks), dim3(256), 0,
                       tr->stream, tr->partial, tr->losses, nb, count, 0, tr->params, tr->mom, tr->vel, 0.f, 1.f,
                       1.f, tr->grad, tr->loss);
    MLP_HIP(hipGetLastError());
    MLP_HIP(hipMemcpyAsync(grad, tr->grad, sizeof(float) * tlbm::kMlpParams, hipMemcpyDeviceToHost, tr->stream));
    MLP_HIP(hipMemcpyAsync(loss, tr->loss, sizeof(double), hipMemcpyDeviceToHost, tr->stream));
    MLP_HIP(hipStreamSynchronize(tr->stream));
    return TLBM_OK;
}

int tlbm_mlp_trainer_params(tlbm_mlp_trainer *tr, float *params) {
    if (!tr || !params) return mfail(TLBM_EINVAL, "null argument");
    MLP_HIP(hipMemcpyAsync(params, tr->params, sizeof(float) * tlbm::kMlpParams, hipMemcpyDeviceToHost, tr->stream));
    MLP_HIP(hipStreamSynchronize(tr->stream));
    return TLBM_OK;
}

int tlbm_mlp_infer(const float *params, const float *x, int64_t n, float *z) {
    if (!params || !x || !z || n <= 0) return mfail(TLBM_EINVAL, "bad inference arguments");
    tlbm::MlpPacked host;
    tlbm::mlp_pack(params, &host);
    tlbm::MlpPacked *dm = nullptr;
    float *dx = nullptr, *dz = nullptr;
    int rc = TLBM_OK;
    if (hipMalloc(&dm, sizeof host) != hipSuccess || hipMalloc(&dx, sizeof(float) * size_t(n) * tlbm::kMlpIn) != hipSuccess ||
        hipMalloc(&dz, sizeof(float) * size_t(n)) != hipSuccess) {
        rc = mfail(TLBM_ENOMEM, "device allocation failed");
    } else if (hipMemcpy(dm, &host, sizeof host, hipMemcpyHostToDevice) != hipSuccess ||
               hipMemcpy(dx, x, sizeof(float) * size_t(n) * tlbm::kMlpIn, hipMemcpyHostToDevice) != hipSuccess) {
        rc = mfail(TLBM_EHIP, "upload failed");
    } else {
        hipLaunchKernelGGL(tlbm::k_mlp_infer, dim3(unsigned((n + 255) / 256)), dim3(256), 0, 0, dx, n, dm, dz);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
            hipMemcpy(z, dz, sizeof(float) * size_t(n), hipMemcpyDeviceToHost) != hipSuccess)
            rc = mfail(TLBM_EHIP, "inference failed");
    }
    if (dm) (void)hipFree(dm);
    if (dx) (void)hipFree(dx);
    if (dz) (void)hipFree(dz);
    return rc;
}

}  // extern "C"
