// rankpred.hip -- MLP predictor of the ACA+ rank of an admissible block.
//
// No reference counterpart: aca.jl:36-106 runs ACA+ adaptively with growing
// storage.  The predictor maps block geometry and tolerance to the rank ACA+
// will reach, so the batched device ACA+ (aca_gpu.hip) can give every block a
// fixed term capacity up front; blocks that outgrow it continue in a further
// pass, which leaves the factors unchanged.
//
// Network: 9 -> H -> H -> 1 with ReLU, inputs the scale-free block features
// of host_hmatrix.cpp (block_features: cluster sizes relative to their
// distance, tolerance relative to the entries, point counts, cluster shapes),
// normalised by the training set's mean / standard deviation, output
// z ~ log(1 + rank).  Weights are held in BF16 for the forward pass (FP32
// master copy for Adam), all accumulation is FP32.  Loss: mean squared error.
//
// Kernels:
//   k_mlp_grad    a 256-thread workgroup takes 32 samples: activations and
//                 their gradients live in padded LDS tiles (8 threads per
//                 sample for the 64-wide layers), the weight gradients
//                 dW2 = dA2^T H1 and dW1 = dA1^T X are summed over the
//                 workgroup's samples in sample order; one partial gradient
//                 row per workgroup.  Bound by LDS reads: a thread owns 8 (16)
//                 neighbouring outputs, reads their weights as 16-byte vectors
//                 and each shared operand once for all of them (W2 is held both
//                 ways round for that); 24.5 -> 20.2 us per 4,096 samples.
//   k_mlp_adam    thread per parameter: sums the partial rows in workgroup
//                 order (deterministic), applies Adam, refreshes the BF16 copy;
//                 one more workgroup sums the losses.  Bound by the latency of
//                 the partial rows, so 16 of them are in flight per thread and a
//                 workgroup is one wave; 30.5 + 5.7 us (with a loss
//                 sum of its own) -> 6.7 us.
//   k_mlp_predict thread per sample, BF16 weights expanded into LDS.
#include "device_op.hpp"

#include <cmath>
#include <numeric>
#include <random>

namespace hmx {

namespace {

constexpr int kIn = kRankFeatures;
constexpr int kH = 64;
constexpr int kGradThreads = 256;  // threads of a gradient workgroup
constexpr int kGS = 32;            // samples per gradient workgroup
constexpr int kPad = kH + 4;  // LDS row stride: 16-byte aligned rows, four banks apart
constexpr int kNParams = kIn * kH + kH + kH * kH + kH + kH + 1;
// parameter offsets
constexpr int oW1 = 0, oB1 = oW1 + kIn * kH, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH,
              oB3 = oW3 + kH;
static_assert(oB3 + 1 == kNParams, "parameter layout");

__host__ __device__ inline float bf16_round(float x) {
    // round to nearest even on the upper 16 bits (NaN kept quiet)
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7fffffffu) > 0x7f800000u)
        u |= 0x00400000u;
    else
        u += 0x7fffu + ((u >> 16) & 1u);
    return __builtin_bit_cast(float, u & 0xffff0000u);
}

struct Norm {
    float mean[kIn];
    float inv_std[kIn];
};

// weights (BF16 values stored as FP32) -> LDS
__device__ inline void load_weights(const float* __restrict__ wq, float* lw) {
    for (int p = threadIdx.x; p < kNParams; p += blockDim.x) lw[p] = wq[p];
}

__device__ inline void normalise(const float* __restrict__ x, const Norm& nm, float* xn) {
#pragma unroll
    for (int i = 0; i < kIn; i++) xn[i] = (x[i] - nm.mean[i]) * nm.inv_std[i];
}

// Eight consecutive floats of an LDS row, as two 16-byte reads.
struct alignas(16) F4 {
    float v[4];
};
__device__ inline void load8(const float* p, float (&w)[8]) {
    const F4 x = reinterpret_cast<const F4*>(p)[0], y = reinterpret_cast<const F4*>(p)[1];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        w[c] = x.v[c];
        w[4 + c] = y.v[c];
    }
}

__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(const float* __restrict__ wq,
                                                           const float* __restrict__ X,
                                                           const float* __restrict__ T,
                                                           const int32_t* __restrict__ idx,
                                                           int64_t first, int64_t count,
                                                           float inv_batch, Norm nm,
                                                           float* __restrict__ part,
                                                           float* __restrict__ loss_part) {
    __shared__ float lw[kNParams];         // W1, b1, (W2 unused here), b2, W3, b3
    __shared__ alignas(16) float lw2[kH * kPad];   // W2[a][b], padded rows
    __shared__ alignas(16) float lw2t[kH * kPad];  // W2[a][b] at [b][a]
    __shared__ float xs[kGS][kIn];
    __shared__ alignas(16) float h1[kGS][kPad];    // relu(A1)
    __shared__ float a2[kGS][kPad];        // A2, later dA1
    __shared__ float d2[kGS][kPad];        // dA2
    __shared__ float zr[kGS][8];
    __shared__ float dzs[kGS], lred[kGS];
    const int t = threadIdx.x;
    for (int p = t; p < kNParams; p += kGradThreads) lw[p] = wq[p];
    for (int p = t; p < kH * kH; p += kGradThreads) {
        const float w = wq[oW2 + p];
        lw2[(p / kH) * kPad + p % kH] = w;
        lw2t[(p % kH) * kPad + p / kH] = w;
    }
    float target = 0.f;
    bool live = false;
    if (t < kGS) {
        const int64_t sidx = static_cast<int64_t>(blockIdx.x) * kGS + t;
        live = sidx < count;
        float xn[kIn] = {};
        if (live) {
            const int64_t row = idx ? idx[first + sidx] : first + sidx;
            normalise(X + row * kIn, nm, xn);
            target = T[row];
        }
#pragma unroll
        for (int i = 0; i < kIn; i++) xs[t][i] = xn[i];
    }
    __syncthreads();
    // forward: thread -> sample s, eight output units a0 .. a0 + 7
    const int s = t >> 3, a0 = (t & 7) * 8;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int a = a0 + c;
        float acc = lw[oB1 + a];
#pragma unroll
        for (int i = 0; i < kIn; i++) acc += lw[oW1 + a * kIn + i] * xs[s][i];
        h1[s][a] = acc > 0.f ? acc : 0.f;
    }
    __syncthreads();
    float zp = 0.f;
    {
        float acc[8];
#pragma unroll
        for (int c = 0; c < 8; c++) acc[c] = lw[oB2 + a0 + c];
#pragma unroll 8
        for (int b = 0; b < kH; b++) {
            float w[8];
            load8(lw2t + b * kPad + a0, w);
            const float h = h1[s][b];
#pragma unroll
            for (int c = 0; c < 8; c++) acc[c] += w[c] * h;
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int a = a0 + c;
            a2[s][a] = acc[c];
            zp += lw[oW3 + a] * (acc[c] > 0.f ? acc[c] : 0.f);
        }
    }
    zr[s][t & 7] = zp;
    __syncthreads();
    if (t < kGS) {
        float z = lw[oB3];
#pragma unroll
        for (int q = 0; q < 8; q++) z += zr[t][q];
        const float diff = live ? z - target : 0.f;
        dzs[t] = 2.f * diff * inv_batch;
        lred[t] = diff * diff;
    }
    __syncthreads();
    {  // dA2 = dz * W3 where A2 > 0
        const float dz = dzs[s];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int a = a0 + c;
            d2[s][a] = a2[s][a] > 0.f ? dz * lw[oW3 + a] : 0.f;
        }
    }
    __syncthreads();
    float* g = part + static_cast<int64_t>(blockIdx.x) * kNParams;
    {  // dW2[a][b0 .. b0+15] and db2[a] over the workgroup's samples, in order
        const int a = t >> 2, b0 = (t & 3) * 16;
        float acc[16];
#pragma unroll
        for (int c = 0; c < 16; c++) acc[c] = 0.f;
        float db2 = 0.f;
#pragma unroll 4
        for (int r = 0; r < kGS; r++) {
            const float d = d2[r][a];
            db2 += d;
            float h[2][8];
            load8(&h1[r][b0], h[0]);
            load8(&h1[r][b0 + 8], h[1]);
#pragma unroll
            for (int c = 0; c < 16; c++) acc[c] += d * h[c / 8][c % 8];
        }
#pragma unroll
        for (int c = 0; c < 16; c++) g[oW2 + a * kH + b0 + c] = acc[c];
        if ((t & 3) == 0) g[oB2 + a] = db2;
    }
    if (t < kH) {  // dW3[a] = sum_s dz * relu(A2[s][a])
        float w3 = 0.f;
        for (int r = 0; r < kGS; r++) w3 += dzs[r] * (a2[r][t] > 0.f ? a2[r][t] : 0.f);
        g[oW3 + t] = w3;
    } else if (t == kH) {
        float db3 = 0.f, l = 0.f;
        for (int r = 0; r < kGS; r++) {
            db3 += dzs[r];
            l += lred[r];
        }
        g[oB3] = db3;
        loss_part[blockIdx.x] = l;
    }
    __syncthreads();
    {  // dA1 = (W2^T dA2) where A1 > 0, written over A2
        float acc[8];
#pragma unroll
        for (int c = 0; c < 8; c++) acc[c] = 0.f;
#pragma unroll 4
        for (int a = 0; a < kH; a++) {
            const float d = d2[s][a];
            float w[8];
            load8(lw2 + a * kPad + a0, w);
#pragma unroll
            for (int c = 0; c < 8; c++) acc[c] += w[c] * d;
        }
#pragma unroll
        for (int c = 0; c < 8; c++) a2[s][a0 + c] = h1[s][a0 + c] > 0.f ? acc[c] : 0.f;
    }
    __syncthreads();
    if (t < kH) {  // dW1[a][:], db1[a]
        float db1 = 0.f;
        float w1[kIn] = {};
        for (int r = 0; r < kGS; r++) {
            const float d = a2[r][t];
            db1 += d;
#pragma unroll
            for (int i = 0; i < kIn; i++) w1[i] += d * xs[r][i];
        }
        g[oB1 + t] = db1;
#pragma unroll
        for (int i = 0; i < kIn; i++) g[oW1 + t * kIn + i] = w1[i];
    }
}

constexpr int kAdamThreads = 64;

// Sum the partial gradient rows in workgroup order; optionally apply Adam.  The
// last workgroup adds the workgroups' losses, in order, to *loss.
__global__ __launch_bounds__(kAdamThreads) void k_mlp_adam(
    const float* __restrict__ part, int nparts, float* __restrict__ grad, float* __restrict__ w,
    float* __restrict__ wq, float* __restrict__ m1, float* __restrict__ m2, float lr, float bc1,
    float bc2, int apply, const float* __restrict__ loss_part, float* __restrict__ loss) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ float lp[kAdamThreads];
        float s = 0.f;
        for (int i0 = 0; i0 < nparts; i0 += kAdamThreads) {
            const int cnt = min(kAdamThreads, nparts - i0);
            if (static_cast<int>(threadIdx.x) < cnt) lp[threadIdx.x] = loss_part[i0 + threadIdx.x];
            __syncthreads();
            if (threadIdx.x == 0)
                for (int i = 0; i < cnt; i++) s += lp[i];
            __syncthreads();
        }
        if (threadIdx.x == 0) loss[0] += s;
        return;
    }
    const int p = blockIdx.x * kAdamThreads + threadIdx.x;
    if (p >= kNParams) return;
    float g = 0.f;
    int r = 0;
    for (; r + 16 <= nparts; r += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = part[static_cast<int64_t>(r + u) * kNParams + p];
#pragma unroll
        for (int u = 0; u < 16; u++) g += v[u];
    }
    for (; r < nparts; r++) g += part[static_cast<int64_t>(r) * kNParams + p];
    grad[p] = g;
    if (!apply) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m1[p] + (1.f - b1) * g;
    const float vv = b2 * m2[p] + (1.f - b2) * g * g;
    m1[p] = mm;
    m2[p] = vv;
    const float upd = lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
    const float nw = w[p] - upd;
    w[p] = nw;
    wq[p] = bf16_round(nw);
}

__global__ __launch_bounds__(256) void k_mlp_predict(const float* __restrict__ wq,
                                                     const float* __restrict__ X, int64_t n,
                                                     Norm nm, float* __restrict__ out) {
    __shared__ float lw[kNParams];
    load_weights(wq, lw);
    __syncthreads();
    const int64_t s = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (s >= n) return;
    float xn[kIn];
    normalise(X + s * kIn, nm, xn);
    float h1[kH];
#pragma unroll
    for (int a = 0; a < kH; a++) {
        float acc = lw[oB1 + a];
#pragma unroll
        for (int i = 0; i < kIn; i++) acc += lw[oW1 + a * kIn + i] * xn[i];
        h1[a] = acc > 0.f ? acc : 0.f;
    }
    float z = lw[oB3];
    for (int a = 0; a < kH; a++) {
        float acc = lw[oB2 + a];
#pragma unroll
        for (int b = 0; b < kH; b++) acc += lw[oW2 + a * kH + b] * h1[b];
        z += lw[oW3 + a] * (acc > 0.f ? acc : 0.f);
    }
    out[s] = z;
}

template <typename T>
T* dalloc(int64_t n) {
    T* p = nullptr;
    HIPCHECK(hipMalloc(&p, std::max<int64_t>(n, 1) * sizeof(T)));
    return p;
}

}  // namespace

struct RankPredictor {
    int device = 0;
    int64_t step = 0;
    Norm norm{};
    bool norm_set = false;
    float* w = nullptr;   // FP32 master
    float* wq = nullptr;  // BF16 values (as FP32)
    float* m1 = nullptr;
    float* m2 = nullptr;
    float* grad = nullptr;
    ~RankPredictor() {
        for (float* p : {w, wq, m1, m2, grad})
            if (p) (void)hipFree(p);
    }
};

int64_t rankpred_nparams() { return kNParams; }

RankPredictor* rankpred_create(int hidden, uint64_t seed, int device) {
    if (hidden != kH) throw Error(HMX_ERR_UNSUPPORTED, "rank predictor: hidden width must be 64");
    auto p = std::make_unique<RankPredictor>();
    p->device = device;
    DeviceGuard guard(device);
    // He-uniform initialisation from a seeded generator, biases zero
    std::vector<float> w(kNParams, 0.f);
    std::mt19937_64 rng(seed);
    auto fill = [&](int off, int fan_in, int count) {
        const double lim = std::sqrt(6.0 / fan_in);
        std::uniform_real_distribution<double> u(-lim, lim);
        for (int i = 0; i < count; i++) w[off + i] = static_cast<float>(u(rng));
    };
    fill(oW1, kIn, kIn * kH);
    fill(oW2, kH, kH * kH);
    fill(oW3, kH, kH);
    std::vector<float> wq(kNParams);
    for (int i = 0; i < kNParams; i++) wq[i] = bf16_round(w[i]);
    p->w = dalloc<float>(kNParams);
    p->wq = dalloc<float>(kNParams);
    p->m1 = dalloc<float>(kNParams);
    p->m2 = dalloc<float>(kNParams);
    p->grad = dalloc<float>(kNParams);
    HIPCHECK(hipMemcpy(p->w, w.data(), kNParams * 4, hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(p->wq, wq.data(), kNParams * 4, hipMemcpyHostToDevice));
    HIPCHECK(hipMemset(p->m1, 0, kNParams * 4));
    HIPCHECK(hipMemset(p->m2, 0, kNParams * 4));
    for (int i = 0; i < kIn; i++) {
        p->norm.mean[i] = 0.f;
        p->norm.inv_std[i] = 1.f;
    }
    return p.release();
}

void rankpred_destroy(RankPredictor* p) { delete p; }

// Copy of the weights and normalisation with a fresh optimiser state (Adam
// moments zero, step 0), for fine-tuning on new data.
RankPredictor* rankpred_clone(const RankPredictor& src) {
    DeviceGuard guard(src.device);
    auto p = std::make_unique<RankPredictor>();
    p->device = src.device;
    p->norm = src.norm;
    p->norm_set = src.norm_set;
    for (float** dst : {&p->w, &p->wq, &p->m1, &p->m2, &p->grad}) *dst = dalloc<float>(kNParams);
    HIPCHECK(hipMemcpy(p->w, src.w, kNParams * 4, hipMemcpyDeviceToDevice));
    HIPCHECK(hipMemcpy(p->wq, src.wq, kNParams * 4, hipMemcpyDeviceToDevice));
    HIPCHECK(hipMemset(p->m1, 0, kNParams * 4));
    HIPCHECK(hipMemset(p->m2, 0, kNParams * 4));
    return p.release();
}

static void set_norm_from(RankPredictor& p, const float* X, int64_t n) {
    for (int i = 0; i < kIn; i++) {
        double s = 0, s2 = 0;
        for (int64_t r = 0; r < n; r++) s += X[r * kIn + i];
        const double mu = s / std::max<int64_t>(n, 1);
        for (int64_t r = 0; r < n; r++) s2 += (X[r * kIn + i] - mu) * (X[r * kIn + i] - mu);
        const double sd = std::sqrt(s2 / std::max<int64_t>(n, 1));
        p.norm.mean[i] = static_cast<float>(mu);
        p.norm.inv_std[i] = sd > 1e-6 ? static_cast<float>(1.0 / sd) : 1.f;
    }
    p.norm_set = true;
}

// One gradient evaluation over rows [first, first + count) of the (optionally
// permuted) set; leaves the summed gradient in p.grad and, if apply, takes an
// Adam step.  Returns the number of partial rows.
static int grad_pass(RankPredictor& p, const float* dX, const float* dT, const int32_t* didx,
                     int64_t first, int64_t count, float* part, float* loss_part, float* dloss,
                     float lr, bool apply, hipStream_t st) {
    const int nparts = static_cast<int>((count + kGS - 1) / kGS);
    hipLaunchKernelGGL(k_mlp_grad, dim3(nparts), dim3(kGradThreads), 0, st, p.wq, dX, dT, didx,
                       first, count, 1.f / static_cast<float>(count), p.norm, part, loss_part);
    HIPCHECK(hipGetLastError());
    float bc1 = 1.f, bc2 = 1.f;
    if (apply) {
        p.step++;
        bc1 = 1.f - std::pow(0.9f, static_cast<float>(p.step));
        bc2 = 1.f - std::pow(0.999f, static_cast<float>(p.step));
    }
    hipLaunchKernelGGL(k_mlp_adam, dim3((kNParams + kAdamThreads - 1) / kAdamThreads + 1),
                       dim3(kAdamThreads), 0, st, part, nparts, p.grad, p.w, p.wq, p.m1, p.m2, lr,
                       bc1, bc2, apply ? 1 : 0, loss_part, dloss);
    HIPCHECK(hipGetLastError());
    return nparts;
}

void rankpred_train(RankPredictor& p, const float* X, const float* T, int64_t n, int epochs,
                    int batch, float lr, uint64_t seed, float* loss_hist) {
    if (n <= 0 || epochs <= 0 || batch <= 0) throw Error(HMX_ERR_ARG, "rank predictor: empty training set");
    DeviceGuard guard(p.device);
    if (!p.norm_set) set_norm_from(p, X, n);
    float* dX = dalloc<float>(n * kIn);
    float* dT = dalloc<float>(n);
    int32_t* didx = dalloc<int32_t>(n);
    const int maxparts = (batch + kGS - 1) / kGS;
    float* part = dalloc<float>(static_cast<int64_t>(maxparts) * kNParams);
    float* lpart = dalloc<float>(maxparts);
    // one loss per epoch, read back at the end: the host shuffles the next epoch while
    // the GPU runs this one
    float* dloss = dalloc<float>(epochs);
    auto cleanup = [&] {
        for (void* q : {(void*)dX, (void*)dT, (void*)didx, (void*)part, (void*)lpart, (void*)dloss})
            (void)hipFree(q);
    };
    try {
        HIPCHECK(hipMemcpy(dX, X, n * kIn * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(dT, T, n * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemset(dloss, 0, epochs * sizeof(float)));
        std::vector<int32_t> perm(n);
        std::iota(perm.begin(), perm.end(), 0);
        std::mt19937_64 rng(seed);
        for (int e = 0; e < epochs; e++) {
            std::shuffle(perm.begin(), perm.end(), rng);
            HIPCHECK(hipMemcpy(didx, perm.data(), n * 4, hipMemcpyHostToDevice));
            for (int64_t first = 0; first < n; first += batch) {
                const int64_t cnt = std::min<int64_t>(batch, n - first);
                grad_pass(p, dX, dT, didx, first, cnt, part, lpart, dloss + e, lr, true, nullptr);
            }
        }
        if (loss_hist) {
            HIPCHECK(hipMemcpy(loss_hist, dloss, epochs * sizeof(float), hipMemcpyDeviceToHost));
            for (int e = 0; e < epochs; e++) loss_hist[e] /= static_cast<float>(n);
        }
        HIPCHECK(hipDeviceSynchronize());
    } catch (...) {
        (void)hipDeviceSynchronize();
        cleanup();
        throw;
    }
    cleanup();
}

void rankpred_grad(RankPredictor& p, const float* X, const float* T, int64_t n, float* grad,
                   float* loss) {
    if (n <= 0) throw Error(HMX_ERR_ARG, "rank predictor: empty batch");
    DeviceGuard guard(p.device);
    if (!p.norm_set) set_norm_from(p, X, n);
    float* dX = dalloc<float>(n * kIn);
    float* dT = dalloc<float>(n);
    const int nparts = static_cast<int>((n + kGS - 1) / kGS);
    float* part = dalloc<float>(static_cast<int64_t>(nparts) * kNParams);
    float* lpart = dalloc<float>(nparts);
    float* dloss = dalloc<float>(1);
    auto cleanup = [&] {
        for (void* q : {(void*)dX, (void*)dT, (void*)part, (void*)lpart, (void*)dloss}) (void)hipFree(q);
    };
    try {
        HIPCHECK(hipMemcpy(dX, X, n * kIn * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(dT, T, n * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemset(dloss, 0, 4));
        grad_pass(p, dX, dT, nullptr, 0, n, part, lpart, dloss, 0.f, false, nullptr);
        HIPCHECK(hipMemcpy(grad, p.grad, kNParams * 4, hipMemcpyDeviceToHost));
        float l = 0;
        HIPCHECK(hipMemcpy(&l, dloss, 4, hipMemcpyDeviceToHost));
        if (loss) *loss = l / static_cast<float>(n);
    } catch (...) {
        (void)hipDeviceSynchronize();
        cleanup();
        throw;
    }
    cleanup();
}

void rankpred_predict(const RankPredictor& p, const float* X, int64_t n, float* z_out) {
    if (n <= 0) return;
    DeviceGuard guard(p.device);
    float* dX = dalloc<float>(n * kIn);
    float* dz = dalloc<float>(n);
    try {
        HIPCHECK(hipMemcpy(dX, X, n * kIn * 4, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_mlp_predict, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                           nullptr, p.wq, dX, n, p.norm, dz);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipMemcpy(z_out, dz, n * 4, hipMemcpyDeviceToHost));
    } catch (...) {
        (void)hipFree(dX);
        (void)hipFree(dz);
        throw;
    }
    (void)hipFree(dX);
    (void)hipFree(dz);
}

void rankpred_params(RankPredictor& p, float* master, float* bf16, float* norm, bool get) {
    DeviceGuard guard(p.device);
    if (get) {
        if (master) HIPCHECK(hipMemcpy(master, p.w, kNParams * 4, hipMemcpyDeviceToHost));
        if (bf16) HIPCHECK(hipMemcpy(bf16, p.wq, kNParams * 4, hipMemcpyDeviceToHost));
        if (norm)
            for (int i = 0; i < kIn; i++) {
                norm[i] = p.norm.mean[i];
                norm[kIn + i] = p.norm.inv_std[i];
            }
        return;
    }
    if (master) {
        std::vector<float> q(kNParams);
        for (int i = 0; i < kNParams; i++) q[i] = bf16_round(master[i]);
        HIPCHECK(hipMemcpy(p.w, master, kNParams * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(p.wq, q.data(), kNParams * 4, hipMemcpyHostToDevice));
        HIPCHECK(hipMemset(p.m1, 0, kNParams * 4));
        HIPCHECK(hipMemset(p.m2, 0, kNParams * 4));
        p.step = 0;
    }
    if (norm) {
        for (int i = 0; i < kIn; i++) {
            p.norm.mean[i] = norm[i];
            p.norm.inv_std[i] = norm[kIn + i];
        }
        p.norm_set = true;
    }
}

}  // namespace hmx
