// aca_gpu.hip -- batched FP64 ACA+ on the GPU with a rank capacity per block.
//
// Restates ACA_plus (aca.jl:36-106) for built-in kernels: one 256-thread
// workgroup per admissible block runs the adaptive cross approximation with
// the reference's pivot rules (aca.jl:65-87), residual order (aca.jl:43-57),
// term normalisation (aca.jl:92-93) and stop test (aca.jl:95-99).  Every
// element of a residual row / column is computed by one thread in the same
// operation order as the host restatement (contraction off), the pivot search
// is a total-order argmax (largest |r|, lowest index on ties), and the stop
// test's sums of squares use the fixed 256-lane order of sumsq_lanes, so the
// factors are bit-identical to the host ACA+.
//
// Each block gets term slots for `cap` terms (the rank capacity, e.g. from the
// rank predictor).  A block that reaches its capacity without meeting the stop
// test is not finished: its state (terms, last residual row and column, used
// pivots) is kept and it continues in the next pass with a doubled capacity.
// Because ACA+ is sequential and deterministic, capping and continuing gives
// exactly the factors of an uncapped run; the capacity only changes the
// schedule (passes, launches) and the padding (slots never filled).
#include "device_op.hpp"

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <iterator>
#include <numeric>

namespace hmx {

namespace {

constexpr int kAcaThreads = 256;
static_assert(kAcaThreads == kSumLanes, "stop-test sum order is defined over 256 lanes");

struct AcaTask {
    int64_t t0, s0;  // first permuted target row / source column
    int64_t uoff;    // term q of U at U + uoff + q*m
    int64_t voff;    // term q of V at V + voff + q*n
    int64_t woff;    // residual row (n) then residual column (m) at work + woff
    int64_t foff;    // used-column (n) then used-row (m) flags at flags + foff
    int32_t m, n;
    int32_t kcap;    // term slots of this pass
    int32_t kmax;    // min(m, n)  (aca.jl:60 with max_iter = n_rows)
    int32_t sid;     // state index
    int32_t pad;
};

struct AcaState {
    int32_t k;
    int32_t done;
};

struct Best {
    double v;
    int i;
};

// (vb, ib) replaces (va, ia): larger value under isless (NaN largest), lower
// index on ties; index -1 is "none".
__device__ __forceinline__ bool better(double vb, int ib, double va, int ia) {
    if (ib < 0) return false;
    if (ia < 0) return true;
    const bool na = isnan(va), nb = isnan(vb);
    if (na || nb) return na && nb ? ib < ia : nb;
    if (vb != va) return vb > va;
    return ib < ia;
}

// argmax_not_in_list(abs.(r), used) (aca.jl:9-17) over len entries.
__device__ Best block_argmax(const double* r, const uint8_t* used, int len, Best* lds) {
    Best b{0.0, -1};
    for (int j = threadIdx.x; j < len; j += kAcaThreads) {
        if (used[j]) continue;
        const double a = fabs(r[j]);
        if (better(a, j, b.v, b.i)) b = Best{a, j};
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double ov = __shfl_xor(b.v, off);
        const int oi = __shfl_xor(b.i, off);
        if (better(ov, oi, b.v, b.i)) b = Best{ov, oi};
    }
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = b;
    __syncthreads();
    Best r0 = lds[0];
#pragma unroll
    for (int w = 1; w < kAcaThreads / 64; w++)
        if (better(lds[w].v, lds[w].i, r0.v, r0.i)) r0 = lds[w];
    __syncthreads();
    return r0;
}

// Fold the 256 lane partials: p[l] += p[l + off], off = 128 ... 1.
__device__ void tree_fold2(double* pa, double* pb) {
#pragma clang fp contract(off)
    for (int off = kAcaThreads / 2; off >= 1; off >>= 1) {
        if (static_cast<int>(threadIdx.x) < off) {
            pa[threadIdx.x] = pa[threadIdx.x] + pa[threadIdx.x + off];
            pb[threadIdx.x] = pb[threadIdx.x] + pb[threadIdx.x + off];
        }
        __syncthreads();
    }
}

// Entry (i, j) of the permuted matrix: xt / xs hold the coordinates of the point
// of every permuted index; for the dipole tensor ct / cs hold each index's
// component (its degree of freedom within the point).
__device__ inline double aca_entry(int kid, const double* xt, const int8_t* ct, const double* xs,
                                   const int8_t* cs, int64_t i, int64_t j) {
#pragma clang fp contract(off)
    const double* a = xt + 3 * i;
    const double* b = xs + 3 * j;
    if (kid == HMX_KERNEL_DIPOLE)
        return dip_component(ct[i], cs[j], a[0] - b[0], a[1] - b[1], a[2] - b[2]);
    return kernel_entry(kid, a, b);
}

__global__ __launch_bounds__(kAcaThreads) void k_aca(const AcaTask* __restrict__ tasks,
                                                     AcaState* __restrict__ states,
                                                     const double* __restrict__ xt,
                                                     const double* __restrict__ xs,
                                                     const int8_t* __restrict__ ct,
                                                     const int8_t* __restrict__ cs,
                                                     double* U, double* V,
                                                     double* __restrict__ work,
                                                     uint8_t* __restrict__ flags, int kid,
                                                     double eps) {
#pragma clang fp contract(off)
    const AcaTask T = tasks[blockIdx.x];
    const AcaState st0 = states[T.sid];
    if (st0.done) return;
    const int m = T.m, n = T.n, tid = threadIdx.x;
    double* rrow = work + T.woff;
    double* rcol = rrow + n;
    uint8_t* usedc = flags + T.foff;
    uint8_t* usedr = usedc + n;
    double* Ub = U + T.uoff;
    double* Vb = V + T.voff;
    __shared__ Best red[kAcaThreads / 64];
    __shared__ double pu[kAcaThreads], pv[kAcaThreads];
    int k = st0.k;
    int done = 0;

    // calc_residual_rows / calc_residual_cols (aca.jl:43-57)
    auto residual_row = [&](int I) {
        for (int j = tid; j < n; j += kAcaThreads) {
            double e = aca_entry(kid, xt, ct, xs, cs, T.t0 + I, T.s0 + j);
            for (int q = 0; q < k; q++)
                e = e - Ub[static_cast<int64_t>(q) * m + I] * Vb[static_cast<int64_t>(q) * n + j];
            rrow[j] = e;
        }
        __syncthreads();
    };
    auto residual_col = [&](int J) {
        for (int i = tid; i < m; i += kAcaThreads) {
            double e = aca_entry(kid, xt, ct, xs, cs, T.t0 + i, T.s0 + J);
            for (int q = 0; q < k; q++)
                e = e - Ub[static_cast<int64_t>(q) * m + i] * Vb[static_cast<int64_t>(q) * n + J];
            rcol[i] = e;
        }
        __syncthreads();
    };

    while (k < T.kmax && k < T.kcap) {
        int rp = 0, cp = 0;
        double rval = 0.0, cval = 0.0;  // first step: pivot (1,1) of a zero residual
        if (k > 0) {
            const Best bc = block_argmax(rrow, usedc, n, red);
            const Best br = block_argmax(rcol, usedr, m, red);
            cp = bc.i;
            cval = bc.v;
            rp = br.i;
            rval = br.v;
        }
        if (rval > cval) {  // aca.jl:79-87
            residual_row(rp);
            cp = block_argmax(rrow, usedc, n, red).i;
            residual_col(cp);
        } else {
            residual_col(cp);
            rp = block_argmax(rcol, usedr, m, red).i;
            residual_row(rp);
        }
        const double piv = rrow[cp];
        double su = 0.0, sv = 0.0;
        for (int j = tid; j < n; j += kAcaThreads) {  // aca.jl:92
            const double v = rrow[j] / piv;
            Vb[static_cast<int64_t>(k) * n + j] = v;
            const double sq = v * v;
            sv = sv + sq;
        }
        for (int i = tid; i < m; i += kAcaThreads) {  // aca.jl:93
            const double u = rcol[i];
            Ub[static_cast<int64_t>(k) * m + i] = u;
            const double sq = u * u;
            su = su + sq;
        }
        pu[tid] = su;
        pv[tid] = sv;
        if (tid == 0) {
            usedr[rp] = 1;
            usedc[cp] = 1;
        }
        __syncthreads();
        tree_fold2(pu, pv);
        const double step = sqrt(pu[0] * pv[0]);  // aca.jl:95
        __syncthreads();
        k++;
        if (step < eps) {  // aca.jl:97-99
            done = 1;
            break;
        }
    }
    if (k >= T.kmax) done = 1;
    if (tid == 0) states[T.sid] = AcaState{k, done};
}

// Copy the first `len` doubles of each segment (continuation of a block into
// a larger slot).  One workgroup per segment.
struct Seg {
    int64_t src, dst, len;
};

__global__ __launch_bounds__(256) void k_copy_segs(const Seg* __restrict__ segs,
                                                   const double* __restrict__ from,
                                                   double* __restrict__ to) {
    const Seg s = segs[blockIdx.x];
    for (int64_t i = threadIdx.x; i < s.len; i += 256) to[s.dst + i] = from[s.src + i];
}

// ---- recompression (SVD_recompress, aca.jl:123-143) on the device ------------------
// On the ACA+ terms still in the slot pool: Householder QR of U (m x k) and V'
// (n x k) in place (k_rec_qr, a wave or four per side), the k x k core R_U R_V',
// one-sided Jacobi SVD, truncation (k_rec_core, a wave per block), then U' = Q_U
// (W_r S_r) and V = (Q_V Z_r)' (k_rec_apply, a wave per eight columns).  The
// operation order is the host's (svd_recompress): reflector sums in the 64-lane
// order of dot_lanes64, every other sum sequential in one lane, contraction
// off, so the factors are bit-identical to the host recompression.  The
// helpers are inlined: as called functions they made the kernels reserve up to 212
// VGPRs, and the recompression was 5% slower (measured when two kernels of one wave
// per block did all of it).
struct RecTask {
    int64_t uoff, voff;  // ACA terms: U m x k, V' n x k, column-major, in the pool
    int64_t soff;        // scratch: M, Z, W, Z2 (k*k each), nrm, sig, ord, tu, tv (k each)
    int64_t ooff;        // output: U' (m x r column-major) then V (r x n row-major)
    int32_t m, n, k, r;
};

// Order the memory operations of one wave: its lanes' earlier stores are seen by its
// lanes' later loads.  The vector memory and LDS operations of a wave are processed in
// order, so nothing is waited for (a workgroup barrier waits for every store).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double wave_fold(double p) {
#pragma clang fp contract(off)
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) p = p + __shfl_down(p, off);
    return __shfl(p, 0);
}

// The folds of eight values at once: w[q] = wave_fold(p[q]) bit for bit.  Each
// level adds the same two lanes' values (in either order), but after the first one a
// half wave carries four of the eight sums, after the second a quarter two, and then
// every lane one: 10 exchanges instead of 48.
__device__ __forceinline__ void wave_fold8(const double (&p)[8], double (&w)[8], int lane) {
#pragma clang fp contract(off)
    double a[4], b[2];
    const bool h32 = lane & 32, h16 = lane & 16, h8 = lane & 8;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const double keep = h32 ? p[q + 4] : p[q], send = h32 ? p[q] : p[q + 4];
        a[q] = keep + __shfl_xor(send, 32);
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const double keep = h16 ? a[q + 2] : a[q], send = h16 ? a[q] : a[q + 2];
        b[q] = keep + __shfl_xor(send, 16);
    }
    const double keep = h8 ? b[1] : b[0], send = h8 ? b[0] : b[1];
    double c = keep + __shfl_xor(send, 8);
#pragma unroll
    for (int off = 4; off >= 1; off >>= 1) c = c + __shfl_xor(c, off);
#pragma unroll
    for (int q = 0; q < 8; q++)  // sum q sits in the eight lanes from this one on
        w[q] = __shfl(c, (q & 4 ? 32 : 0) + (q & 2 ? 16 : 0) + (q & 1 ? 8 : 0));
}

// sum_i x[i*sx] * y[i*sy], i < n, in the 64-lane order
__device__ __forceinline__ double wave_dot(const double* x, int64_t sx, const double* y, int64_t sy, int n,
                           int lane) {
#pragma clang fp contract(off)
    double p = 0.0;
    for (int i = lane; i < n; i += 64) {
        const double pr = x[i * sx] * y[i * sy];
        p = p + pr;
    }
    return wave_fold(p);
}

// Apply the reflector (1, a[j+1..m)) with factor t to columns c0 .. c0+nc-1
// (nc <= kReflCols) of B, element i of column c at B[c*cs + i*es]:
//   w = (b[j] + sum_{i>j} a[i] b[i]) * t;  b[j] -= w;  b[i] -= a[i] w.
// Every column keeps the operation order of one wave_dot and one update (lane
// partial sums over i = lane + 64 s, then the shuffle fold), so the result is
// the same bit for bit; the columns share one pass over a and one pair of
// barriers instead of one each.
constexpr int kReflCols = 8;

template <int NC>
__device__ __forceinline__ void reflect_cols_n(const double* a, int m, int j, double t, double* B,
                                               int64_t cs, int64_t es, int c0, int lane) {
#pragma clang fp contract(off)
    static_assert(kReflCols == 8, "wave_fold8");
    double* col[NC];
    double p[8], bj[NC], w[8];
#pragma unroll
    for (int q = NC; q < 8; q++) p[q] = 0.0;
#pragma unroll
    for (int q = 0; q < NC; q++) {
        col[q] = B + (c0 + q) * cs;
        p[q] = 0.0;
        bj[q] = col[q][j * es];
    }
    for (int i = j + 1 + lane; i < m; i += 64) {
        const double ai = a[i];
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const double pr = ai * col[q][i * es];
            p[q] = p[q] + pr;
        }
    }
    wave_fold8(p, w, lane);
#pragma unroll
    for (int q = 0; q < NC; q++) {
        w[q] = bj[q] + w[q];
        w[q] = w[q] * t;
    }
    wave_sync();
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NC; q++) col[q][j * es] = bj[q] - w[q];
    }
    for (int i = j + 1 + lane; i < m; i += 64) {
        const double ai = a[i];
#pragma unroll
        for (int q = 0; q < NC; q++) {
            double* b = col[q] + i * es;
            *b = *b - ai * w[q];
        }
    }
    wave_sync();
}

__device__ __forceinline__ void reflect_cols(const double* a, int m, int j, double t, double* B,
                                             int64_t cs, int64_t es, int c0, int nc, int lane) {
    switch (nc) {
    case 1: reflect_cols_n<1>(a, m, j, t, B, cs, es, c0, lane); break;
    case 2: reflect_cols_n<2>(a, m, j, t, B, cs, es, c0, lane); break;
    case 3: reflect_cols_n<3>(a, m, j, t, B, cs, es, c0, lane); break;
    case 4: reflect_cols_n<4>(a, m, j, t, B, cs, es, c0, lane); break;
    case 5: reflect_cols_n<5>(a, m, j, t, B, cs, es, c0, lane); break;
    case 6: reflect_cols_n<6>(a, m, j, t, B, cs, es, c0, lane); break;
    case 7: reflect_cols_n<7>(a, m, j, t, B, cs, es, c0, lane); break;
    default: reflect_cols_n<8>(a, m, j, t, B, cs, es, c0, lane); break;
    }
}

// Householder QR of A (m x k) in place by WAVES waves of a workgroup.  Every wave forms
// the norm of the reflector's column by itself (the same bits), the waves share its
// scaling and the columns it is applied to; each column keeps its order of operations.
template <int WAVES>
__device__ __forceinline__ void group_qr(int m, int k, double* A, double* tau) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    auto sync = [] {
        if constexpr (WAVES == 1)
            wave_sync();
        else
            __syncthreads();
    };
    for (int j = 0; j < k; j++) {
        double* a = A + static_cast<int64_t>(j) * m;
        const double alpha = a[j];
        const double xs = wave_dot(a + j + 1, 1, a + j + 1, 1, m - j - 1, lane);
        if (xs == 0.0) {
            if (threadIdx.x == 0) tau[j] = 0.0;
            sync();
            continue;
        }
        const double nrm = sqrt(alpha * alpha + xs);
        const double beta = alpha >= 0.0 ? -nrm : nrm;
        const double t = (beta - alpha) / beta;
        const double scale = 1.0 / (alpha - beta);
        sync();  // every wave has read the column
        for (int i = j + 1 + threadIdx.x; i < m; i += 64 * WAVES) a[i] = a[i] * scale;
        if (threadIdx.x == 0) {
            a[j] = beta;
            tau[j] = t;
        }
        sync();
        // columns per pass: kReflCols, fewer where that leaves a wave without columns
        const int left = k - j - 1, per = min(kReflCols, (left + WAVES - 1) / WAVES);
        for (int c = j + 1 + wave * per; c < k; c += WAVES * per)
            reflect_cols(a, m, j, t, A, m, 1, c, min(per, k - c), lane);
        sync();
    }
}

// C <- Q C for nc <= 8 columns of length m (column q at C + q*m), with the columns
// in registers: lane l holds rows l + 64 s, s < SLOTS (m <= 64 * SLOTS).  A
// reflector's sums keep the order of reflect_cols: the lane that holds row i adds its
// products in the order of s, and the partial sums are rotated to the lane (i - j - 1)
// % 64 before the fold.
template <int SLOTS>
__device__ __forceinline__ void wave_apply_regs(int m, int k, const double* A, const double* tau,
                                                double (&c)[SLOTS][8], int lane) {
#pragma clang fp contract(off)
    double an[SLOTS];
    auto load = [&](int j, double (&a)[SLOTS]) {
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
            const int i = lane + 64 * s;
            a[s] = i < m ? A[static_cast<int64_t>(j) * m + i] : 0.0;
        }
    };
    load(k - 1, an);
    for (int j = k - 1; j >= 0; j--) {
        double a[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; s++) a[s] = an[s];
        if (j > 0) load(j - 1, an);  // the next reflector, while this one is applied
        const double t = tau[j];
        if (t == 0.0) continue;
        double p[8], bj[8], w[8];
        const int from = (lane + j + 1) & 63;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            double x = 0.0, y = c[0][q];
#pragma unroll
            for (int s = 0; s < SLOTS; s++) {
                const int i = lane + 64 * s;
                const double pr = a[s] * c[s][q];
                if (i > j && i < m) x = x + pr;
                if (s == j >> 6) y = c[s][q];
            }
            p[q] = __shfl(x, from);
            bj[q] = __shfl(y, j & 63);
        }
        wave_fold8(p, w, lane);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            w[q] = bj[q] + w[q];
            w[q] = w[q] * t;
#pragma unroll
            for (int s = 0; s < SLOTS; s++) {
                const int i = lane + 64 * s;
                if (i == j)
                    c[s][q] = bj[q] - w[q];
                else if (i > j && i < m)
                    c[s][q] = c[s][q] - a[s] * w[q];
            }
        }
    }
}

// R_U R_V' -> one-sided Jacobi SVD -> sorted singular values, W, Z2 and the
// truncation rank.  M and Z (k x k) live in LDS up to k = kLdsK and in the block's
// global scratch beyond; the arithmetic and its order are the same either way.
// In LDS a column has an odd stride, so that the lanes of a round, each in
// another column, read distinct banks (an even one put all 16 pairs of k = 32 on
// one bank).  The LDS of a launch is sized by its k class (kRecClass).  Cores of
// k > 32 used to rotate in global memory: of the 79,786 blocks at N = 32,768 (tol
// 1e-6) the 17,815 of k > 32 took 116 of the 150 ms of the kernel, and now 31.
constexpr int kLdsK = 64;
constexpr int kRecClass[] = {32, 40, kLdsK};
__host__ __device__ constexpr int rec_stride(int k) { return k | 1; }
constexpr size_t rec_lds_bytes(int k) { return size_t(2) * k * rec_stride(k) * sizeof(double); }

template <bool IN_LDS>
__device__ __forceinline__ void rec_svd(RecTask& T, const double* QU, const double* QV, double* M,
                                        double* Z, double* W, double* Z2, double* nrm, double* sig,
                                        double* ord, int m, int n, int k, double eps, int lane) {
#pragma clang fp contract(off)
    const int ld = IN_LDS ? rec_stride(k) : k;  // column stride of M and Z
    for (int idx = lane; idx < k * k; idx += 64) {  // (R_U R_V')[i, j]
        const int i = idx % k, j = idx / k;
        double s = 0.0;
        for (int l = max(i, j); l < k; l++) {
            const double pr = QU[i + static_cast<int64_t>(l) * m] * QV[j + static_cast<int64_t>(l) * n];
            s = s + pr;
        }
        M[i + j * ld] = s;
        Z[i + j * ld] = i == j ? 1.0 : 0.0;
    }
    wave_sync();
    // one-sided Jacobi, round-robin sweeps: the k'/2 disjoint pairs of a round
    // are rotated in parallel, one lane per pair (the host does them in order;
    // disjoint rotations commute exactly)
    const double tol = 2.220446049250313e-16;
    const int kp = k + (k & 1);
    if constexpr (IN_LDS) {
        // At most 32 pairs, four lanes each (two beyond 16 pairs).  The lanes of a pair
        // share its three sums (each is one lane's, in the host's order), all form the
        // rotation (the same bits), and each applies it to its share of the elements.
        const int per = kp / 2 <= 16 ? 4 : 2;
        const int pi = lane / per, part = lane % per, first = lane - part;
        for (int sweep = 0; sweep < 80; sweep++) {
            bool rotated = false;
            for (int rnd = 0; rnd + 1 < kp; rnd++) {
                const int a = pi == 0 ? 0 : 1 + (pi - 1 + rnd) % (kp - 1);
                const int b = 1 + (kp - 2 - pi + rnd) % (kp - 1);
                const int p = min(a, b), q = max(a, b);
                const bool live = pi < kp / 2 && q < k;
                double* ap = M + (live ? p : 0) * ld;
                double* aq = M + (live ? q : 0) * ld;
                double al, be, ga;
                if (per == 4) {  // lanes 0, 1, 2: alpha, beta, gamma
                    const double* u = part == 1 ? aq : ap;
                    const double* v = part == 0 ? ap : aq;
                    double sum = 0.0;
#pragma unroll 4
                    for (int i = 0; i < k; i++) {
                        const double uv = u[i] * v[i];
                        sum = sum + uv;
                    }
                    al = __shfl(sum, first);
                    be = __shfl(sum, first + 1);
                    ga = __shfl(sum, first + 2);
                } else {  // lane 0: alpha and gamma, lane 1: beta (and gamma again)
                    const double* u = part == 1 ? aq : ap;
                    double sum = 0.0, cross = 0.0;
#pragma unroll 4
                    for (int i = 0; i < k; i++) {
                        const double uu = u[i] * u[i], xy = ap[i] * aq[i];
                        sum = sum + uu;
                        cross = cross + xy;
                    }
                    al = __shfl(sum, first);
                    be = __shfl(sum, first + 1);
                    ga = cross;
                }
                if (live && !(ga == 0.0 || fabs(ga) <= tol * sqrt(al * be))) {
                    rotated = true;
                    const double zeta = (be - al) / (2.0 * ga);
                    const double t =
                        (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
                    const double c = 1.0 / sqrt(1.0 + t * t);
                    const double s = c * t;
                    double* zp = Z + p * ld;
                    double* zq = Z + q * ld;
                    for (int i = part; i < k; i += per) {
                        const double x = ap[i], y = aq[i];
                        ap[i] = c * x - s * y;
                        aq[i] = s * x + c * y;
                        const double zx = zp[i], zy = zq[i];
                        zp[i] = c * zx - s * zy;
                        zq[i] = s * zx + c * zy;
                    }
                }
                wave_sync();
            }
            if (!__any(rotated)) break;
        }
    } else {
        for (int sweep = 0; sweep < 80; sweep++) {
            bool rotated = false;
            for (int rnd = 0; rnd + 1 < kp; rnd++) {
                for (int pi = lane; pi < kp / 2; pi += 64) {
                    const int a = pi == 0 ? 0 : 1 + (pi - 1 + rnd) % (kp - 1);
                    const int b = 1 + (kp - 2 - pi + rnd) % (kp - 1);
                    const int p = min(a, b), q = max(a, b);
                    if (q >= k) continue;
                    double* ap = M + p * ld;
                    double* aq = M + q * ld;
                    double al = 0.0, be = 0.0, ga = 0.0;
                    for (int i = 0; i < k; i++) {
                        const double x = ap[i], y = aq[i];
                        const double xx = x * x, yy = y * y, xy = x * y;
                        al = al + xx;
                        be = be + yy;
                        ga = ga + xy;
                    }
                    if (ga == 0.0 || fabs(ga) <= tol * sqrt(al * be)) continue;
                    rotated = true;
                    const double zeta = (be - al) / (2.0 * ga);
                    const double t =
                        (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
                    const double c = 1.0 / sqrt(1.0 + t * t);
                    const double s = c * t;
                    double* zp = Z + p * ld;
                    double* zq = Z + q * ld;
                    for (int i = 0; i < k; i++) {
                        const double x = ap[i], y = aq[i];
                        ap[i] = c * x - s * y;
                        aq[i] = s * x + c * y;
                        const double zx = zp[i], zy = zq[i];
                        zp[i] = c * zx - s * zy;
                        zq[i] = s * zx + c * zy;
                    }
                }
                wave_sync();
            }
            if (!__any(rotated)) break;
        }
    }
    for (int j = lane; j < k; j += 64) {
        double s = 0.0;
        for (int i = 0; i < k; i++) {
            const double pr = M[i + j * ld] * M[i + j * ld];
            s = s + pr;
        }
        nrm[j] = sqrt(s);
    }
    wave_sync();
    if (lane == 0) {  // stable sort by descending norm
        for (int j = 0; j < k; j++) ord[j] = j;
        for (int j = 1; j < k; j++) {
            const double key = ord[j];
            int x = j - 1;
            while (x >= 0 && nrm[static_cast<int>(ord[x])] < nrm[static_cast<int>(key)]) {
                ord[x + 1] = ord[x];
                x--;
            }
            ord[x + 1] = key;
        }
    }
    wave_sync();
    for (int idx = lane; idx < k * k; idx += 64) {
        const int i = idx % k, j = idx / k, o = static_cast<int>(ord[j]);
        W[i + j * k] = nrm[o] > 0.0 ? M[i + o * ld] / nrm[o] : 0.0;
        Z2[i + j * k] = Z[i + o * ld];
    }
    for (int j = lane; j < k; j += 64) sig[j] = nrm[static_cast<int>(ord[j])];
    wave_sync();
    if (lane == 0) {  // reverse(sqrt.(cumsum(reverse(sig.^2)))), first index below eps
        double acc = 0.0;
        for (int i = k - 1; i >= 0; i--) {
            const double s2 = sig[i] * sig[i];
            acc = (i == k - 1) ? s2 : acc + s2;
            nrm[i] = sqrt(acc);
        }
        int r = k;
        for (int i = 0; i < k; i++)
            if (nrm[i] < eps) {
                r = i;
                break;
            }
        T.r = r;
    }
}

// QR of one side of a block (blockIdx.y: U, V), WAVES waves.  With one wave a block
// that fits the launch's LDS is factored there: its chain of short passes is bound by
// their latency.  The blocks of more than kWideRows rows on a side take four waves: with
// one wave for both sides of every block the largest blocks alone set the time of the
// launch (N = 32,768, tol 1e-6: QR and core together 66 -> 60 ms, of which the QR 23).
constexpr int kWideRows = 512;
constexpr int kQrLds = 2112;  // doubles: 64 x 33

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_rec_qr(const RecTask* __restrict__ tasks,
                                                       const int32_t* __restrict__ which,
                                                       double* pool, double* scratch) {
    const RecTask& T = tasks[which[blockIdx.x]];
    const bool vside = blockIdx.y == 1;
    const int m = vside ? T.n : T.m, k = T.k;
    if (k == 0) return;
    double* A = pool + (vside ? T.voff : T.uoff);
    double* tau = scratch + T.soff + 4 * k * k + (vside ? 4 : 3) * k;
    if constexpr (WAVES == 1) {
        __shared__ double lds[kQrLds];
        const int64_t len = static_cast<int64_t>(m) * k;
        if (len <= kQrLds) {
            for (int i = threadIdx.x; i < len; i += 64) lds[i] = A[i];
            wave_sync();
            group_qr<1>(m, k, lds, tau);
            for (int i = threadIdx.x; i < len; i += 64) A[i] = lds[i];
            return;
        }
    }
    group_qr<WAVES>(m, k, A, tau);
}

// Core SVD of a block whose two sides are factored.
__global__ __launch_bounds__(64) void k_rec_core(RecTask* __restrict__ tasks, const double* pool,
                                                 double* __restrict__ scratch, double eps) {
#pragma clang fp contract(off)
    RecTask& T = tasks[blockIdx.x];
    const int lane = threadIdx.x, m = T.m, n = T.n, k = T.k;
    if (k == 0) {
        if (lane == 0) T.r = 0;
        return;
    }
    const double* QU = pool + T.uoff;
    const double* QV = pool + T.voff;
    double* M = scratch + T.soff;
    double* Z = M + k * k;
    double* W = Z + k * k;
    double* Z2 = W + k * k;
    double* nrm = Z2 + k * k;
    double* sig = nrm + k;
    double* ord = sig + k;  // followed by the reflector factors of U and of V
    extern __shared__ double mz[];
    if (k <= kLdsK)
        rec_svd<true>(T, QU, QV, mz, mz + k * rec_stride(k), W, Z2, nrm, sig, ord, m, n, k, eps, lane);
    else
        rec_svd<false>(T, QU, QV, M, Z, W, Z2, nrm, sig, ord, m, n, k, eps, lane);
}

// U' = Q_U (W_r S_r) and V = (Q_V Z_r)', eight columns of one of them per wave
// (blockIdx.y: side, then column chunk; the columns of a side do not depend on each
// other).  With a wave per block the launch lasted as long as its largest block: one
// wave walked k reflectors over all columns of both sides.  Columns of up to 256 rows
// stay in registers from the first reflector to the last.  N = 32,768, tol
// 1e-6: 44 -> 23 ms.
template <int SLOTS>
__device__ __forceinline__ void rec_apply_regs(int m, int k, int nc, const double* A,
                                               const double* tau, const double* W,
                                               const double* sig, double* out, int lane) {
#pragma clang fp contract(off)
    double c[SLOTS][8];
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
        const int i = lane + 64 * s;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            c[s][q] = 0.0;
            if (q < nc && i < k) c[s][q] = sig ? W[i + q * k] * sig[q] : W[i + q * k];
        }
    }
    wave_apply_regs<SLOTS>(m, k, A, tau, c, lane);
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
        const int i = lane + 64 * s;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (q < nc && i < m) out[static_cast<int64_t>(q) * m + i] = c[s][q];
    }
}

__global__ __launch_bounds__(64) void k_rec_apply(const RecTask* __restrict__ tasks,
                                                  const double* __restrict__ pool,
                                                  const double* __restrict__ scratch,
                                                  double* __restrict__ out, int chunks) {
#pragma clang fp contract(off)
    const RecTask T = tasks[blockIdx.x];
    const bool vside = static_cast<int>(blockIdx.y) >= chunks;
    const int c0 = (static_cast<int>(blockIdx.y) - (vside ? chunks : 0)) * kReflCols;
    const int lane = threadIdx.x, k = T.k, r = T.r, m = vside ? T.n : T.m;
    if (c0 >= r) return;
    const int nc = min(kReflCols, r - c0);
    const double* base = scratch + T.soff;
    const double* W = base + (vside ? 3 : 2) * k * k + static_cast<int64_t>(c0) * k;
    const double* sig = vside ? nullptr : base + 4 * k * k + k + c0;
    const double* tau = base + 4 * k * k + (vside ? 4 : 3) * k;
    const double* A = pool + (vside ? T.voff : T.uoff);
    // U: m x r column-major; then V: r x n, row-major
    double* O = out + T.ooff + (vside ? static_cast<int64_t>(T.m) * r : 0) + static_cast<int64_t>(c0) * m;
    if (m <= 64)
        rec_apply_regs<1>(m, k, nc, A, tau, W, sig, O, lane);
    else if (m <= 128)
        rec_apply_regs<2>(m, k, nc, A, tau, W, sig, O, lane);
    else if (m <= 256)
        rec_apply_regs<4>(m, k, nc, A, tau, W, sig, O, lane);
    else {
        for (int64_t idx = lane; idx < static_cast<int64_t>(m) * nc; idx += 64) {
            const int i = static_cast<int>(idx % m), q = static_cast<int>(idx / m);
            O[idx] = i < k ? (sig ? W[i + q * k] * sig[q] : W[i + q * k]) : 0.0;
        }
        wave_sync();
        for (int j = k - 1; j >= 0; j--) {
            const double t = tau[j];
            if (t == 0.0) continue;
            reflect_cols(A + static_cast<int64_t>(j) * m, m, j, t, O, m, 1, 0, nc, lane);
        }
    }
}

int64_t round_cap(int64_t c, int64_t kmax) {
    c = std::max<int64_t>(4, (c + 3) / 4 * 4);
    return std::min(c, kmax);
}

}  // namespace

int64_t aca_round_cap(int64_t c, int64_t kmax) { return round_cap(c, kmax); }

void gpu_aca(const HMatrix& h, const std::vector<AcaBlock>& blocks, std::vector<int32_t> caps,
             double eps, double svd_eps, int nthreads, AcaStats* stats, const AcaDone& on_done,
             const AcaSlabDone& on_slab, const std::vector<int64_t>& probe, const AcaRefine& refine) {
    // The 1/r kernel and the dipole tensor: their entries (subtractions,
    // products, sqrt, division) are correctly rounded on both sides, so the
    // device reproduces the host factors exactly; the log kernel's device log()
    // is not guaranteed to match the host's.
    const int kid = h.src.kernel_id;
    if (kid == HMX_KERNEL_LAPLACE) {
        if (h.target_dims != 1 || h.source_dims != 1)
            throw Error(HMX_ERR_UNSUPPORTED, "GPU ACA+ with the 1/r kernel needs dims == 1");
    } else if (kid == HMX_KERNEL_DIPOLE) {
        if (h.target_dims != 3 || h.source_dims != 3)
            throw Error(HMX_ERR_UNSUPPORTED, "GPU ACA+ with the dipole tensor needs dims == 3");
    } else {
        throw Error(HMX_ERR_UNSUPPORTED,
                    "GPU ACA+ supports the built-in 1/r kernel and the dipole tensor");
    }
    DeviceGuard guard(h.device);
    AcaStats S{};
    const auto wall0 = std::chrono::steady_clock::now();

    // Permuted coordinates: permuted index p is original index tmap[p] - 1,
    // which is point (tmap[p] - 1) / dims, component (tmap[p] - 1) % dims
    // (the interleaved index map of tree.jl:59-64).
    const bool dip = kid == HMX_KERNEL_DIPOLE;
    std::vector<double> xtp(3 * h.m), xsp(3 * h.n);
    std::vector<int8_t> ctp(dip ? h.m : 0), csp(dip ? h.n : 0);
    auto permuted = [&](const std::vector<int64_t>& map, const double* x, int64_t dims,
                        std::vector<double>& xp, std::vector<int8_t>& cp) {
        for (size_t p = 0; p < map.size(); p++) {
            const int64_t o = map[p] - 1, pt = o / dims;
            for (int c = 0; c < 3; c++) xp[3 * p + c] = x[3 * pt + c];
            if (!cp.empty()) cp[p] = static_cast<int8_t>(o % dims);
        }
    };
    permuted(h.tmap, h.src.xt, h.target_dims, xtp, ctp);
    permuted(h.smap, h.src.xs, h.source_dims, xsp, csp);
    double* dxt = upload(xtp);
    double* dxs = upload(xsp);
    int8_t* dct = upload(ctp);  // nullptr for the scalar kernel
    int8_t* dcs = upload(csp);
    std::vector<void*> owned = {dxt, dxs};
    if (dct) owned.push_back(dct);
    if (dcs) owned.push_back(dcs);
    auto release = [&](void* p) {
        if (!p) return;
        auto it = std::find(owned.begin(), owned.end(), p);
        if (it != owned.end()) owned.erase(it);
        (void)hipFree(p);
    };
    auto free_all = [&] {
        for (void* p : owned)
            if (p) (void)hipFree(p);
        owned.clear();
    };
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // Host side of finished blocks: their terms are packed on the device,
    // copied into one of two pinned staging buffers and handed to a worker that
    // copies recompressed factors into slabs (on_slab), or transposes V and calls
    // on_done (recompression on the host), on nthreads threads while
    // the GPU proceeds with the next pass or chunk.
    struct Staging {
        double* host = nullptr;
        int64_t cap = 0;
        std::future<void> job;
    };
    Staging stage[2];
    int next_stage = 0;
    const bool verbose = std::getenv("HMX_VERBOSE") != nullptr;
    auto wall = [&] {
        return std::chrono::duration<double>(std::chrono::steady_clock::now() - wall0).count();
    };
    auto wait_jobs = [&] {
        for (auto& st : stage)
            if (st.job.valid()) st.job.get();
    };
    auto free_staging = [&] {
        for (auto& st : stage) {
            if (st.job.valid()) st.job.wait();
            if (st.host) (void)hipHostFree(st.host);
            st.host = nullptr;
        }
    };
    try {
        HIPCHECK(hipEventCreate(&e0));
        HIPCHECK(hipEventCreate(&e1));
        HIPCHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_rec_core),
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(rec_lds_bytes(kLdsK))));
        const int64_t nb = static_cast<int64_t>(blocks.size());
        // most expensive first: cost ~ (m + n) * cap^2
        auto cost = [&](int64_t b) {
            const double c = caps[b];
            return double(blocks[b].m + blocks[b].n) * c * c;
        };
        auto by_cost = [&](std::vector<int64_t>& v) {
            std::stable_sort(v.begin(), v.end(),
                             [&](int64_t a, int64_t b) { return cost(a) > cost(b); });
        };
        // Device memory per chunk (term slots + residual workspace): a third of
        // the free memory, at most 64 GiB.  Fewer, larger chunks mean fewer
        // launches whose tails (the largest blocks, one workgroup each) leave
        // the GPU idle: measured on a 1,048,576-point planar grid, 8 -> 64 GiB
        // took the ACA+ and recompression kernels from 2.34 s to 1.71 s.
        const char* env = std::getenv("HMX_ACA_CHUNK_BYTES");
        size_t free_b = 0, total_b = 0;
        HIPCHECK(hipMemGetInfo(&free_b, &total_b));
        const int64_t budget =
            env ? std::atoll(env)
                : std::max<int64_t>(int64_t(1) << 30,
                                    std::min<int64_t>(int64_t(64) << 30, static_cast<int64_t>(free_b / 3)));
        int64_t done_blocks = 0;
        std::vector<int64_t> seen_ids;
        std::vector<int32_t> seen_ranks;
        // Hand finished blocks to the host: copy `tot` doubles at dsrc into a
        // pinned staging buffer, then a worker hands on the entries of `outs`.
        struct Out {
            int64_t block, m, n, k, aca_k, off;
        };
        auto stage_out = [&](std::vector<Out>&& outs, const double* dsrc, int64_t tot,
                             bool recompressed) {
            Staging& st = stage[next_stage];
            next_stage ^= 1;
            if (st.job.valid()) st.job.get();  // the buffer's previous job is done
            if (tot > st.cap) {
                if (st.host) HIPCHECK(hipHostFree(st.host));
                st.host = nullptr;
                st.cap = 0;
                HIPCHECK(hipHostMalloc(reinterpret_cast<void**>(&st.host), tot * sizeof(double),
                                       hipHostMallocDefault));
                st.cap = tot;
            }
            if (tot > 0)
                HIPCHECK(hipMemcpy(st.host, dsrc, tot * sizeof(double), hipMemcpyDeviceToHost));
            const double* hbuf = st.host;
            if (recompressed) {
                // consecutive blocks share a slab; at least a few slabs per thread
                const int64_t lim = std::min(kSlabBytes / 8, std::max<int64_t>(
                                                                 1 << 15, tot / (4 * std::max(1, nthreads))));
                std::vector<std::pair<size_t, size_t>> cuts;
                for (size_t a = 0; a < outs.size();) {
                    size_t b = a;
                    int64_t len = 0;
                    while (b < outs.size() && (b == a || len + outs[b].k * (outs[b].m + outs[b].n) <= lim)) {
                        len += outs[b].k * (outs[b].m + outs[b].n);
                        b++;
                    }
                    cuts.push_back({a, b});
                    a = b;
                }
                st.job = std::async(std::launch::async, [outs = std::move(outs), cuts = std::move(cuts),
                                                         hbuf, nthreads, &on_slab] {
                    parallel_for(static_cast<int64_t>(cuts.size()), nthreads, [&](int64_t c) {
                        auto s = std::make_unique<FactorSlab>();
                        const int64_t base = outs[cuts[c].first].off;
                        int64_t len = 0;
                        for (size_t q = cuts[c].first; q < cuts[c].second; q++) {
                            const Out& o = outs[q];
                            s->parts.push_back({o.block, o.aca_k, o.m, o.n, o.k, o.off - base});
                            len = o.off - base + o.k * (o.m + o.n);
                        }
                        s->data.resize(static_cast<size_t>(len));
                        advise_huge_pages(s->data.data(), static_cast<size_t>(len) * sizeof(double));
                        if (len) std::memcpy(s->data.data(), hbuf + base, static_cast<size_t>(len) * sizeof(double));
                        on_slab(std::move(s));
                    });
                });
                return;
            }
            st.job = std::async(std::launch::async, [outs = std::move(outs), hbuf, nthreads, &on_done] {
                parallel_for(static_cast<int64_t>(outs.size()), nthreads, [&](int64_t f) {
                    const Out& o = outs[f];
                    LowRank L;
                    L.m = o.m;
                    L.n = o.n;
                    L.k = o.k;
                    L.U.assign(hbuf + o.off, hbuf + o.off + o.k * o.m);
                    const double* src = hbuf + o.off + o.k * o.m;
                    L.V.resize(static_cast<size_t>(o.k * o.n));  // terms q: V row q contiguous over n
                    for (int64_t q = 0; q < o.k; q++)
                        for (int64_t j = 0; j < o.n; j++) L.V[q + j * o.k] = src[q * o.n + j];
                    on_done(o.block, o.aca_k, std::move(L));
                });
            });
        };
        // ACA+ factors as they are (recompression on the host)
        auto emit_raw = [&](const std::vector<int64_t>& finished, const std::vector<AcaTask>& tasks,
                            const std::vector<AcaState>& hstate, const double* pool,
                            const std::vector<int64_t>& order, int64_t pos) {
            std::vector<Out> outs;
            std::vector<Seg> pack;
            int64_t ptot = 0;
            for (int64_t t : finished) {
                const AcaTask& T = tasks[t];
                const int64_t k = hstate[t].k;
                outs.push_back(Out{order[pos + T.sid], T.m, T.n, k, k, ptot});
                if (k > 0) {
                    pack.push_back(Seg{T.uoff, ptot, k * T.m});
                    pack.push_back(Seg{T.voff, ptot + k * T.m, k * T.n});
                }
                ptot += k * (T.m + T.n);
            }
            double* dpack = nullptr;
            if (!pack.empty()) {
                HIPCHECK(hipMalloc(&dpack, ptot * sizeof(double)));
                owned.push_back(dpack);
                Seg* dps = upload(pack);
                owned.push_back(dps);
                hipLaunchKernelGGL(k_copy_segs, dim3(pack.size()), dim3(256), 0, nullptr, dps, pool,
                                   dpack);
                HIPCHECK(hipGetLastError());
                HIPCHECK(hipDeviceSynchronize());
                release(dps);
            }
            stage_out(std::move(outs), dpack, ptot, false);
            release(dpack);
        };
        // recompression on the device, in sub-batches of bounded scratch
        auto emit_recompressed = [&](const std::vector<int64_t>& finished,
                                     const std::vector<AcaTask>& tasks,
                                     const std::vector<AcaState>& hstate, double* pool,
                                     const std::vector<int64_t>& order, int64_t pos) {
            const int64_t rec_budget = int64_t(1) << 28;  // doubles of scratch per sub-batch
            size_t f0 = 0;
            while (f0 < finished.size()) {
                std::vector<RecTask> rt;
                std::vector<int64_t> ids;
                int64_t sc = 0;
                size_t f1 = f0;
                while (f1 < finished.size()) {
                    const AcaTask& T = tasks[finished[f1]];
                    const int64_t k = hstate[finished[f1]].k;
                    const int64_t need = 4 * k * k + 5 * k;
                    if (f1 > f0 && sc + need > rec_budget) break;
                    rt.push_back(RecTask{T.uoff, T.voff, sc, 0, T.m, T.n, static_cast<int32_t>(k), 0});
                    ids.push_back(finished[f1]);
                    sc += need;
                    f1++;
                }
                // by k class, so that each core launch reserves the LDS its blocks need
                // (beyond kLdsK first, as the longest)
                auto k_class = [](int32_t k) {
                    int c = 0;
                    for (int lim : kRecClass) c += k > lim;
                    return c;
                };
                std::vector<size_t> ord(rt.size());
                std::iota(ord.begin(), ord.end(), size_t(0));
                std::stable_sort(ord.begin(), ord.end(), [&](size_t a, size_t b) {
                    return k_class(rt[a].k) > k_class(rt[b].k);
                });
                {
                    std::vector<RecTask> rs(rt.size());
                    std::vector<int64_t> is(rt.size());
                    for (size_t q = 0; q < ord.size(); q++) {
                        rs[q] = rt[ord[q]];
                        is[q] = ids[ord[q]];
                    }
                    rt.swap(rs);
                    ids.swap(is);
                }
                double* dscr = nullptr;
                HIPCHECK(hipMalloc(&dscr, std::max<int64_t>(sc, 1) * sizeof(double)));
                owned.push_back(dscr);
                RecTask* drt = upload(rt);
                owned.push_back(drt);
                HIPCHECK(hipEventRecord(e0, nullptr));
                // the blocks whose QR takes four waves, then the others
                std::vector<int32_t> which(rt.size());
                std::iota(which.begin(), which.end(), 0);
                const size_t nwide = static_cast<size_t>(
                    std::stable_partition(which.begin(), which.end(),
                                          [&](int32_t q) {
                                              return std::max(rt[q].m, rt[q].n) > kWideRows;
                                          }) -
                    which.begin());
                int32_t* dwhich = upload(which);
                owned.push_back(dwhich);
                if (nwide > 0)
                    hipLaunchKernelGGL(k_rec_qr<4>, dim3(nwide, 2), dim3(256), 0, nullptr, drt, dwhich,
                                       pool, dscr);
                if (rt.size() > nwide)
                    hipLaunchKernelGGL(k_rec_qr<1>, dim3(rt.size() - nwide, 2), dim3(64), 0, nullptr,
                                       drt, dwhich + nwide, pool, dscr);
                HIPCHECK(hipGetLastError());
                for (size_t q0 = 0; q0 < rt.size();) {
                    const int c = k_class(rt[q0].k);
                    size_t q1 = q0;
                    while (q1 < rt.size() && k_class(rt[q1].k) == c) q1++;
                    const size_t lds = c < int(std::size(kRecClass)) ? rec_lds_bytes(kRecClass[c]) : 0;
                    hipLaunchKernelGGL(k_rec_core, dim3(q1 - q0), dim3(64), lds, nullptr, drt + q0,
                                       pool, dscr, svd_eps);
                    HIPCHECK(hipGetLastError());
                    q0 = q1;
                }
                HIPCHECK(hipMemcpy(rt.data(), drt, rt.size() * sizeof(RecTask), hipMemcpyDeviceToHost));
                std::vector<Out> outs;
                int64_t otot = 0;
                for (size_t q = 0; q < rt.size(); q++) {
                    rt[q].ooff = otot;
                    const AcaTask& T = tasks[ids[q]];
                    outs.push_back(Out{order[pos + T.sid], T.m, T.n, rt[q].r, rt[q].k, otot});
                    otot += int64_t(rt[q].r) * (T.m + T.n);
                }
                HIPCHECK(hipMemcpy(drt, rt.data(), rt.size() * sizeof(RecTask), hipMemcpyHostToDevice));
                double* dout = nullptr;
                HIPCHECK(hipMalloc(&dout, std::max<int64_t>(otot, 1) * sizeof(double)));
                owned.push_back(dout);
                int32_t rmax = 0;
                for (const RecTask& t : rt) rmax = std::max(rmax, t.r);
                const int chunks = (rmax + kReflCols - 1) / kReflCols;
                if (chunks > 0)
                    hipLaunchKernelGGL(k_rec_apply, dim3(rt.size(), 2 * chunks), dim3(64), 0, nullptr,
                                       drt, pool, dscr, dout, chunks);
                HIPCHECK(hipGetLastError());
                HIPCHECK(hipEventRecord(e1, nullptr));
                HIPCHECK(hipEventSynchronize(e1));
                float ms = 0;
                HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
                S.recompress_ms += ms;
                stage_out(std::move(outs), dout, otot, true);
                release(dout);
                release(dwhich);
                release(drt);
                release(dscr);
                f0 = f1;
            }
        };
        // Run the listed blocks (in this order) in memory-bounded chunks.
        auto run_list = [&](const std::vector<int64_t>& order, bool collect) {
        const int64_t nl = static_cast<int64_t>(order.size());
        int64_t pos = 0;
        while (pos < nl) {
            // one chunk: term slots + residual workspace within the budget
            int64_t end = pos, bytes = 0;
            while (end < nl) {
                const AcaBlock& B = blocks[order[end]];
                const int64_t c = round_cap(caps[order[end]], std::min(B.m, B.n));
                const int64_t add = (B.m + B.n) * (8 * c + 9);
                if (end > pos && bytes + add > budget) break;
                bytes += add;
                end++;
            }
            const int64_t nc = end - pos;
            std::vector<AcaTask> tasks(nc);
            int64_t wtot = 0;
            for (int64_t t = 0; t < nc; t++) {
                const AcaBlock& B = blocks[order[pos + t]];
                AcaTask& a = tasks[t];
                a.t0 = B.t0;
                a.s0 = B.s0;
                a.m = static_cast<int32_t>(B.m);
                a.n = static_cast<int32_t>(B.n);
                a.kmax = static_cast<int32_t>(std::min(B.m, B.n));
                a.kcap = static_cast<int32_t>(round_cap(caps[order[pos + t]], a.kmax));
                a.sid = static_cast<int32_t>(t);
                a.woff = wtot;
                a.foff = wtot;
                wtot += B.m + B.n;
            }
            double* work = nullptr;
            uint8_t* flags = nullptr;
            AcaState* dstate = nullptr;
            HIPCHECK(hipMalloc(&work, std::max<int64_t>(wtot, 1) * sizeof(double)));
            owned.push_back(work);
            HIPCHECK(hipMalloc(&flags, std::max<int64_t>(wtot, 1)));
            owned.push_back(flags);
            HIPCHECK(hipMalloc(&dstate, nc * sizeof(AcaState)));
            owned.push_back(dstate);
            HIPCHECK(hipMemset(work, 0, wtot * sizeof(double)));
            HIPCHECK(hipMemset(flags, 0, wtot));
            HIPCHECK(hipMemset(dstate, 0, nc * sizeof(AcaState)));
            std::vector<AcaState> hstate(nc);
            std::vector<int64_t> active(nc);
            for (int64_t t = 0; t < nc; t++) active[t] = t;
            double* pool = nullptr;  // previous pass's slots (continuing blocks)
            int pass = 0;
            while (!active.empty()) {
                // slots for the active blocks: U terms then V terms
                int64_t tot = 0;
                std::vector<Seg> segs;
                std::vector<int64_t> old_u(active.size()), old_v(active.size());
                for (size_t a = 0; a < active.size(); a++) {
                    AcaTask& T = tasks[active[a]];
                    old_u[a] = T.uoff;
                    old_v[a] = T.voff;
                    T.uoff = tot;
                    tot += int64_t(T.m) * T.kcap;
                }
                for (size_t a = 0; a < active.size(); a++) {
                    AcaTask& T = tasks[active[a]];
                    T.voff = tot;
                    tot += int64_t(T.n) * T.kcap;
                    const int k = hstate[active[a]].k;
                    if (pass > 0 && k > 0) {
                        segs.push_back(Seg{old_u[a], T.uoff, int64_t(k) * T.m});
                        segs.push_back(Seg{old_v[a], T.voff, int64_t(k) * T.n});
                    }
                    S.slot_elems += int64_t(T.m + T.n) * T.kcap;
                }
                double* npool = nullptr;
                HIPCHECK(hipMalloc(&npool, std::max<int64_t>(tot, 1) * sizeof(double)));
                owned.push_back(npool);
                Seg* dsegs = nullptr;
                if (!segs.empty()) {
                    dsegs = upload(segs);
                    owned.push_back(dsegs);
                    hipLaunchKernelGGL(k_copy_segs, dim3(segs.size()), dim3(256), 0, nullptr,
                                       dsegs, pool, npool);
                    HIPCHECK(hipGetLastError());
                }
                std::vector<AcaTask> launch(active.size());
                for (size_t a = 0; a < active.size(); a++) launch[a] = tasks[active[a]];
                AcaTask* dt = upload(launch);
                owned.push_back(dt);
                HIPCHECK(hipEventRecord(e0, nullptr));
                hipLaunchKernelGGL(k_aca, dim3(launch.size()), dim3(kAcaThreads), 0, nullptr, dt,
                                   dstate, dxt, dxs, dct, dcs, npool, npool, work, flags, kid,
                                   eps);
                HIPCHECK(hipGetLastError());
                HIPCHECK(hipEventRecord(e1, nullptr));
                HIPCHECK(hipEventSynchronize(e1));
                float ms = 0;
                HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
                S.kernel_ms += ms;
                S.launches++;
                HIPCHECK(hipMemcpy(hstate.data(), dstate, nc * sizeof(AcaState),
                                   hipMemcpyDeviceToHost));
                release(dt);
                release(dsegs);
                release(pool);
                pool = npool;
                std::vector<int64_t> finished, cont;
                for (int64_t t : active) (hstate[t].done ? finished : cont).push_back(t);
                if (pass == 0) S.unconverged_first += static_cast<int64_t>(cont.size());

                for (int64_t t : finished) {
                    const AcaTask& T = tasks[t];
                    const int64_t k = hstate[t].k;
                    if (collect) {
                        seen_ids.push_back(order[pos + T.sid]);
                        seen_ranks.push_back(static_cast<int32_t>(k));
                    }
                    S.used_elems += int64_t(T.m + T.n) * k;
                }
                if (svd_eps >= 0.0)
                    emit_recompressed(finished, tasks, hstate, pool, order, pos);
                else
                    emit_raw(finished, tasks, hstate, pool, order, pos);
                done_blocks += static_cast<int64_t>(finished.size());
                for (int64_t t : cont) {
                    AcaTask& T = tasks[t];
                    T.kcap = static_cast<int32_t>(round_cap(2 * int64_t(T.kcap), T.kmax));
                }
                active.swap(cont);
                pass++;
                if (verbose)
                    std::fprintf(stderr, "[hmx] GPU ACA+ chunk %lld pass %d: %lld of %lld blocks done, "
                                         "%.1f ms ACA+ kernels, %.1f ms recompression, %.2f s wall\n",
                                 static_cast<long long>(S.chunks), pass,
                                 static_cast<long long>(done_blocks), static_cast<long long>(nb),
                                 S.kernel_ms, S.recompress_ms, wall());
            }
            S.passes = std::max<int64_t>(S.passes, pass);
            for (void* p : owned)
                if (p != dxt && p != dxs && p != dct && p != dcs) (void)hipFree(p);
            owned.assign({dxt, dxs});
            if (dct) owned.push_back(dct);
            if (dcs) owned.push_back(dcs);
            S.chunks++;
            pos = end;
        }
        };
        if (!probe.empty() && refine) {
            // probe blocks first; their ACA+ ranks then refine the capacities of
            // the others before those run
            std::vector<char> in_probe(static_cast<size_t>(nb), 0);
            std::vector<int64_t> first;
            for (int64_t b : probe)
                if (b >= 0 && b < nb && !in_probe[b]) {
                    in_probe[b] = 1;
                    first.push_back(b);
                }
            by_cost(first);
            run_list(first, true);
            S.probe_blocks = static_cast<int64_t>(first.size());
            refine(seen_ids, seen_ranks, caps);
            std::vector<int64_t> rest;
            for (int64_t b = 0; b < nb; b++)
                if (!in_probe[b]) rest.push_back(b);
            by_cost(rest);
            run_list(rest, false);
        } else {
            std::vector<int64_t> all(nb);
            for (int64_t b = 0; b < nb; b++) all[b] = b;
            by_cost(all);
            run_list(all, false);
        }
        wait_jobs();
        S.blocks = nb;
    } catch (...) {
        (void)hipDeviceSynchronize();
        free_staging();
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        free_all();
        throw;
    }
    free_staging();
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    free_all();
    S.wall_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - wall0).count();
    if (stats) *stats = S;
}

}  // namespace hmx
