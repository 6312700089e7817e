// device_op.hpp -- host-side state of a device-resident H-matrix operator and
// the stage launcher shared by the single and batched products.
#pragma once

#include "kernels.hpp"

namespace hmx {

// Scratch of one pass width: three arrays in one allocation, which S is the start of.
struct ScratchW {
    void* S = nullptr;  // (s0 + n + R + 1 + TK) x W source rows (staging_layout)
    void* P = nullptr;   // far-field partial rows x W
    void* LP = nullptr;  // leaf-result rows x W
};

struct Scratch {
    ScratchW w[5];  // W = 1, 4, 16, 32, 48
    uint64_t last_use = 0;  // DeviceOp::use_clock at the stream's last product
    size_t bytes = 0;       // bytes held by the arrays of every width
    int refused = 1 << 30;  // narrowest wide pass that was refused its scratch
};

constexpr int kMaxWidth = 48;  // widest pass
inline int w_slot(int W) { return W == 1 ? 0 : W == 4 ? 1 : 1 + W / 16; }

struct DeviceOp {
    int storage = 0, device = 0;
    int64_t m = 0, n = 0, R = 0;
    int64_t s0 = 0;  // unused S rows before X (HMX_STAGING_ROW_OFFSET)
    void* panel = nullptr;
    int64_t panel_elems = 0;
    PairItem* itemsB = nullptr;
    int64_t nB = 0;
    int32_t* colidx = nullptr;
    int64_t ncol = 0;
    FarItem* itemsA = nullptr;
    int64_t nA = 0;
    ReduceGroup* groups = nullptr;
    int64_t nG = 0;
    int64_t npartial = 0;
    int64_t nlrows = 0;         // leaf-result rows of one pass
    RowSrc* rowsrc = nullptr;   // per original target row
    bool direct = false;        // the leaf kernel writes Y (no item is cut, few rows)
    int32_t* tmap0 = nullptr;
    int32_t* inv_smap = nullptr;
    int32_t* smap0 = nullptr;   // small operators only (xdir): permuted source -> original row
    int32_t* colx = nullptr;    // and the leaf columns with X by original row
    // host copies of the work lists (the batched operator re-packs them)
    std::vector<PairItem> hItemsB;
    std::vector<FarItem> hItemsA;
    std::vector<ReduceGroup> hGroups;
    std::mutex mu;
    std::map<void*, Scratch> scratch;
    uint64_t use_clock = 0;
    bool profiling = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev[4];
    double ms[4] = {0, 0, 0, 0};
    int64_t launches[4] = {0, 0, 0, 0};
};

inline StagingLayout staging(const DeviceOp& op, int W) {
    return staging_layout(op.s0 + op.n, op.R, op.storage, W);
}
// Clear rows n + R .. end of S on `st`: the zero row and the padding rows must
// read 0, every other row is written before it is read.  A row is W * s_elem
// bytes, a multiple of 16 for W >= 4 (W = 1: cleared from the 16-byte word that
// holds row n + R, before X and T are written).
inline void zero_staging_tail(void* S, const StagingLayout& lay, hipStream_t st) {
    const int64_t n16 = (lay.zero_end - lay.zero_begin) / 16;
    hipLaunchKernelGGL(k_zero16, dim3(static_cast<unsigned>((n16 + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<uint4*>(static_cast<char*>(S) + lay.zero_begin), n16);
    HIPCHECK(hipGetLastError());
}
// element size of the partial sums
inline size_t p_elem(int storage) { return storage == HMX_F64 ? 8 : 4; }

template <typename T, typename A>
T* upload(const std::vector<T, A>& v) {
    T* d = nullptr;
    if (v.empty()) return nullptr;
    HIPCHECK(hipMalloc(&d, v.size() * sizeof(T)));
    HIPCHECK(hipMemcpy(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return d;
}

struct DeviceGuard {
    int prev = 0;
    explicit DeviceGuard(int dev) {
        HIPCHECK(hipGetDevice(&prev));
        if (prev != dev) HIPCHECK(hipSetDevice(dev));
    }
    ~DeviceGuard() { (void)hipSetDevice(prev); }
};

// Clear the zero and padding rows of new scratch, so that whatever runs next on `st`
// reads zeros.  On that stream itself: a clear on the null stream is not ordered before
// the work of a stream created without that dependence, and would overwrite rows that the
// first product has already written.  While `st` is being captured (a relaxed capture may
// allocate) the launch would only be recorded, and a product that runs before the graph
// does would read uncleared rows; the clear then runs at once on a stream of its own.
inline void clear_new_staging(void* S, const StagingLayout& lay, hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) {
        zero_staging_tail(S, lay, st);
        return;
    }
    (void)hipGetLastError();
    hipStream_t own = nullptr;
    HIPCHECK(hipStreamCreateWithFlags(&own, hipStreamNonBlocking));
    try {
        zero_staging_tail(S, lay, own);
        HIPCHECK(hipStreamSynchronize(own));
    } catch (...) {
        (void)hipStreamDestroy(own);
        throw;
    }
    HIPCHECK(hipStreamDestroy(own));
}

// Byte sizes of the three arrays of one pass width, each a multiple of 256.
struct ScratchSizes {
    size_t s, p, lp;
    size_t total() const { return s + p + lp; }
};
inline ScratchSizes scratch_sizes(const DeviceOp& op, int W) {
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t pe = p_elem(op.storage);
    return {up(static_cast<size_t>(staging(op, W).zero_end)),
            up(static_cast<size_t>(std::max<int64_t>(op.npartial, 1)) * W * pe),
            up(static_cast<size_t>(std::max<int64_t>(op.nlrows, 1)) * W * pe)};
}

// Allocate the scratch of one pass width, with its zero rows cleared before anything
// else on `st`.  Returns the status of the allocation; every other failure throws, and `s`
// is set only when all has succeeded.
inline hipError_t alloc_scratch(const DeviceOp& op, int W, hipStream_t st, ScratchW& s) {
    const ScratchSizes z = scratch_sizes(op, W);
    ScratchW n;
    const hipError_t e = hipMalloc(&n.S, z.total());
    if (e != hipSuccess) return e;
    try {
        clear_new_staging(n.S, staging(op, W), st);
    } catch (...) {
        (void)hipFree(n.S);
        throw;
    }
    n.P = static_cast<char*>(n.S) + z.s;
    n.LP = static_cast<char*>(n.P) + z.p;
    s = n;
    return hipSuccess;
}

// Work lists of one launch (one H-matrix, or a batch of them).
struct StageArrays {
    const FarItem* itemsA = nullptr;
    int64_t nA = 0;
    const ReduceGroup* groups = nullptr;
    int64_t nG = 0;
    const PairItem* itemsB = nullptr;
    int64_t nB = 0;
    int64_t gather_n = 0;   // largest source size over the instances
    int gather_insts = 1;   // instances (grid.y of the gather and the finish)
    int64_t out_m = 0;      // largest target size over the instances that need k_finish
    bool wide = false;      // an instance's S has 4 GiB or more: 64-bit S loads
    bool xdir = false;      // X is read in place (one right-hand side): no gather
};
// S of 4 GiB or more: beyond the reach of 32-bit buffer offsets
inline bool wide_staging(const StagingLayout& L) { return L.bytes >= (int64_t(1) << 32); }

// HIP-event timing of one stage on the launch stream (only when profiling).
struct StageTimer {
    DeviceOp* op;
    hipStream_t st;
    int stage;
    hipEvent_t a = nullptr, b = nullptr;
    StageTimer(DeviceOp* o, hipStream_t s, int k) : op(o), st(s), stage(k) {
        if (!op || !op->profiling) return;
        HIPCHECK(hipEventCreate(&a));
        HIPCHECK(hipEventCreate(&b));
        HIPCHECK(hipEventRecord(a, st));
    }
    ~StageTimer() {
        if (!op || !op->profiling || !a) return;
        (void)hipEventRecord(b, st);
        std::lock_guard<std::mutex> g(op->mu);
        op->ev[stage].push_back({a, b});
    }
};

// The stages of a product pass: gather X -> S, far-field panels (V*X),
// partial reduce, leaf panels -> leaf-result rows, and their piece sums into Y
// (k_finish, timed with the far-field partial reduce as stage 2, so that
// stage 3 is the leaf kernel alone).
template <typename TS, int W, typename TIO, bool BATCH>
void launch_stages(const StageArrays& A, const InstDesc& one, const InstDesc* insts,
                   hipStream_t st, DeviceOp* prof) {
    if constexpr (W == 1 && !BATCH && std::is_same<TIO, typename Store<TS>::acc>::value) {
        if (A.xdir) {
            if (A.nA) {
                StageTimer t(prof, st, 1);
                hipLaunchKernelGGL((k_far<TS, 1, kPanelPolicy, false, false, true>), dim3(A.nA),
                                   dim3(kWaves * 64), 0, st, A.itemsA, one, insts);
            }
        }
    }
    if (!A.xdir) {
        StageTimer t(prof, st, 0);
        hipLaunchKernelGGL((k_gather<TS, W, TIO, BATCH>),
                           dim3(static_cast<unsigned>((A.gather_n + 255) / 256), A.gather_insts),
                           dim3(256), 0, st, one, insts);
    }
    if (A.nA && !A.xdir) {
        StageTimer t(prof, st, 1);
        if (A.wide)
            hipLaunchKernelGGL((k_far<TS, W, kPanelPolicy, BATCH, true>), dim3(A.nA),
                               dim3(kWaves * 64), 0, st, A.itemsA, one, insts);
        else
            hipLaunchKernelGGL((k_far<TS, W, kPanelPolicy, BATCH, false>), dim3(A.nA),
                               dim3(kWaves * 64), 0, st, A.itemsA, one, insts);
    }
    if (A.nG) {
        StageTimer t(prof, st, 2);
        hipLaunchKernelGGL((k_reduce<TS, W, BATCH>), dim3(A.nG), dim3(256), 0, st, A.groups, one,
                           insts);
    }
    if constexpr (W == 1 && !BATCH && std::is_same<TIO, typename Store<TS>::acc>::value) {
        if (A.nB && A.xdir) {
            StageTimer t(prof, st, 3);
            hipLaunchKernelGGL((k_leaf<TS, 1, kPanelPolicy, false, false, true>), dim3(A.nB),
                               dim3(kWaves * 64), 0, st, A.itemsB, one, insts);
        }
    }
    if (A.nB && !A.xdir) {
        StageTimer t(prof, st, 3);
        if (A.wide)
            hipLaunchKernelGGL((k_leaf<TS, W, kPanelPolicy, BATCH, true>), dim3(A.nB),
                               dim3(kWaves * 64), 0, st, A.itemsB, one, insts);
        else
            hipLaunchKernelGGL((k_leaf<TS, W, kPanelPolicy, BATCH, false>), dim3(A.nB),
                               dim3(kWaves * 64), 0, st, A.itemsB, one, insts);
    }
    if (A.out_m) {
        StageTimer t(prof, st, 2);
        constexpr int rows = kFinRows<W>;
        hipLaunchKernelGGL((k_finish<TS, W, TIO, BATCH>),
                           dim3(static_cast<unsigned>((A.out_m + rows - 1) / rows), A.gather_insts, kSlices<W>),
                           dim3(256), 0, st, one, insts);
    }
}

// Dispatch order of leaf work items (see device.hip).
void order_leaf_items(std::vector<PairItem>& items, const char* order);

}  // namespace hmx
