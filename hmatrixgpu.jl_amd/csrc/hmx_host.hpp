// hmx_host.hpp -- internal host-side structures of libhmx (not part of the ABI).
//
// Host code follows Julia 1.10 Float64 semantics wherever the reference's
// results must be reproduced bit for bit (cluster tree, block tree, ACA+); the
// whole host side is compiled with -ffp-contract=off.
#pragma once

#include <atomic>
#include <cstdint>
#include <functional>
#include <memory>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/hmx.h"

namespace hmx {

// Error carrying an hmx_status code; converted to a return code + thread-local
// message at the C boundary.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

// ---- cluster tree (tree.jl:6-20) ------------------------------------------
struct BuildOptions;

struct ClusterNode {
    int64_t start;  // 1-based
    int64_t end;    // 1-based, exclusive
    double center[3];
    double radius;
    int64_t left, right;  // node ids, -1 for none
    bool leaf;
};

struct ClusterTree {
    int64_t npts = 0, dims = 1;
    std::vector<int64_t> index_map;  // 1-based, length npts*dims
    std::vector<ClusterNode> nodes;  // pre-order; node 0 is the root
    std::vector<int64_t> leaves;     // leaf node ids in increasing start order
};

std::unique_ptr<ClusterTree> build_cluster_tree(const double* xyz, int64_t npts, int64_t leaf,
                                                int64_t dims);
void tree_info(const ClusterTree& t, int64_t* depth, int64_t* pmax, int64_t* pmin);

// Julia LinearAlgebra.generic_norm2 for a 3-vector.
double norm3(const double v[3]);

// ---- block tree (block.jl:2-16) --------------------------------------------
struct BlockNode {
    int64_t t, s;        // cluster node ids
    int64_t left, right; // block node ids, -1 for none
    bool adm, dense;
};

struct BlockTree {
    const ClusterTree* T = nullptr;
    const ClusterTree* S = nullptr;
    std::vector<BlockNode> nodes;  // node 0 is the root
};

std::unique_ptr<BlockTree> build_block_tree(const ClusterTree& T, const ClusterTree& S, double eta);
// merge_dense_matrices! (block.jl:98-112) on the subtree rooted at node `root`
void merge_dense(BlockTree& b, int64_t root = 0);
// DFS pre-order lists of (target node, source node)
void traverse(const BlockTree& b, std::vector<std::pair<int64_t, int64_t>>* direct,
              std::vector<std::pair<int64_t, int64_t>>* approx);

// ---- entries -----------------------------------------------------------------
// Evaluates K[rows, cols] (0-based original indices) into a column-major buffer.
struct EntrySource {
    int32_t kernel_id = 0;
    const double* xt = nullptr;  // 3 x Nt
    const double* xs = nullptr;  // 3 x Ns
    hmx_block_fn fill = nullptr;
    void* ctx = nullptr;
    // scalar entry for built-in kernels
    double entry(int64_t i, int64_t j) const;
    // K[rows[0..nr), cols[0..nc)] -> out (column-major, nr x nc)
    void block(const int64_t* rows, int64_t nr, const int64_t* cols, int64_t nc, double* out) const;
    bool thread_safe() const { return kernel_id != HMX_KERNEL_CALLBACK; }
};

// ---- low rank (aca.jl) ----------------------------------------------------------
struct LowRank {
    int64_t m = 0, n = 0, k = 0;
    std::vector<double> U;  // m x k column-major
    std::vector<double> V;  // k x n column-major
};

// Row/column oracles for ACA+: fill residual-free matrix row I (n values) or
// column J (m values); 0-based local indices.
using RowFn = std::function<void(int64_t, double*)>;
LowRank aca_plus(int64_t m, int64_t n, const RowFn& row, const RowFn& col, double eps,
                 int64_t max_iter);
LowRank svd_recompress(const LowRank& in, double eps);
// Fixed-order sum of squares used by the ACA+ stop test (host and device).
constexpr int kSumLanes = 256;
double sumsq_lanes(const double* x, int64_t n);
// Dot product in the fixed 64-lane order of the QR reflectors (host and device).
double dot_lanes64(const double* x, const double* y, int64_t n);

// ---- H-matrix -----------------------------------------------------------------
// Allocator whose construct() without arguments default-initialises: resizing a
// vector of doubles then leaves the new elements unset instead of writing zeros.
// The H-matrix payloads (tens of GB) are always written in full afterwards, by
// several threads, so a single-threaded zero fill first would only cost time.
template <typename T>
struct DefaultInitAlloc : std::allocator<T> {
    template <typename U>
    struct rebind {
        using other = DefaultInitAlloc<U>;
    };
    DefaultInitAlloc() = default;
    template <typename U>
    DefaultInitAlloc(const DefaultInitAlloc<U>&) noexcept {}
    template <typename U>
    void construct(U* p) noexcept(std::is_nothrow_default_constructible<U>::value) {
        ::new (static_cast<void*>(p)) U;
    }
    template <typename U, typename... Args>
    void construct(U* p, Args&&... args) {
        ::new (static_cast<void*>(p)) U(std::forward<Args>(args)...);
    }
};
using Payload = std::vector<double, DefaultInitAlloc<double>>;
// Ask for transparent huge pages on a large, not yet touched buffer (its first
// writes then fault 2 MiB pages instead of 4 KiB ones); a no-op where the
// kernel does not honour the advice.
void advise_huge_pages(void* p, size_t bytes);

struct DenseBlock {
    int64_t r0, r1, c0, c1;  // 1-based inclusive (hmatrix.jl:185)
    int64_t off;             // 0-based offset in the flattened dense payload
};
struct LowRankBlock {
    int64_t r0, r1, c0, c1;  // 1-based inclusive
    int64_t k;
    int64_t uoff, voff;      // 0-based offsets in U_data / V_data
    int64_t vx0;             // 0-based first row in Vx_buffer
    int64_t snode;           // source cluster node id (groups the V*X work)
};

struct DeviceOp;  // device-resident operator for one storage precision
void device_destroy(DeviceOp* op);
struct DeviceOpDeleter {
    void operator()(DeviceOp* op) const { device_destroy(op); }
};

struct HMatrix {
    int64_t m = 0, n = 0;
    std::vector<int64_t> tmap, smap;  // 1-based
    std::vector<DenseBlock> dense;    // direct list, then storage fallbacks
    std::vector<LowRankBlock> lowrank;
    Payload U, V;                     // flattened row-major payloads (FP64)
    Payload D;                        // flattened dense payload; filled only for
                                      // callback kernels or on export
    bool D_ready = false;
    int64_t R = 0, dlen = 0;
    EntrySource src;
    std::vector<double> xt_copy, xs_copy;  // owned copies of the coordinates
    std::vector<int64_t> target_leaf_start;  // 0-based start rows of target leaves (+ end)
    double build_seconds = 0.0;
    int32_t device = 0;
    int64_t target_dims = 1, source_dims = 1;
    std::unique_ptr<DeviceOp, DeviceOpDeleter> dev[3];
    // per admissible block, approx-list order (hmatrix.jl:189-213)
    struct ApproxStat {
        float feat[9];     // rank-predictor inputs (block_features, host_hmatrix.cpp)
        int32_t aca_rank;  // ACA+ terms before recompression
        int32_t rank;      // rank after recompression
        int32_t cap;       // first rank capacity of the device ACA+ (0: host ACA+)
    };
    std::vector<ApproxStat> approx_stats;
    // batches (batch.hip) holding pointers to this H-matrix's device operators;
    // while non-zero the operators may not be released, rebuilt or destroyed
    std::atomic<int> batch_refs{0};
    void ensure_dense_payload();
};

std::unique_ptr<HMatrix> build_hmatrix(const ClusterTree& T, const ClusterTree& S,
                                       const EntrySource& src, double eta, double eps,
                                       bool svd, int nthreads,
                                       const BuildOptions* opt = nullptr);

// On-disk H-matrix (host_io.cpp).  save() writes the dense payload when it is
// present or with_dense is set (it is always present for callback kernels);
// load() validates the file and returns a host operator with no device storage.
void save_hmatrix(HMatrix& h, const char* path, bool with_dense);
std::unique_ptr<HMatrix> load_hmatrix(const char* path);
// Digests of the index maps, the block tables (list order), the U payload and
// the V payload: equal digests <=> equal layouts (up to hash collisions).
void layout_checksums(const HMatrix& h, uint64_t out[4]);

// sparsify_hmatrix (hmatrix.jl:234-274): the merged dense blocks as CSR,
// original index spaces, 0-based, columns sorted within each row.
struct CsrMatrix {
    int64_t m = 0, n = 0;
    std::vector<int64_t> rowptr, col;
    std::vector<double> val;
};
CsrMatrix sparsify(const ClusterTree& T, const ClusterTree& S, const EntrySource& src, double eta,
                   int nthreads);

// Simple fixed-size worker pool: run f(i) for i in [0,n) on `threads` threads.
void parallel_for(int64_t n, int threads, const std::function<void(int64_t)>& f);
int default_threads();

// ---- device side (device.hip) -------------------------------------------------
void device_build(HMatrix& h, int storage);
void device_matvec(HMatrix& h, int storage, const void* X, int64_t ldx, void* Y, int64_t ldy,
                   int nrhs, int io_dtype, void* stream);
// The same product with its scratch in a static device array of
// kNoAllocScratchBytes per GPU: no device allocation, shared by every call on
// that GPU (calls that overlap on one GPU race).
constexpr size_t kNoAllocScratchBytes = size_t(128) << 20;
void device_matvec_noalloc(HMatrix& h, int storage, const void* X, int64_t ldx, void* Y,
                           int64_t ldy, int nrhs, int io_dtype, void* stream);
// mul!/`*` on host FP64 arrays (the reference's HMatrixCPU product): stages x
// to the device, runs the FP64 GPU product (materialising the FP64 operator on
// h.device on first use) and copies y back; synchronous.
void device_matvec_host(HMatrix& h, const double* x, int64_t ldx, double* y, int64_t ldy,
                        int nrhs);
// Free the per-stream scratch of `stream` (or of every stream) of every storage
// precision after synchronising those streams; returns the allocations freed.
int64_t device_release_scratch(HMatrix& h, void* stream, bool all_streams);
// bytes of product scratch held and (operator, stream) entries holding it
void device_scratch_usage(const HMatrix& h, int64_t* bytes, int64_t* entries);
int64_t device_panel_bytes(const DeviceOp* op);
int64_t device_index_bytes(const DeviceOp* op);
void device_profile_enable(HMatrix& h, bool on);
void device_profile_read(HMatrix& h, double* ms, int64_t* launches, bool reset);

// ---- batched ACA+ on the device (aca_gpu.hip) ------------------------------------
struct AcaBlock {
    int64_t t0, s0;  // 0-based first row / column in the permuted index spaces
    int64_t m, n;
};
struct AcaStats {
    int64_t blocks = 0;
    int64_t chunks = 0;             // memory-bounded groups of blocks
    int64_t passes = 0;             // most capacity passes any chunk needed
    int64_t launches = 0;           // ACA+ kernel launches
    int64_t unconverged_first = 0;  // blocks that outgrew their first capacity
    int64_t probe_blocks = 0;       // blocks run before the capacities were refined
    int64_t slot_elems = 0;         // sum over passes of (m + n) * capacity
    int64_t used_elems = 0;         // sum of (m + n) * final rank
    double kernel_ms = 0.0;         // ACA+ kernel time (HIP events)
    double recompress_ms = 0.0;     // device recompression time (HIP events)
    double wall_s = 0.0;            // whole phase including copies and callbacks
};
// ACA+ (eps is the ACA tolerance) of every block with the given initial rank
// capacities; on_done(b, factors) is called from host worker threads as blocks
// finish.  Built-in scalar kernels only.
// Optional probe phase: the blocks listed in `probe` run first, then
// refine(ids, aca_ranks, caps) may rewrite the capacities of the other blocks.
using AcaRefine = std::function<void(const std::vector<int64_t>&, const std::vector<int32_t>&,
                                     std::vector<int32_t>&)>;
// svd_eps < 0: on_done(block, aca_rank, factors) receives the ACA+ terms of every
// block.  svd_eps >= 0: on_slab receives their device recompression at svd_eps
// (bit-identical to svd_recompress) instead.
using AcaDone = std::function<void(int64_t, int64_t, LowRank&&)>;
// Recompressed factors of many blocks in one buffer: per part U (m x k column-major)
// at off, then V (k x n, row-major).  One buffer of up to kSlabBytes instead of two
// vectors per block: its pages are faulted 2 MiB at a time (the factors of N = 32,768,
// 2.5 GB, took 0.36 s to place into fresh per-block vectors).
struct FactorSlab {
    struct Part {
        int64_t block, aca_k, m, n, k, off;
    };
    Payload data;
    std::vector<Part> parts;
};
constexpr int64_t kSlabBytes = int64_t(16) << 20;
using AcaSlabDone = std::function<void(std::unique_ptr<FactorSlab>)>;
void gpu_aca(const HMatrix& h, const std::vector<AcaBlock>& blocks, std::vector<int32_t> caps,
             double eps, double svd_eps, int nthreads, AcaStats* stats, const AcaDone& on_done,
             const AcaSlabDone& on_slab, const std::vector<int64_t>& probe = {}, const AcaRefine& refine = nullptr);
// capacity rounding of a pass (multiple of 4, at least 4, at most kmax)
int64_t aca_round_cap(int64_t c, int64_t kmax);

// ---- rank predictor (rankpred.hip) ----------------------------------------------
// 6 -> 64 -> 64 -> 1 MLP on (log diam_s, log diam_t, log dist, log n_s, log n_t,
// log tol) -> z = log(1 + ACA+ rank).  Rows of X are samples (6 floats).
struct RankPredictor;
RankPredictor* rankpred_create(int hidden, uint64_t seed, int device);
void rankpred_destroy(RankPredictor* p);
RankPredictor* rankpred_clone(const RankPredictor& p);
int64_t rankpred_nparams();
void rankpred_train(RankPredictor& p, const float* X, const float* Z, int64_t n, int epochs,
                    int batch, float lr, uint64_t seed, float* loss_hist);
void rankpred_grad(RankPredictor& p, const float* X, const float* Z, int64_t n, float* grad,
                   float* loss);
void rankpred_predict(const RankPredictor& p, const float* X, int64_t n, float* z_out);
void rankpred_params(RankPredictor& p, float* master, float* bf16, float* norm, bool get);
constexpr int kRankFeatures = HMX_RANK_FEATURES;

// ---- staging array of the device product ------------------------------------------
// Element sizes of a storage precision, and of its staging rows for a pass of
// W right-hand sides (BF16 keeps X and T in BF16 only on the 16-wide MFMA path).
inline size_t elem_size(int storage) { return storage == HMX_F64 ? 8 : storage == HMX_F32 ? 4 : 2; }
inline int tk_of(int storage) { return static_cast<int>(64 / elem_size(storage)); }
inline size_t s_elem(int storage, int W) {
    return storage == HMX_F64 ? 8 : (W >= 16 && storage == HMX_BF16 ? 2 : 4);
}
// The staging array S of one pass: rows n + R + 1 + TK (X permuted, T = V X,
// a zero row, one k-tile of padding rows), each W elements.  Rows are 32-bit
// indices (bounded by 2^31); an array below 4 GiB is read through 32-bit buffer
// offsets, a larger one through 64-bit global loads.  [zero_begin, zero_end) is
// the 16-byte-aligned byte range that must read zero (the zero row and the
// padding rows).
struct StagingLayout {
    int64_t rows = 0, row_bytes = 0, bytes = 0, zero_begin = 0, zero_end = 0;
};
inline StagingLayout staging_layout(int64_t n, int64_t R, int storage, int W) {
    if (n < 0 || R < 0 || (storage != HMX_F64 && storage != HMX_F32 && storage != HMX_BF16) ||
        (W != 1 && W != 4 && W != 16 && W != 32 && W != 48))
        throw Error(HMX_ERR_ARG, "staging layout: bad argument");
    StagingLayout L;
    L.rows = n + R + 1 + tk_of(storage);
    if (L.rows >= (int64_t(1) << 31))
        throw Error(HMX_ERR_UNSUPPORTED,
                    "source/T staging array has 2^31 rows or more (32-bit row index)");
    L.row_bytes = static_cast<int64_t>(W * s_elem(storage, W));
    L.bytes = L.rows * L.row_bytes;
    L.zero_begin = ((n + R) * L.row_bytes) & ~int64_t(15);
    L.zero_end = (L.bytes + 15) & ~int64_t(15);
    return L;
}

// Options of the H-matrix build beyond the reference's keywords.
struct BuildOptions {
    int aca_device = 0;                       // 0 host threads, 1 batched ACA+ on the GPU
    int device = 0;                           // GPU ordinal of the device ACA+
    int initial_rank = 16;                    // first capacity without a predictor
    const RankPredictor* predictor = nullptr;  // capacity from the predicted rank
    double cap_margin = 0.25;                 // capacity = (1 + margin) * predicted rank
    int refine_samples = 0;                   // probe blocks that fine-tune a copy of the
    int refine_epochs = 200;                  // predictor on this build's own ACA+ ranks
    AcaStats* stats = nullptr;
};

// Thread-local message returned by hmx_last_error().
void set_last_error(const char* msg);

}  // namespace hmx

// Opaque ABI handle of a rank predictor (include/hmx.h).
struct hmx_rankpred {
    struct Del {
        void operator()(hmx::RankPredictor* p) const { hmx::rankpred_destroy(p); }
    };
    std::unique_ptr<hmx::RankPredictor, Del> p;
};

// Opaque ABI handle of an H-matrix (include/hmx.h).
struct hmx_hmatrix {
    std::unique_ptr<hmx::HMatrix> h;
};
