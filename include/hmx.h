/*
 * hmx.h -- C ABI of the MI355X (gfx950) H-matrix engine (libhmx.so).
 *
 * Every entry point mirrors a HMatrixGPU.jl v0.1.0 interface (cited per
 * function) so that the Julia package (ccall), the Python mirror (ctypes) and
 * C/C++ callers bind the same symbols.  Conventions:
 *   - every function returns an int status, 0 == HMX_OK; on failure
 *     hmx_last_error() returns a thread-local message;
 *   - indices crossing the ABI are int64 and 1-based wherever the reference
 *     stores them 1-based (index maps, node ranges, block tables);
 *   - point coordinates are a 3 x N column-major double array (the Julia
 *     Matrix{Float64} the reference takes);
 *   - device pointers are plain addresses on the current HIP device; streams
 *     are hipStream_t passed as void*.
 */
#ifndef HMX_H
#define HMX_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- status, types ------------------------------------------------------ */
enum hmx_status {
    HMX_OK = 0,
    HMX_ERR_ARG = 1,           /* bad argument (NULL handle, size mismatch, ...)   */
    HMX_ERR_DIMS = 2,          /* dims <= 0, tree.jl:46-48                         */
    HMX_ERR_EMPTY_CLUSTER = 3, /* a split left an empty cluster (the reference
                                  throws reducing over an empty point set)        */
    HMX_ERR_NOMEM = 4,
    HMX_ERR_HIP = 5,           /* HIP runtime error / no device                    */
    HMX_ERR_CALLBACK = 6,      /* user entry callback returned non-zero            */
    HMX_ERR_STATE = 7,         /* object not in the required state                 */
    HMX_ERR_UNSUPPORTED = 8
};

enum hmx_dtype { HMX_F64 = 0, HMX_F32 = 1, HMX_BF16 = 2 };

/* Built-in kernels evaluated natively on host and device.                     */
enum hmx_kernel_id {
    HMX_KERNEL_CALLBACK = 0, /* entries come from an hmx_block_fn               */
    HMX_KERNEL_LAPLACE = 1,  /* 1/|x-y|; 0 where points coincide (the diagonal)  */
    HMX_KERNEL_LOG2D = 2,    /* -log(d)/(2*pi); 1.0 where d < 1e-12              */
    HMX_KERNEL_DIPOLE = 3    /* dipolar (demagnetisation) tensor, dims = 3 on both
                                trees: entry (3p+a, 3q+b) = N_ab(x_p - y_q),
                                N = -(3 r r^T - |r|^2 I) / (4 pi |r|^5), 0 at r = 0
                                (examples/hmatrix_vector.jl:12-51)               */
};

typedef struct hmx_tree hmx_tree;
typedef struct hmx_blocktree hmx_blocktree;
typedef struct hmx_lowrank hmx_lowrank;
typedef struct hmx_hmatrix hmx_hmatrix;

/* Matrix entries for HMX_KERNEL_CALLBACK: fill out[i + j*nrows] = K[rows[i], cols[j]]
 * (1-based original indices, column-major), i.e. Julia's K[rows, cols]
 * getindex contract used at hmatrix.jl:183,195-196,209.  Return 0 on success. */
typedef int (*hmx_block_fn)(void* ctx, const int64_t* rows, int64_t nrows, const int64_t* cols,
                            int64_t ncols, double* out);

/* One row (or column) of the matrix given to ACA_plus: out has n_cols (n_rows)
 * entries; index is 1-based.  Mirrors calc_rows / calc_cols, aca.jl:36. */
typedef int (*hmx_vec_fn)(void* ctx, int64_t index, double* out);

const char* hmx_last_error(void);
int hmx_version(int32_t* major, int32_t* minor, int32_t* patch);

/* ---- cluster tree: replaces ClusterTree(...) (tree.jl:45-67, build_tree_node
 *      tree.jl:70-116, update_tree_indices! tree.jl:123-137) ------------------ */
int hmx_tree_build(const double* xyz, int64_t npoints, int32_t max_points_per_leaf, int32_t dims,
                   hmx_tree** out);
/* number of index_map entries (npoints*dims) and of nodes (pre-order) */
int hmx_tree_sizes(const hmx_tree* t, int64_t* nindex, int64_t* nnodes);
/* ClusterTree fields (tree.jl:6-20): index_map (1-based), per node start_idx,
 * end_idx (exclusive), center (3 per node), radius, left/right child node ids
 * (-1 = none), is_leaf.  Any output pointer may be NULL. */
int hmx_tree_export(const hmx_tree* t, int64_t* index_map, int64_t* start_idx, int64_t* end_idx,
                    double* center, double* radius, int64_t* left, int64_t* right,
                    int8_t* is_leaf);
/* info(::ClusterTree), tree.jl:153-187 */
int hmx_tree_info(const hmx_tree* t, int64_t* depth, int64_t* max_points, int64_t* min_points);
int hmx_tree_destroy(hmx_tree* t);

/* ---- block tree: replaces BlockTree(X, Y; eta) (block.jl:31-44,58-90),
 *      merge_dense_matrices! (block.jl:98-112) and traverse (block.jl:127-155) - */
int hmx_blocktree_build(const hmx_tree* target, const hmx_tree* source, double eta,
                        hmx_blocktree** out);
int hmx_blocktree_merge_dense(hmx_blocktree* b);
/* merge_dense_matrices!(node::BlockTreeNode) (block.jl:98-112) on the subtree
 * rooted at block node `node` (the ids of hmx_blocktree_export, 0 = root):
 * a node with two children becomes dense iff both children are, bottom-up;
 * only is_dense flags change. */
int hmx_blocktree_merge_dense_node(hmx_blocktree* b, int64_t node);
/* nnodes, and the lengths of direct_list / approx_list traverse() returns */
int hmx_blocktree_sizes(const hmx_blocktree* b, int64_t* nnodes, int64_t* ndirect,
                        int64_t* napprox);
/* BlockTreeNode fields (block.jl:2-9): target/source cluster node ids,
 * is_admissible, is_dense, left/right block node ids (-1 = none). */
int hmx_blocktree_export(const hmx_blocktree* b, int64_t* target_node, int64_t* source_node,
                         int8_t* is_admissible, int8_t* is_dense, int64_t* left, int64_t* right);
/* traverse(): (target node, source node) pairs, 2 x n each, DFS order */
int hmx_blocktree_traverse(const hmx_blocktree* b, int64_t* direct, int64_t* approx);
int hmx_blocktree_destroy(hmx_blocktree* b);

/* ---- low-rank compression: replaces ACA_plus (aca.jl:36-106) and
 *      SVD_recompress (aca.jl:123-143) ---------------------------------------- */
/* max_iter <= 0 means the reference default (n_rows). */
int hmx_aca_plus(int64_t n_rows, int64_t n_cols, hmx_vec_fn calc_rows, hmx_vec_fn calc_cols,
                 void* ctx, double eps, int64_t max_iter, hmx_lowrank** out);
int hmx_lowrank_create(int64_t m, int64_t n, int64_t k, const double* U, const double* V,
                       hmx_lowrank** out);
int hmx_lowrank_sizes(const hmx_lowrank* lr, int64_t* m, int64_t* n, int64_t* rank);
/* U: m x k column-major, V: k x n column-major */
int hmx_lowrank_export(const hmx_lowrank* lr, double* U, double* V);
int hmx_svd_recompress(const hmx_lowrank* in, double eps, hmx_lowrank** out);
int hmx_lowrank_destroy(hmx_lowrank* lr);

/* ---- H-matrix: replaces HMatrix(K, X, Y; eta, eps, flatten, ...,
 *      svd_recompress) (hmatrix.jl:72-148, build_matrices hmatrix.jl:170-217) --
 * kernel_id selects a built-in kernel (target_xyz / source_xyz: 3 x N column-
 * major, the same arrays the trees were built from) or HMX_KERNEL_CALLBACK
 * (fill/ctx).  storage_mask: OR of (1 << HMX_F64 | HMX_F32 | HMX_BF16), the
 * storage precisions to materialise on `device` (0 = host-only build; the
 * reference layout can still be exported).  nthreads <= 0: library default.  */
int hmx_hmatrix_build(const hmx_tree* target, const hmx_tree* source, int32_t kernel_id,
                      const double* target_xyz, const double* source_xyz, hmx_block_fn fill,
                      void* ctx, double eta, double eps, int32_t svd_recompress,
                      int32_t storage_mask, int32_t device, int32_t nthreads, hmx_hmatrix** out);
/* ---- sparse near field: sparsify_hmatrix(K, X, Y; eta) (hmatrix.jl:234-274) --
 * Builds the block tree of (target, source) at eta, merges dense blocks
 * (block.jl:98-112) and returns every entry of the dense blocks as a sparse
 * matrix in the ORIGINAL index spaces: CSR, 0-based, columns sorted within a
 * row (the reference returns a SparseMatrixCSC with the same entries).
 * Kernel arguments as for hmx_hmatrix_build; nthreads <= 0: default. */
typedef struct hmx_csr hmx_csr;
int hmx_sparsify(const hmx_tree* target, const hmx_tree* source, int32_t kernel_id,
                 const double* target_xyz, const double* source_xyz, hmx_block_fn fill, void* ctx,
                 double eta, int32_t nthreads, hmx_csr** out);
int hmx_csr_sizes(const hmx_csr* c, int64_t* m, int64_t* n, int64_t* nnz);
/* rowptr: m + 1 entries, colidx / values: nnz entries; any may be NULL */
int hmx_csr_export(const hmx_csr* c, int64_t* rowptr, int64_t* colidx, double* values);
int hmx_csr_destroy(hmx_csr* c);

/* ---- build options beyond the reference's keywords ------------------------- */
typedef struct hmx_rankpred hmx_rankpred;
typedef struct hmx_build_options {
    int32_t aca_device;   /* 0: ACA+ on host threads (the default build);
                             1: batched FP64 ACA+ on the GPU (built-in 1/r kernel
                                with dims 1, or the dipole tensor with dims 3) */
    int32_t initial_rank; /* first rank capacity per block without a predictor (0: 16) */
    const hmx_rankpred* predictor; /* NULL or a trained predictor: capacity per block
                                      = ceil((1 + cap_margin) * predicted ACA+ rank) */
    double cap_margin;
    int32_t refine_samples; /* > 0 (with a predictor): ACA+ first runs on about this many
                               evenly spaced blocks, a copy of the predictor is fine-tuned
                               on their ranks (refine_epochs, on the GPU) and predicts the
                               capacities of the rest; the caller's predictor is unchanged */
    int32_t refine_epochs;  /* 0: 200 (minibatches of 256, Adam from a fresh state) */
} hmx_build_options;
typedef struct hmx_build_stats {
    int64_t blocks;            /* admissible blocks */
    int64_t chunks;            /* memory-bounded groups of blocks of the GPU ACA+ */
    int64_t passes;            /* capacity passes (1 = every block fit its first capacity) */
    int64_t launches;          /* GPU ACA+ kernel launches */
    int64_t unconverged_first; /* blocks that outgrew their first capacity */
    int64_t probe_blocks;      /* blocks run before the capacities were refined */
    int64_t slot_elems;        /* sum over passes of (m + n) * capacity (allocated terms) */
    int64_t used_elems;        /* sum of (m + n) * ACA+ rank (filled terms) */
    double aca_kernel_ms;      /* GPU ACA+ kernel time */
    double recompress_ms;      /* GPU recompression (QR + Jacobi SVD) kernel time */
    double aca_wall_s;         /* GPU ACA+ phase incl. copies and recompression */
    double build_s;            /* host build (trees, ACA+, recompression, layout) */
    double total_s;            /* build_s + device upload of the requested storage */
} hmx_build_stats;
/* hmx_hmatrix_build with options (NULL = defaults) and statistics (may be
 * NULL).  The result is identical for every option: the GPU ACA+ reproduces
 * the host ACA+ factors bit for bit, and the rank capacity only changes the
 * schedule.  No reference counterpart beyond HMatrix(...) (hmatrix.jl:72-148,
 * ACA_plus aca.jl:36-106), which always runs ACA+ serially on the host. */
int hmx_hmatrix_build_ex(const hmx_tree* target, const hmx_tree* source, int32_t kernel_id,
                         const double* target_xyz, const double* source_xyz, hmx_block_fn fill,
                         void* ctx, double eta, double eps, int32_t svd_recompress,
                         int32_t storage_mask, int32_t device, int32_t nthreads,
                         const hmx_build_options* options, hmx_build_stats* stats,
                         hmx_hmatrix** out);
/* Rank-predictor inputs per admissible block (see hmx_hmatrix_block_features). */
#define HMX_RANK_FEATURES 9

/* Per admissible block in approx-list order (block.jl:127-155 traverse order):
 * HMX_RANK_FEATURES floats features[9*b ...], chosen to be unchanged when all
 * coordinates are scaled by one factor (diam = 2 * radius of tree.jl:86-87,
 * dist = centre distance of block.jl:63, p = 1 for the 1/r kernel, 3 for the
 * dipole tensor, 0 otherwise):
 *   log(diam_s / dist), log(diam_t / dist), log(tol * dist^p), log n_s, log n_t,
 *   then per cluster (source, then target) 0.5 log(l2 / l1), 0.5 log(l3 / l1)
 *   for the eigenvalues l1 >= l2 >= l3 of its points' covariance;
 * then the ACA+ rank, the rank after recompression and the first GPU capacity
 * (0 for a host build).  *count = number of admissible blocks; the arrays may
 * be NULL.  No reference counterpart (training data of the rank predictor). */
int hmx_hmatrix_block_features(const hmx_hmatrix* h, int64_t* count, float* features,
                               int32_t* aca_rank, int32_t* rank, int32_t* capacity);

/* ---- rank predictor (no reference counterpart) ------------------------------
 * MLP 9 -> 64 -> 64 -> 1 (ReLU) from the block features above to
 * log(1 + ACA+ rank); BF16 weights with FP32 accumulation, trained on the GPU
 * (Adam, mean squared error).  features: n rows of HMX_RANK_FEATURES floats. */
int hmx_rankpred_create(int32_t hidden /* 64 */, uint64_t seed, int32_t device,
                        hmx_rankpred** out);
int hmx_rankpred_nparams(int64_t* n);
/* minibatch Adam over `epochs` shuffled passes; loss_per_epoch (may be NULL)
 * receives the epoch's mean squared error in log(1 + rank).  The feature
 * normalisation (mean, 1/std) is fixed from the first training set. */
int hmx_rankpred_train(hmx_rankpred* p, const float* features, const float* ranks, int64_t n,
                       int32_t epochs, int32_t batch, float lr, uint64_t seed,
                       float* loss_per_epoch);
/* loss and its gradient w.r.t. the parameters over one batch of n samples */
int hmx_rankpred_grad(hmx_rankpred* p, const float* features, const float* ranks, int64_t n,
                      float* grad, float* loss);
/* predicted ACA+ ranks (real valued) */
int hmx_rankpred_predict(const hmx_rankpred* p, const float* features, int64_t n, float* ranks);
/* get (get=1) or set (get=0) the FP32 master parameters, their BF16 values (get
 * only) and the normalisation norm[0..8] = mean, norm[9..17] = 1/std.  Parameter
 * order: W1 (64x9 row-major), b1, W2 (64x64), b2, W3 (64), b3. */
int hmx_rankpred_params(hmx_rankpred* p, int32_t get, float* master, float* bf16, float* norm);
int hmx_rankpred_destroy(hmx_rankpred* p);

/* (Re)build the device operator of every precision in storage_mask on `device`
 * from the host-side H-matrix (the reference's kernel_array uploads,
 * hmatrix.jl:104,133-147), replacing an existing one; release frees it. */
int hmx_hmatrix_materialize(hmx_hmatrix* h, int32_t storage_mask, int32_t device);
int hmx_hmatrix_release(hmx_hmatrix* h, int32_t storage_mask);
/* Free the per-stream product scratch (see hmx_matvec) that `stream` holds, or
 * that every stream holds when all_streams != 0, for every materialised
 * precision, after synchronising those streams.  Each stream that has run a
 * product keeps, per pass width W used (1, 4, 16, 32 or 48 columns), the
 * staging array of hmx_staging_layout, about (n + R) * W elements, and W partial
 * sums (FP64, or FP32 for the other storages) per leaf-result row (one set of a
 * leaf's rows for each piece that it is cut into) and far-field chunk row: 1.6 GB
 * at N = 262,144 with FP32 storage and W = 16, 4.8 GB with W = 48.  The scratch of
 * a wider pass serves the passes of 16 and 32 columns too, and one of 32 or 48 is
 * allocated only within half of the free device memory (or HMX_WIDE_SCRATCH_LIMIT
 * bytes); hmx_hmatrix_scratch_usage reports what is held.  It is kept until this
 * call, hmx_hmatrix_release or hmx_hmatrix_destroy; the next product on the
 * stream allocates it again.  At most HMX_SCRATCH_STREAMS streams (default 8)
 * hold scratch per materialised precision: a product on a further stream first
 * frees the scratch of the least recently used one, after a device
 * synchronisation.  No reference counterpart (the reference keeps one
 * Vx_buffer per H-matrix, hmatrix.jl:135). */
int hmx_hmatrix_release_scratch(hmx_hmatrix* h, void* stream, int32_t all_streams);
/* Product scratch currently held: *bytes over every materialised precision,
 * stream and pass width, and *entries = the (precision, stream) pairs holding
 * it.  No reference counterpart (monitoring of the scratch above). */
int hmx_hmatrix_scratch_usage(const hmx_hmatrix* h, int64_t* bytes, int64_t* entries);
/* Size of the source/T staging array that one product pass of `width`
 * right-hand sides (1, 4 or 16) allocates for an operator of `storage` precision
 * with n source rows and R stacked low-rank rows (sizes[4] of hmx_hmatrix_sizes).
 * A product with nrhs > 16 runs ceil(nrhs / 48) passes of 16, 32 or 48, the wider
 * ones with two or three times the bytes of 16, or narrower passes where that
 * memory is not to be had.  The array has *rows rows of *bytes / *rows bytes, of
 * which [*zero_begin, *zero_end) must read zero (cleared at allocation, and by
 * hmx_matvec_noalloc on every call).  The kernels read an array below 4 GiB through 32-bit buffer offsets and a larger
 * one through 64-bit global loads; rows are 32-bit indices, so
 * HMX_ERR_UNSUPPORTED from 2^31 rows.  No reference counterpart (memory
 * planning for the reference's Vx_buffer, hmatrix.jl:135). */
int hmx_staging_layout(int64_t n, int64_t R, int32_t storage, int32_t width, int64_t* rows,
                       int64_t* bytes, int64_t* zero_begin, int64_t* zero_end);
/* sizes[0..7] = m, n, n_dense, n_lowrank, R (= length(Vx_buffer)), length of
 * dense_blocks, U_matrices, V_matrices in the flattened layout. */
int hmx_hmatrix_sizes(const hmx_hmatrix* h, int64_t* sizes);
/* The reference's flattened layout (HMatrix{T} fields, hmatrix.jl:46-57,
 * 95-147) exactly: index maps (1-based), dense_block_indices 5 x n_dense,
 * U_block_indices 5 x n_lowrank (rows 3-4 = Vx range), V_block_indices 3 x R,
 * row-major payloads.  Any pointer may be NULL. */
int hmx_hmatrix_export_reference_layout(const hmx_hmatrix* h, int64_t* target_index_map,
                                        int64_t* source_index_map, int64_t* dense_block_indices,
                                        int64_t* U_block_indices, int64_t* V_block_indices,
                                        double* dense_blocks, double* U_matrices,
                                        double* V_matrices);
/* HMatrixCPU's dense_block_indices / approx_block_indices (hmatrix.jl:18-27):
 * (row_start, row_end, col_start, col_end), 1-based inclusive, 4 x n each, in
 * list order (dense: direct list then storage fallbacks). */
int hmx_hmatrix_export_block_ranges(const hmx_hmatrix* h, int64_t* dense_ranges,
                                    int64_t* lowrank_ranges);
/* info(::HMatrixCPU) (hmatrix.jl:289-330) plus byte counts:
 * out[0] leaves, [1] admissible_leaves, [2] full_leaves, [3] min_rank,
 * [4] max_rank, [5] min_dense_size, [6] max_dense_size, [7] compression_ratio,
 * [8] nnz_D, [9] nnz_U, [10] nnz_V, [11] device panel bytes F64, [12] F32,
 * [13] BF16, [14] device index/plan bytes (all storages), [15] build seconds */
int hmx_hmatrix_info(const hmx_hmatrix* h, double* out);
/* Layout digests: out[0] index maps, out[1] block tables in list order (ranges,
 * ranks, payload offsets), out[2] U payload, out[3] V payload (64-bit hashes of
 * the FP64 words).  Two builds with equal digests have the same flattened
 * layout (hmatrix.jl:95-147) bit for bit, without exporting it; used to show
 * that every ACA+ schedule (host threads, GPU, predictor capacities) yields the
 * same H-matrix.  No reference counterpart (its tests compare the fields). */
int hmx_hmatrix_checksum(const hmx_hmatrix* h, uint64_t* out);
/* ---- on-disk H-matrix (no reference counterpart: the reference rebuilds
 *      every HMatrix from its kernel, hmatrix.jl:72-148) ----------------------
 * hmx_hmatrix_save writes the host operator (index maps, block lists, FP64
 * factors, the entry source: coordinates for built-in kernels, the dense
 * payload for callback kernels; the per-block rank statistics) to `path`
 * through a temporary file renamed at the end.  flags: HMX_SAVE_DENSE also
 * writes the dense payload of a built-in kernel (evaluating it on the host if
 * needed).  Device storage is not saved.
 * hmx_hmatrix_load reads such a file, checks its checksums and every index
 * against the sizes it addresses (HMX_ERR_ARG on any mismatch), and returns an
 * H-matrix equal to the saved one, materialised in `storage_mask` on `device`
 * like hmx_hmatrix_build.  Files are little-endian, version 1. */
enum { HMX_SAVE_DENSE = 1 };
int hmx_hmatrix_save(hmx_hmatrix* h, const char* path, int32_t flags);
int hmx_hmatrix_load(const char* path, int32_t storage_mask, int32_t device, hmx_hmatrix** out);
int hmx_hmatrix_destroy(hmx_hmatrix* h);

/* ---- product: replaces mul!(result, H::HMatrix{T}, x) (mult.jl:159-189) ----
 * Y[:, c] = H * X[:, c] for c < nrhs.  X (n x nrhs, leading dim ldx) and Y
 * (m x nrhs, ldy) are device pointers of io_dtype (HMX_F64 or HMX_F32) on the
 * H-matrix's device; `storage` selects which materialised precision is used.
 * Y is fully overwritten (no zeroing needed); X is read-only.  Asynchronous
 * and stream-ordered on `stream` (NULL = default stream).  Scratch is per
 * (H-matrix, stream), so concurrent calls on different streams are safe;
 * concurrent calls on one stream are ordered by the stream.  The first call on
 * a new stream allocates its scratch (hipMalloc), and so does the first with a
 * wider pass (nrhs 1, 2-4, 5-16, 17-32 and 33 or more differ).  Under stream
 * capture a product with nrhs > 4 allocates nothing once the stream has run any
 * product with nrhs > 4. */
int hmx_matvec(hmx_hmatrix* h, int32_t storage, const void* X, int64_t ldx, void* Y, int64_t ldy,
               int32_t nrhs, int32_t io_dtype, void* stream);

/* ---- product on host vectors: replaces mul!(result::Vector, H::HMatrixCPU,
 *      x::Vector) (mult.jl:6-32) and *(H::HMatrixCPU, x::Vector) (mult.jl:35-39)
 * y[:, c] = H * x[:, c] for c < nrhs, with x (n x nrhs, leading dim ldx) and y
 * (m x nrhs, ldy) FP64 HOST arrays.  The product runs on the GPU: x is copied
 * to the device, the FP64 operator computes the product there (it is
 * materialised on the H-matrix's device on the first call if the build did
 * not request it -- the flatten=false / HMatrixCPU case), and y is copied back
 * before the call returns.  y is fully overwritten; x is read-only.  There is
 * no CPU product in this library. */
int hmx_matvec_host(hmx_hmatrix* h, const double* x, int64_t ldx, double* y, int64_t ldy,
                    int32_t nrhs);

/* hmx_matvec without any device allocation.  No counterpart in the reference
 * (whose mul! reuses the Vx_buffer allocated with the H-matrix, hmatrix.jl:135):
 * it is for callers that cannot allocate, such as code under HIP graph
 * capture, tight serving loops and harnesses that forbid hipMalloc.  Same
 * arguments, semantics and results (bit for bit) as hmx_matvec, but the
 * per-call scratch (the source / T rows and the partial sums, about
 * (n + R) * 16 * 4 bytes for FP32 with 16 RHS) lives in one static device
 * array of 128 MiB per GPU, held from the first load of the library's kernels
 * on that GPU until the process ends.  A product that needs more is refused
 * with HMX_ERR_UNSUPPORTED before anything is launched.  Every call on a GPU
 * uses the same array, so calls that overlap on one GPU (different streams,
 * threads or H-matrices) race: the caller must order them.  It calls no
 * hipMalloc / hipFree; X, Y and the H-matrix's device operator are the
 * caller's, as for hmx_matvec. */
int hmx_matvec_noalloc(hmx_hmatrix* h, int32_t storage, const void* X, int64_t ldx, void* Y,
                       int64_t ldy, int32_t nrhs, int32_t io_dtype, void* stream);

/* ---- batched products of independent H-matrices (no reference counterpart:
 *      the reference runs one mul! per H-matrix, mult.jl:159-189) -------------
 * All members must be materialised in `storage` on one device.  While the batch
 * exists its members cannot be released, re-materialised or destroyed (those
 * calls return HMX_ERR_STATE).  Calls of one batch on different streams must
 * not overlap (the batch owns one set of scratch arrays).  Every stage of the product is one kernel over
 * all members, and the four stages are replayed as one captured hipGraph per
 * call.  1 <= nrhs <= 16 (the same for all members). */
typedef struct hmx_batch hmx_batch;
int hmx_batch_create(hmx_hmatrix* const* members, int32_t count, int32_t storage, int32_t nrhs,
                     int32_t io_dtype, hmx_batch** out);
/* X[i], Y[i]: device pointers of member i (column-major, leading dims ldx[i],
 * ldy[i]; NULL ld arrays mean n_i / m_i).  Asynchronous on `stream`. */
int hmx_batch_matvec(hmx_batch* b, const void* const* X, const int64_t* ldx, void* const* Y,
                     const int64_t* ldy, void* stream);
/* Autotuner: times every candidate (RHS path: 4-wide VALU or 16-wide MFMA when
 * nrhs <= 4; leaf dispatch order: 0 largest first, 1 tree, 2 XCD chunks) on the
 * given operands, keeps the fastest, appends it to the file named by
 * HMX_TUNE_CACHE (read back by hmx_batch_create).  best_ms may be NULL. */
int hmx_batch_autotune(hmx_batch* b, const void* const* X, const int64_t* ldx, void* const* Y,
                       const int64_t* ldy, int32_t iters, void* stream, double* best_ms);
int hmx_batch_set_config(hmx_batch* b, int32_t rhs_width, int32_t order);
int hmx_batch_get_config(const hmx_batch* b, int32_t* rhs_width, int32_t* order);
int hmx_batch_destroy(hmx_batch* b);

/* Per-stage kernel timing with HIP events recorded on the launch stream
 * (stage 0 gather, 1 far-field V*X, 2 partial reduce, 3 near+far U panel
 * product).  enable != 0 starts recording; read returns summed milliseconds
 * and launch counts per stage after synchronising the recorded events. */
int hmx_profile_enable(hmx_hmatrix* h, int32_t enable);
int hmx_profile_read(hmx_hmatrix* h, double* ms, int64_t* launches, int32_t reset);

#ifdef __cplusplus
}
#endif
#endif
