// device.hip -- gfx950 device layout, panel generation and the H-matrix product.
//
// Reference counterpart: the two KernelAbstractions kernels and the driver of
// mult.jl:41-189 (V_mult_vec_kernel!, DU_mult_vec_kernel!, mul!).  The work is
// reorganised for CDNA4 instead of translated:
//
//   * Leaf panels.  Every output row belongs to exactly one target-tree leaf.
//     For each leaf (split into row groups of <= 64 rows) all its near-field
//     dense-block rows and all its low-rank U rows are packed into ONE panel
//     of `rows x K` entries, K = sum of the dense blocks' column counts plus
//     the ranks of the low-rank blocks covering the leaf.  Column c of the
//     panel multiplies row colidx[c] of a combined source array
//         S = [ X permuted by source_index_map (n rows) ; T = V*X (R rows) ; 0 ].
//     The product of a leaf is then one small GEMM  Y_leaf = P_leaf * S[colidx]
//     written once, with no atomics and no O(m * blocks) scan (the reference's
//     DU kernel tests every block for every row, mult.jl:95-118).
//   * Far field.  V rows are grouped by source cluster (all blocks sharing a
//     source cluster read the same contiguous S rows) into panels of <= 64
//     rank-rows; long clusters are split into column chunks whose partial
//     results are summed in a fixed order (deterministic, atomic-free).
//   * Tiles.  A panel is stored as k-tiles of TK = 64 bytes / sizeof(storage)
//     columns; inside a k-tile, row tiles of 16 rows are stored chunk-major so
//     that lane l of a wave reads 16 contiguous bytes = row (l % 16), chunk
//     (l / 16): one fully coalesced 1 KiB load per wave per 16x TK tile, which
//     is exactly the A-operand layout of MFMA 16x16x4 (f32/f64) and 16x16x32
//     (bf16).  Partial row tiles are stored compactly (no padding bytes).
//   * Multi-RHS (16 columns) runs on MFMA with the RHS as the N dimension;
//     a single RHS is a VALU GEMV over the same tiles.
//
// Stages per call (one launch each, stream ordered): gather X -> S, far-field
// panels (V*X), partial reduce, leaf panels (near field + U*T) -> leaf-result
// rows, sum of each row's pieces -> Y.
#include "device_op.hpp"

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <cstdio>
#include <string>
#include <vector>

namespace hmx {

namespace {



// Dispatch order of the leaf items.  "xcd" (the default of a single
// operator): the tree-ordered (spatially coherent) item list is cut into kXcds
// contiguous chunks of equal work and interleaved, so that with round-robin
// workgroup placement (workgroup i -> XCD i % kXcds) every XCD's L2 serves one
// compact region and neighbouring row groups share their S rows there.  Once
// the leaf items are split into pieces of similar size this measured 3% faster
// than largest first ("lpt", which was best while a few whole items lasted
// most of the launch).  "tree" keeps tree order.  HMX_ITEM_ORDER overrides.
constexpr int kXcds = 8;

}  // namespace

// Work of a leaf item in panel elements per wave plus a fixed cost.
int64_t leaf_item_work(const PairItem& it) {
    const int64_t a = int64_t(it.sh_kt) * (it.rows[0] + it.rows[1]) +
                      int64_t(it.pr_kt[0]) * it.rows[0] + int64_t(it.pr_kt[1]) * it.rows[1];
    return a * 64 + 4096;
}

// Size of the k-range pieces that leaf items are cut into, from the leaf bytes of
// the operator: total / kLeafPieces, at least 1 MiB, so that no item outlasts the
// launch (swept at N = 262,144).  An operator of at most kSmallLeaf bytes has fewer
// whole items than the workgroups that are resident, or too few rounds of them; it takes
// total / kSmallPieces, between 64 and 384 KiB.  us per product with 1 MiB pieces and with
// this rule: N = 4,096 FP64 with one right-hand side 78 and 39, FP32 with 16 47 and 29;
// N = 14,000 FP32 with four 130 and 119; N = 16,384 BF16 with 16 109 and 98; N = 20,011
// FP32 with three 187 and 182.  Finer pieces pay for their start-up, about 5 us of one
// workgroup each, and a batch of such operators, which fills the GPU without cutting its
// members (and must cut them as their own products do, for the same bits), pays for every
// one: 16 members of 2,048 .. 16,384 points take 461 us with 1 MiB pieces, 473 us with at
// most 384 KiB, 484 us with at most 256 KiB.  Above the line the larger pieces are as
// good for one product too (N = 16,384 FP64 with 40: 437 against 450 us).
constexpr int64_t kLeafPieces = 12288, kSmallPieces = 512;
constexpr int64_t kMiB = int64_t(1) << 20;
constexpr int64_t kSmallLeaf = 800 * kMiB;
constexpr int kMaxPieces = 64;
// Target rows up to which an operator without cut items writes Y from the leaf
// kernel: scattered stores, but one launch less (N = 1,000, one right-hand side:
// 17.3 -> 14.5 us per product).
constexpr int64_t kDirectRows = 8192;
// Source rows and panel bytes up to which a product with one right-hand side reads X in
// place, without the gather launch (about 3 us).  A larger operator reads each X row many
// times, through scattered loads where S has it in tree order.  us per product, gathered
// and in place: circle N = 1,000 FP64 15.0 and 12.1, N = 4,000 17.8 and 14.8; cube N =
// 1,200 FP64 17.3 and 14.4, N = 4,096 BF16 (30 MB) 17.8 and 16.0, but N = 2,500 FP64
// (48 MB) 24.0 and 26.1, N = 12,000 on the circle 24.3 and 25.8.
constexpr int64_t kXdirRows = 8192, kXdirBytes = 32 * kMiB;

int64_t leaf_piece_bytes(int64_t total, int64_t pieces) {
    // HMX_LEAF_MIN_PIECE sets the smallest piece (bytes), e.g. to split the
    // items of small operators in tests
    const char* min_env = std::getenv("HMX_LEAF_MIN_PIECE");
    const int64_t min_piece =
        min_env ? std::max<int64_t>(4096, std::atoll(min_env))
        : total > kSmallLeaf
            ? kMiB
            : std::min(kMiB * 3 / 8, std::max(kMiB / 16, total / kSmallPieces));
    return std::max(total / pieces, min_piece);
}

// Cut the leaf items into pieces of about `piece` bytes along k, so that the
// launch has several items per resident workgroup and no single item outlasts the rest.
// Every piece gets its own leaf-result rows; `src` (per permuted target row)
// says which rows to sum.  Returns the leaf-result rows used.
int64_t split_leaf_items(std::vector<PairItem>& items, int TK, int64_t piece,
                         std::vector<RowSrc>& src) {
    std::vector<PairItem> out;
    out.reserve(items.size());
    int64_t nrows = 0;
    for (const PairItem& it : items) {
        const int64_t c =
            piece > 0 ? std::min<int64_t>(kMaxPieces, (leaf_item_work(it) + piece - 1) / piece) : 1;
        const int32_t rows = it.rows[0] + it.rows[1];
        for (int g = 0; g < 2; g++)
            for (int32_t r = 0; r < it.rows[g]; r++)
                src[it.out_off[g] + r] = RowSrc{static_cast<uint32_t>(nrows + g * it.rows[0] + r),
                                                static_cast<int16_t>(c), static_cast<int16_t>(rows)};
        // Piece boundaries along the work of the panels: the shared tiles (both
        // row groups together), then the private ones in proportion.  Each piece
        // is one contiguous k-range of each row group.
        const int64_t wsh = int64_t(it.sh_kt) * rows;
        const int64_t wpr = int64_t(it.pr_kt[0]) * it.rows[0] + int64_t(it.pr_kt[1]) * it.rows[1];
        auto bound = [&](int64_t p, int32_t& sh, int32_t (&pr)[2]) {
            const int64_t w = (wsh + wpr) * p / c;
            sh = static_cast<int32_t>(std::min<int64_t>(it.sh_kt, w / rows));
            for (int g = 0; g < 2; g++)
                pr[g] = p == c     ? it.pr_kt[g]
                        : w <= wsh ? 0
                                   : static_cast<int32_t>(it.pr_kt[g] * (w - wsh) / wpr);
        };
        for (int64_t p = 0; p < c; p++) {
            PairItem q = it;
            int32_t s0, s1, a0[2], a1[2];
            bound(p, s0, a0);
            bound(p + 1, s1, a1);
            q.sh_kt = s1 - s0;
            q.sh_col = it.sh_col + int64_t(s0) * TK;
            for (int gi = 0; gi < 2; gi++) {
                q.pr_kt[gi] = a1[gi] - a0[gi];
                q.pr_col[gi] = it.pr_col[gi] + int64_t(a0[gi]) * TK;
                q.data[gi] = it.data[gi] + int64_t(s0 + a0[gi]) * TK * it.rows[gi];
            }
            q.part = nrows;
            nrows += rows;
            out.push_back(q);
        }
    }
    items.swap(out);
    return nrows;
}

// Cut the (tree-ordered) list into kXcds contiguous chunks of equal work and
// interleave them, so that workgroup i, placed on XCD i % kXcds, takes items
// of chunk i % kXcds (a chunk that runs out borrows from the fullest one).
template <typename T, typename Work>
void xcd_interleave(std::vector<T>& items, Work work) {
    int64_t total = 0;
    for (const T& it : items) total += work(it);
    if (total <= 0) return;
    std::vector<std::vector<T>> chunk(kXcds);
    int64_t acc = 0;
    for (const T& it : items) {
        const int c = static_cast<int>(std::min<int64_t>(kXcds - 1, acc * kXcds / total));
        chunk[c].push_back(it);
        acc += work(it);
    }
    std::vector<size_t> pos(kXcds, 0);
    std::vector<T> out;
    out.reserve(items.size());
    for (size_t p = 0; out.size() < items.size(); p++) {
        int c = static_cast<int>(p % kXcds);
        if (pos[c] == chunk[c].size()) {
            size_t best = 0;
            for (int q = 0; q < kXcds; q++)
                if (chunk[q].size() - pos[q] > chunk[best].size() - pos[best]) best = q;
            c = static_cast<int>(best);
        }
        out.push_back(chunk[c][pos[c]++]);
    }
    items.swap(out);
}

void order_leaf_items(std::vector<PairItem>& items, const char* env) {
    if (items.size() < 2 * kXcds) return;
    auto work = leaf_item_work;
    if (!env || std::string(env) == "lpt") {
        std::stable_sort(items.begin(), items.end(),
                         [&](const PairItem& a, const PairItem& b) { return work(a) > work(b); });
        return;
    }
    if (env && std::string(env) == "tree") return;
    xcd_interleave(items, work);
}

namespace {

// Far-field items: largest first (their B rows are shared inside the
// workgroup, so dispatch order only matters for the tail).
// (The XCD-interleaved tree order measured 14% slower for far items, and
// placing the items that read the same X rows on one XCD at about the same
// time measured the same as largest first.)
void order_far_items(std::vector<FarItem>& items) {
    std::stable_sort(items.begin(), items.end(), [](const FarItem& a, const FarItem& b) {
        return int64_t(a.ktiles) * a.nrg > int64_t(b.ktiles) * b.nrg;
    });
}

// Byte offsets of the three scratch arrays of one pass width inside the static
// scratch of hmx_matvec_noalloc (each 256-byte aligned): S rows, far-field
// partials, leaf-result rows.
struct NoAllocPlan {
    size_t s = 0, p = 0, lp = 0, total = 0;
};
NoAllocPlan noalloc_plan(const DeviceOp& op, int W) {
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t pe = p_elem(op.storage);
    NoAllocPlan pl;
    pl.s = 0;
    pl.p = up(static_cast<size_t>(staging(op, W).bytes));
    pl.lp = pl.p + up(static_cast<size_t>(std::max<int64_t>(op.npartial, 1)) * W * pe);
    pl.total = pl.lp + up(static_cast<size_t>(std::max<int64_t>(op.nlrows, 1)) * W * pe);
    return pl;
}

// Usable bytes of that static scratch: HMX_NOALLOC_LIMIT lowers them, e.g. to exercise
// the size checks on small operators; it never raises them.
size_t noalloc_limit() {
    size_t limit = kNoAllocScratchBytes;
    if (const char* env = std::getenv("HMX_NOALLOC_LIMIT")) {
        const long long v = std::atoll(env);
        if (v >= 0 && static_cast<size_t>(v) < limit) limit = static_cast<size_t>(v);
    }
    return limit;
}

}  // namespace

void device_destroy(DeviceOp* op) {
    if (!op) return;
    (void)hipSetDevice(op->device);
    for (void* p : {op->panel, (void*)op->itemsB, (void*)op->colidx, (void*)op->itemsA,
                    (void*)op->groups, (void*)op->tmap0, (void*)op->rowsrc, (void*)op->inv_smap, (void*)op->smap0, (void*)op->colx})
        if (p) (void)hipFree(p);
    for (auto& kv : op->scratch)
        for (auto& w : kv.second.w)
            if (w.S) (void)hipFree(w.S);
    for (auto& e : op->ev)
        for (auto& pr : e) {
            (void)hipEventDestroy(pr.first);
            (void)hipEventDestroy(pr.second);
        }
    delete op;
}

int64_t device_panel_bytes(const DeviceOp* op) {
    return op ? op->panel_elems * static_cast<int64_t>(elem_size(op->storage)) : 0;
}
int64_t device_index_bytes(const DeviceOp* op) {
    if (!op) return 0;
    return op->ncol * 4 + op->nA * static_cast<int64_t>(sizeof(FarItem)) +
           op->nB * static_cast<int64_t>(sizeof(PairItem)) +
           op->nG * static_cast<int64_t>(sizeof(ReduceGroup)) +
           op->m * static_cast<int64_t>(4 + sizeof(RowSrc)) + op->n * 4 +
           (op->colx ? (op->ncol + op->n) * 4 : 0);
}

// Build the device operator for one storage precision.
void device_build(HMatrix& h, int storage) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
        throw Error(HMX_ERR_HIP, "no HIP device available");
    if (h.device < 0 || h.device >= ndev) throw Error(HMX_ERR_ARG, "invalid device ordinal");
    // Rows of the staging array S before X, left unused: 0 unless
    // HMX_STAGING_ROW_OFFSET is set (a test hook that moves every S row index
    // past a given row, e.g. past 4 GiB of S, without a matrix that large).
    const char* s0env = std::getenv("HMX_STAGING_ROW_OFFSET");
    const int64_t s0 = s0env ? std::max<int64_t>(0, std::atoll(s0env)) : 0;
    if (h.m >= (int64_t(1) << 31) || s0 + h.n + h.R + 64 >= (int64_t(1) << 31))
        throw Error(HMX_ERR_UNSUPPORTED, "matrix too large for 32-bit device indices");
    if ((h.src.kernel_id == HMX_KERNEL_LAPLACE || h.src.kernel_id == HMX_KERNEL_LOG2D) &&
        (h.target_dims != 1 || h.source_dims != 1))
        throw Error(HMX_ERR_UNSUPPORTED, "scalar built-in kernels need dims == 1");
    if (h.src.kernel_id == HMX_KERNEL_DIPOLE && (h.target_dims != 3 || h.source_dims != 3))
        throw Error(HMX_ERR_UNSUPPORTED, "the dipole tensor kernel needs dims == 3");
    DeviceGuard guard(h.device);
    const auto tb0 = std::chrono::steady_clock::now();
    auto since = [&] {
        return std::chrono::duration<double>(std::chrono::steady_clock::now() - tb0).count();
    };
    auto op = std::make_unique<DeviceOp>();
    op->storage = storage;
    op->device = h.device;
    op->m = h.m;
    op->n = h.n;
    op->R = h.R;
    op->s0 = s0;
    const int TK = tk_of(storage);
    // Far-field column chunk, a multiple of every TK.  Source clusters wider than
    // a chunk write partial rows that k_reduce sums; 8192 halves those partials
    // against 2048 (measured: the far kernel's time is the same, the reduce 2x
    // shorter) while keeping items at most 4 x 64 x 8192 entries.  HMX_FAR_CHUNK
    // overrides it.
    const char* ch_env = std::getenv("HMX_FAR_CHUNK");
    const int64_t ch_req = ch_env ? std::atoll(ch_env) : 8192;
    int64_t CH = ch_req >= 32 && ch_req % 32 == 0 ? ch_req : 8192;

    // -- far field: group low-rank blocks by source cluster -----------------------
    // Per source cluster the rank rows of its blocks are stacked (T rows, in
    // this order) and cut into 64-row groups; per column chunk the row-group
    // panels are stored back to back and dispatched kWaves groups at a time.
    std::vector<Item> itemsA;     // one per (row group, chunk): generation only
    std::vector<GenA> gensA;
    std::vector<FarItem> itemsF;  // dispatch
    std::vector<ReduceGroup> groups;
    std::vector<int64_t> vrow;  // per T row: offset of its V row in the V payload
    std::vector<int64_t> trow_of_block(h.lowrank.size());
    int64_t data_off = 0, npartial = 0;
    {
        std::map<int64_t, std::vector<int64_t>> by_src;
        for (size_t b = 0; b < h.lowrank.size(); b++)
            if (h.lowrank[b].k > 0) by_src[h.lowrank[b].snode].push_back(static_cast<int64_t>(b));
        // Where the far field is a few long, thin panels (points on a curve: rank 3 or
        // 4), the longest chain of k-tiles sets the time of its launch: about 0.12 us per
        // tile of one wave, against far bytes / 6 TB/s for the launch as a whole.  Such an
        // operator takes 128 k-tiles per chunk (FP64 on a circle: N = 20,000 49 -> 28 us per
        // product, N = 12,000 33 -> 25 us; operators in a volume never do).
        if (!ch_env) {
            double bytes = 0, chain = 0;
            for (auto& kv : by_src) {
                const LowRankBlock& f = h.lowrank[kv.second[0]];
                const int64_t ncols = f.c1 - f.c0 + 1;
                int64_t Rs = 0;
                for (int64_t b : kv.second) Rs += h.lowrank[b].k;
                const int64_t nrg = (Rs + 63) / 64, split = nrg == 1 ? 4 : nrg == 2 ? 2 : 1;
                bytes += double(Rs) * ncols * elem_size(storage);
                chain = std::max(chain, double(std::min(ncols, CH)) / (TK * split));
            }
            if (chain * 0.12 > 8.0 + 2.0 * bytes / 6e6) CH = 128 * TK;
        }
        int64_t t = 0;
        for (auto& kv : by_src) {
            const auto& blocks = kv.second;
            const LowRankBlock& f = h.lowrank[blocks[0]];
            const int64_t ncols = f.c1 - f.c0 + 1;
            const int64_t tstart = t;
            for (int64_t b : blocks) {
                const LowRankBlock& L = h.lowrank[b];
                trow_of_block[b] = t;
                for (int64_t j = 0; j < L.k; j++) vrow.push_back(L.voff + j * ncols);
                t += L.k;
            }
            const int64_t Rs = t - tstart;
            const int64_t nrg = (Rs + 63) / 64;
            const int64_t nch = (ncols + CH - 1) / CH;
            int64_t pb = -1;
            if (nch > 1) {
                pb = npartial;
                npartial += Rs * nch;
                groups.push_back({pb, tstart, static_cast<int32_t>(Rs), static_cast<int32_t>(nch)});
            }
            for (int64_t c = 0; c < nch; c++) {
                const int64_t nc = std::min<int64_t>(CH, ncols - c * CH);
                const int64_t kt = (nc + TK - 1) / TK;
                for (int64_t g0 = 0; g0 < nrg; g0 += kWaves) {
                    const int64_t g1 = std::min<int64_t>(nrg, g0 + kWaves);
                    FarItem fi{};
                    fi.data_off = data_off;
                    fi.col_off = s0 + (f.c0 - 1) + c * CH;
                    fi.out_off = nch > 1 ? pb + c * Rs + 64 * g0 : tstart + 64 * g0;
                    fi.ktiles = static_cast<int32_t>(kt);
                    fi.ncols = static_cast<int32_t>(nc);
                    fi.nrg = static_cast<int16_t>(g1 - g0);
                    fi.to_T = nch > 1 ? 0 : 1;
                    for (int64_t g = g0; g < g1; g++) {
                        const int32_t rows = static_cast<int32_t>(std::min<int64_t>(64, Rs - 64 * g));
                        Item it{};
                        it.data_off = data_off;
                        it.rows = rows;
                        it.ktiles = static_cast<int32_t>(kt);
                        it.ncols = static_cast<int32_t>(nc);
                        itemsA.push_back(it);
                        gensA.push_back({tstart + 64 * g, c * CH});
                        data_off += kt * TK * rows;
                        fi.rows_last = rows;
                    }
                    itemsF.push_back(fi);
                }
            }
        }
    }
    // -- leaf panels -----------------------------------------------------------------
    const std::vector<int64_t>& ls = h.target_leaf_start;  // 0-based, with end sentinel
    const int64_t nleaf = static_cast<int64_t>(ls.size()) - 1;
    std::vector<std::vector<int32_t>> dense_of(nleaf), lr_of(nleaf);
    auto leaf_range = [&](int64_t r0, int64_t r1) {  // 0-based [r0, r1)
        int64_t a = std::upper_bound(ls.begin(), ls.end(), r0) - ls.begin() - 1;
        int64_t b = std::lower_bound(ls.begin(), ls.end(), r1) - ls.begin();
        return std::make_pair(a, b);
    };
    for (size_t d = 0; d < h.dense.size(); d++) {
        auto [a, b] = leaf_range(h.dense[d].r0 - 1, h.dense[d].r1);
        for (int64_t l = a; l < b; l++) dense_of[l].push_back(static_cast<int32_t>(d));
    }
    for (size_t d = 0; d < h.lowrank.size(); d++) {
        if (h.lowrank[d].k == 0) continue;
        auto [a, b] = leaf_range(h.lowrank[d].r0 - 1, h.lowrank[d].r1);
        for (int64_t l = a; l < b; l++) lr_of[l].push_back(static_cast<int32_t>(d));
    }
    const int64_t zero_row = s0 + h.n + h.R;
    const bool builtin = h.src.kernel_id != HMX_KERNEL_CALLBACK;
    // Row groups (<= 64 rows) in target order; consecutive row groups are paired
    // when they share columns (blocks covering both), choosing the pairing that
    // maximises the shared columns (dynamic programme over the sequence).
    struct Unit {
        int64_t r0;
        int32_t rows;
        int64_t leaf;
    };
    std::vector<Unit> units;
    for (int64_t l = 0; l < nleaf; l++)
        for (int64_t r0 = ls[l]; r0 < ls[l + 1]; r0 += 64)
            units.push_back({r0, static_cast<int32_t>(std::min<int64_t>(64, ls[l + 1] - r0)), l});
    const int64_t nu = static_cast<int64_t>(units.size());
    auto intersect = [](const std::vector<int32_t>& a, const std::vector<int32_t>& b) {
        std::vector<int32_t> out;
        std::set_intersection(a.begin(), a.end(), b.begin(), b.end(), std::back_inserter(out));
        return out;
    };
    auto minus = [](const std::vector<int32_t>& a, const std::vector<int32_t>& b) {
        std::vector<int32_t> out;
        std::set_difference(a.begin(), a.end(), b.begin(), b.end(), std::back_inserter(out));
        return out;
    };
    // Dense blocks of two row groups that cover the same source columns (the
    // same block, or e.g. the blocks of sibling leaves with one neighbour
    // leaf): their columns can share one read of S.  The block tree gives each
    // (row, column) one block, so a source range appears at most once per row
    // group.  Returns the matched blocks of a and of b (in a's order).
    auto match_dense = [&](const std::vector<int32_t>& a, const std::vector<int32_t>& b) {
        std::map<std::pair<int64_t, int64_t>, int32_t> by_cols;
        for (int32_t d : b) by_cols[{h.dense[d].c0, h.dense[d].c1}] = d;
        std::pair<std::vector<int32_t>, std::vector<int32_t>> m;
        for (int32_t d : a) {
            auto f = by_cols.find({h.dense[d].c0, h.dense[d].c1});
            if (f == by_cols.end()) continue;
            m.first.push_back(d);
            m.second.push_back(f->second);
        }
        return m;
    };
    auto ncols_of = [&](const std::vector<int32_t>& dl, const std::vector<int32_t>& ll) {
        int64_t c = 0;
        for (int32_t d : dl) c += h.dense[d].c1 - h.dense[d].c0 + 1;
        for (int32_t b : ll) c += h.lowrank[b].k;
        return c;
    };
    // HMX_LEAF_PAIRING=0 keeps every row group on its own (layout comparison)
    const char* pairing_env = std::getenv("HMX_LEAF_PAIRING");
    const bool pairing = !(pairing_env && std::string(pairing_env) == "0");
    std::vector<int64_t> gain(static_cast<size_t>(std::max<int64_t>(nu, 1)), 0);
    for (int64_t u = 0; pairing && u + 1 < nu; u++) {
        const int64_t la = units[u].leaf, lb = units[u + 1].leaf;
        const int64_t c = ncols_of(match_dense(dense_of[la], dense_of[lb]).first,
                                   intersect(lr_of[la], lr_of[lb]));
        gain[u] = c >= 2 * TK ? c : 0;  // too few shared columns: not worth a segment
    }
    std::vector<int64_t> best(static_cast<size_t>(nu + 1), 0);
    std::vector<char> take(static_cast<size_t>(nu + 1), 0);
    for (int64_t i = 2; i <= nu; i++) {
        best[i] = best[i - 1];
        if (gain[i - 2] > 0 && best[i - 2] + gain[i - 2] > best[i]) {
            best[i] = best[i - 2] + gain[i - 2];
            take[i] = 1;
        }
    }
    std::vector<std::pair<int64_t, int64_t>> groups_b;  // (first unit, second unit or -1)
    for (int64_t i = nu; i > 0;) {
        if (i >= 2 && take[i]) {
            groups_b.push_back({i - 2, i - 1});
            i -= 2;
        } else {
            groups_b.push_back({i - 1, -1});
            i -= 1;
        }
    }
    std::reverse(groups_b.begin(), groups_b.end());

    std::vector<PairItem> itemsB;
    std::vector<Item> gensB;  // one generation item per panel (col_off into cdesc)
    std::vector<int32_t> colidx;
    std::vector<ColDesc> cdesc;
    {
        // upper bounds (every unit's columns, padding of three segments per
        // group), so that the long appends below never reallocate
        int64_t cols = 0;
        for (const Unit& u : units) cols += ncols_of(dense_of[u.leaf], lr_of[u.leaf]);
        const int64_t pad = 3 * TK * static_cast<int64_t>(groups_b.size());
        colidx.reserve(static_cast<size_t>(cols + pad));
        cdesc.reserve(static_cast<size_t>(cols + pad));
        gensB.reserve(3 * groups_b.size());
    }
    // append the columns of the listed blocks for row group starting at r0
    auto add_colidx = [&](const std::vector<int32_t>& dl, const std::vector<int32_t>& ll) {
        const int64_t c0 = static_cast<int64_t>(colidx.size());
        for (int32_t d : dl) {
            const DenseBlock& D = h.dense[d];
            for (int64_t j = 0; j < D.c1 - D.c0 + 1; j++)
                colidx.push_back(static_cast<int32_t>(s0 + D.c0 - 1 + j));
        }
        for (int32_t b : ll) {
            const LowRankBlock& L = h.lowrank[b];
            for (int64_t j = 0; j < L.k; j++)
                colidx.push_back(static_cast<int32_t>(s0 + h.n + trow_of_block[b] + j));
        }
        while ((colidx.size() - c0) % TK) colidx.push_back(static_cast<int32_t>(zero_row));
        return std::make_pair(c0, static_cast<int32_t>((colidx.size() - c0) / TK));
    };
    auto add_panel = [&](const std::vector<int32_t>& dl, const std::vector<int32_t>& ll,
                         const Unit& U) {
        const int64_t c0 = static_cast<int64_t>(cdesc.size());
        for (int32_t d : dl) {
            const DenseBlock& D = h.dense[d];
            const int64_t nn = D.c1 - D.c0 + 1;
            for (int64_t j = 0; j < nn; j++) {
                if (builtin)
                    cdesc.push_back({h.smap[D.c0 - 1 + j] - 1, 0, 0});
                else
                    cdesc.push_back({D.off + (U.r0 - (D.r0 - 1)) * nn + j, static_cast<int32_t>(nn), 2});
            }
        }
        for (int32_t b : ll) {
            const LowRankBlock& L = h.lowrank[b];
            for (int64_t j = 0; j < L.k; j++)
                cdesc.push_back({L.uoff + (U.r0 - (L.r0 - 1)) * L.k + j, static_cast<int32_t>(L.k), 1});
        }
        while ((cdesc.size() - c0) % TK) cdesc.push_back({0, 0, 3});
        const int64_t K = static_cast<int64_t>(cdesc.size()) - c0;
        Item g{};
        g.data_off = data_off;
        g.col_off = c0;
        g.out_off = U.r0;
        g.rows = U.rows;
        g.ktiles = static_cast<int32_t>(K / TK);
        g.ncols = static_cast<int32_t>(K);
        if (K > 0) gensB.push_back(g);
        const int64_t off = data_off;
        data_off += K * U.rows;
        return off;
    };
    for (const auto& gp : groups_b) {
        PairItem it{};
        it.part = -1;
        const Unit& A = units[gp.first];
        it.out_off[0] = A.r0;
        it.rows[0] = A.rows;
        if (gp.second < 0) {
            auto [c0, kt] = add_colidx(dense_of[A.leaf], lr_of[A.leaf]);
            it.pr_col[0] = c0;
            it.pr_kt[0] = kt;
            it.data[0] = add_panel(dense_of[A.leaf], lr_of[A.leaf], A);
        } else {
            const Unit& B = units[gp.second];
            it.out_off[1] = B.r0;
            it.rows[1] = B.rows;
            auto sd = match_dense(dense_of[A.leaf], dense_of[B.leaf]);
            const auto sl = intersect(lr_of[A.leaf], lr_of[B.leaf]);
            auto [sc, skt] = add_colidx(sd.first, sl);
            it.sh_col = sc;
            it.sh_kt = skt;
            const Unit* UU[2] = {&A, &B};
            const std::vector<int32_t> sdq[2] = {sd.first, sd.second};
            for (int q = 0; q < 2; q++) {
                it.data[q] = add_panel(sdq[q], sl, *UU[q]);
                std::vector<int32_t> matched = sdq[q];
                std::sort(matched.begin(), matched.end());
                const auto pd = minus(dense_of[UU[q]->leaf], matched);
                const auto pl = minus(lr_of[UU[q]->leaf], sl);
                auto [pc, pkt] = add_colidx(pd, pl);
                it.pr_col[q] = pc;
                it.pr_kt[q] = pkt;
                add_panel(pd, pl, *UU[q]);
            }
        }
        itemsB.push_back(it);
    }
    op->panel_elems = data_off;
    const double t_plan = since();
    op->npartial = npartial;

    // -- upload and generate ---------------------------------------------------------
    std::vector<int32_t> tmap0(h.m), inv(h.n);
    for (int64_t i = 0; i < h.m; i++) tmap0[i] = static_cast<int32_t>(h.tmap[i] - 1);
    for (int64_t i = 0; i < h.n; i++) inv[h.smap[i] - 1] = static_cast<int32_t>(i);
    op->tmap0 = upload(tmap0);
    op->inv_smap = upload(inv);
    if (h.n <= kXdirRows && data_off * static_cast<int64_t>(elem_size(storage)) <= kXdirBytes && s0 == 0) {
        std::vector<int32_t> smap0(h.n), colx(colidx);
        for (int64_t i = 0; i < h.n; i++) smap0[i] = static_cast<int32_t>(h.smap[i] - 1);
        for (int32_t& c : colx)
            if (c < h.n) c = smap0[c];
        op->smap0 = upload(smap0);
        op->colx = upload(colx);
    }
    // The FP64 staging arrays are allocated before the panel and freed after
    // generation.  Measured on the MI355X, the product's speed depends on where
    // the panel allocation lands relative to the other large buffers of the
    // process (up to 12% for both product kernels, identical traffic); with
    // this order the usual sequence (FP64, FP32, BF16 operators of one
    // H-matrix) placed the FP32 panel in the fast state in every run.
    auto alloc_panel = [&] {
        const size_t bytes = static_cast<size_t>(std::max<int64_t>(data_off, 1)) * elem_size(storage);
        HIPCHECK(hipMalloc(&op->panel, bytes));
        if (std::getenv("HMX_VERBOSE"))
            std::fprintf(stderr, "[hmx] storage %d panel %p, %zu bytes\n", storage, op->panel, bytes);
    };

    double *dU = nullptr, *dV = nullptr, *dD = nullptr, *dxt = nullptr, *dxs = nullptr;
    ColDesc* dcd = nullptr;
    Item *dA = nullptr, *dB = nullptr;
    GenA* dgen = nullptr;
    int64_t* dvrow = nullptr;
    try {
        dU = upload(h.U);
        dV = upload(h.V);
        if (!builtin) {
            h.ensure_dense_payload();
            dD = upload(h.D);
        } else {
            dxt = upload(h.xt_copy);
            dxs = upload(h.xs_copy);
        }
        dcd = upload(cdesc);
        dA = upload(itemsA);
        dB = upload(gensB);
        dgen = upload(gensA);
        dvrow = upload(vrow);
        alloc_panel();
        op->colidx = upload(colidx);
        op->ncol = static_cast<int64_t>(colidx.size());
        const int kid = h.src.kernel_id;
        auto gen = [&](auto tag) {
            using TS = decltype(tag);
            TS* P = static_cast<TS*>(op->panel);
            if (!gensB.empty())
                hipLaunchKernelGGL(k_gen_leaf<TS>, dim3(gensB.size()), dim3(256), 0, 0, dB, P, dcd,
                                   op->tmap0, dxt, dxs, dU, dD, kid);
            if (!itemsA.empty())
                hipLaunchKernelGGL(k_gen_far<TS>, dim3(itemsA.size()), dim3(256), 0, 0, dA, dgen, P,
                                   dvrow, dV);
        };
        if (storage == HMX_F64) gen(double{});
        else if (storage == HMX_F32) gen(float{});
        else gen(bf16s{});
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipDeviceSynchronize());
    } catch (...) {
        for (void* p : {(void*)dU, (void*)dV, (void*)dD, (void*)dxt, (void*)dxs, (void*)dcd,
                        (void*)dA, (void*)dB, (void*)dgen, (void*)dvrow})
            if (p) (void)hipFree(p);
        device_destroy(op.release());
        throw;
    }
    for (void* p : {(void*)dU, (void*)dV, (void*)dD, (void*)dxt, (void*)dxs, (void*)dcd,
                    (void*)dgen, (void*)dvrow, (void*)dA, (void*)dB})
        if (p) (void)hipFree(p);

    // HMX_LEAF_PIECES: target piece count of the split (0 keeps every leaf item whole)
    const char* pieces_env = std::getenv("HMX_LEAF_PIECES");
    const int64_t pieces = pieces_env ? std::atoll(pieces_env) : kLeafPieces;
    int64_t leaf_bytes = 0;
    for (const PairItem& it : itemsB) leaf_bytes += leaf_item_work(it);
    std::vector<RowSrc> src(h.m);
    const size_t whole = itemsB.size();
    const std::vector<PairItem> uncut = itemsB;
    op->nlrows = split_leaf_items(itemsB, TK, pieces > 0 ? leaf_piece_bytes(leaf_bytes, pieces) : 0, src);
    {
        // the finer pieces of a smaller operator must not push a product past the
        // static scratch of hmx_matvec_noalloc
        std::vector<PairItem> coarse = uncut;
        std::vector<RowSrc> csrc(h.m);
        const int64_t fine_rows = op->nlrows;
        const int64_t rows = split_leaf_items(
            coarse, TK, pieces > 0 ? std::max(leaf_bytes / pieces, kMiB) : 0, csrc);
        const size_t limit = noalloc_limit();
        bool refused = false;
        for (int W : {1, 4, 16}) {
            op->nlrows = fine_rows;
            const bool fine_fits = noalloc_plan(*op, W).total <= limit;
            op->nlrows = rows;
            refused = refused || (!fine_fits && noalloc_plan(*op, W).total <= limit);
        }
        if (refused) {
            itemsB.swap(coarse);
            src.swap(csrc);
        } else {
            op->nlrows = fine_rows;
        }
    }
    op->direct = itemsB.size() == whole && h.m <= kDirectRows;
    {
        std::vector<RowSrc> by_row(h.m);  // permuted -> original target rows
        for (int64_t i = 0; i < h.m; i++) by_row[tmap0[i]] = src[i];
        op->rowsrc = upload(by_row);
    }
    op->hItemsA = itemsF;  // tree order, for batched operators
    op->hItemsB = itemsB;
    op->hGroups = groups;
    order_far_items(itemsF);
    const char* order_env = std::getenv("HMX_ITEM_ORDER");
    order_leaf_items(itemsB, order_env ? order_env : "xcd");
    op->itemsA = upload(itemsF);
    op->nA = static_cast<int64_t>(itemsF.size());
    op->itemsB = upload(itemsB);
    op->nB = static_cast<int64_t>(itemsB.size());
    op->groups = upload(groups);
    op->nG = static_cast<int64_t>(groups.size());
    if (std::getenv("HMX_VERBOSE"))
        std::fprintf(stderr, "[hmx] storage %d device build: plan %.2f s, total %.2f s\n", storage,
                     t_plan, since());
    h.dev[storage].reset(op.release());
}

// ---- product ---------------------------------------------------------------------
namespace {

// Streams that keep product scratch per operator (HMX_SCRATCH_STREAMS, default
// 8).  A product on a further stream first frees the scratch of the least
// recently used one, after a device synchronisation: that stream may have
// been destroyed since, so it is not synchronised by its handle.
size_t scratch_stream_limit() {
    const char* e = std::getenv("HMX_SCRATCH_STREAMS");
    const long v = e ? std::atol(e) : 8;
    return static_cast<size_t>(std::max(1L, v));
}

void free_scratch(Scratch& sc) {
    for (auto& w : sc.w)
        if (w.S) HIPCHECK(hipFree(w.S));
    sc = Scratch{};
}

// The scratch of `width` columns in a stream's slots: its own, or (MFMA passes) part of a
// wider one, whose three arrays are large enough.  The zero rows of every width start
// at the same address, so they are cleared once and no pass writes them: the narrower S
// ends with them and begins further back.  A stream that has run a wide product can
// therefore run, and record into a graph, any narrower one without an allocation.
ScratchW held_scratch(const DeviceOp& op, const Scratch& sc, int W) {
    for (int w = W; w <= kMaxWidth && (w == W || W >= 16); w += 16) {
        ScratchW s = sc.w[w_slot(w)];
        if (!s.S) continue;
        s.S = static_cast<char*>(s.S) + staging(op, w).zero_begin - staging(op, W).zero_begin;
        return s;
    }
    return ScratchW{};
}

// The scratch entry of a stream (op.mu is held), made on its first call.
Scratch& stream_scratch(DeviceOp& op, hipStream_t stream) {
    auto it = op.scratch.find(static_cast<void*>(stream));
    if (it == op.scratch.end()) {
        const size_t limit = scratch_stream_limit();
        while (op.scratch.size() >= limit) {
            auto lru = op.scratch.begin();
            for (auto j = op.scratch.begin(); j != op.scratch.end(); ++j)
                if (j->second.last_use < lru->second.last_use) lru = j;
            HIPCHECK(hipDeviceSynchronize());
            free_scratch(lru->second);
            op.scratch.erase(lru);
        }
        it = op.scratch.emplace(static_cast<void*>(stream), Scratch{}).first;
    }
    it->second.last_use = ++op.use_clock;
    return it->second;
}

void keep_scratch(const DeviceOp& op, Scratch& sc, int W, const ScratchW& s) {
    const size_t bytes = scratch_sizes(op, W).total();
    sc.w[w_slot(W)] = s;
    sc.bytes += bytes;
    if (std::getenv("HMX_VERBOSE"))
        std::fprintf(stderr, "[hmx] storage %d W %d source/T rows %p, partials %p (%zu bytes)\n",
                     op.storage, W, s.S, s.P, bytes);
}

// Per-stream scratch of one pass width, allocated on the stream's first call:
// in one allocation.
ScratchW get_scratch(DeviceOp& op, hipStream_t stream, int W) {
    std::lock_guard<std::mutex> g(op.mu);
    Scratch& sc = stream_scratch(op, stream);
    ScratchW s = held_scratch(op, sc, W);
    if (!s.S) {
        HIPCHECK(alloc_scratch(op, W, stream, s));
        keep_scratch(op, sc, W, s);
    }
    return s;
}

// Whether a product reads X in place: one right-hand side of the accumulation type, a
// small operator, and a Y that does not overlap X (the leaf kernel writes Y while
// others still read X).
template <typename TS, int W, typename TIO>
bool reads_x_in_place(const DeviceOp& op, const void* X, const void* Y) {
    if (W != 1 || !op.colx || !std::is_same<TIO, typename Store<TS>::acc>::value) return false;
    const uintptr_t x = reinterpret_cast<uintptr_t>(X), y = reinterpret_cast<uintptr_t>(Y);
    return x + op.n * sizeof(TIO) <= y || y + op.m * sizeof(TIO) <= x;
}

template <typename TS, int W, typename TIO>
void run(DeviceOp& op, const void* X, int64_t ldx, void* Y, int64_t ldy, int nrhs, hipStream_t st) {
    const ScratchW sc = get_scratch(op, st, W);
    InstDesc one{};
    one.panel = op.panel;
    one.colidx = op.colidx;
    one.S = sc.S;
    one.partial = sc.P;
    one.lrows = sc.LP;
    one.rowsrc = op.rowsrc;
    one.direct = op.direct;
    one.io64 = std::is_same<TIO, double>::value;
    one.m = op.m;
    one.tmap0 = op.tmap0;
    one.inv_smap = op.inv_smap;
    one.smap0 = op.smap0;
    one.colx = op.colx;
    one.X = X;
    one.Y = Y;
    one.ldx = ldx;
    one.ldy = ldy;
    one.n = op.n;
    one.s0 = op.s0;
    const StagingLayout lay = staging(op, W);
    one.s_rows = static_cast<uint32_t>(lay.rows);
    one.nrhs = nrhs;
    StageArrays A;
    A.itemsA = op.itemsA;
    A.nA = op.nA;
    A.groups = op.groups;
    A.nG = op.nG;
    A.itemsB = op.itemsB;
    A.nB = op.nB;
    A.gather_n = op.n;
    A.gather_insts = 1;
    A.wide = wide_staging(lay);
    A.xdir = !A.wide && reads_x_in_place<TS, W, TIO>(op, X, Y);
    A.out_m = op.direct ? 0 : op.m;
    for (int rhs0 = 0; rhs0 < nrhs; rhs0 += W) {
        one.rhs0 = rhs0;
        launch_stages<TS, W, TIO, false>(A, one, nullptr, st, &op);
    }
    HIPCHECK(hipGetLastError());
}

// RHS width of a pass: one column -> VALU GEMV, up to 4 -> VALU 4-wide, more ->
// MFMA passes of 16, 32 or 48 columns.  A pass reads the whole matrix, so the
// fewest passes of at most 48 columns are taken, and of those the narrowest that
// hold nrhs.  At N = 16,384 a pass of 16 / 32 / 48 takes 311 / 372 / 444 us (FP64),
// 160 / 194 / 238 us (FP32) and 96 / 112 / 144 us (BF16): every wider pass beats the
// narrow ones that it stands for, from 17 columns on (370, 193 and 108 us with 17,
// against 621, 321 and 192 us for two passes of 16).
int pass_width(int nrhs) {
    if (nrhs <= 4) return nrhs == 1 ? 1 : 4;
    const int passes = (nrhs + 47) / 48;
    return 16 * ((nrhs + 16 * passes - 1) / (16 * passes));
}

// Bytes that the scratch of a wide pass may take: half of the device memory that is
// free, so that it does not starve the caller's own allocations, or
// HMX_WIDE_SCRATCH_LIMIT where that is less.
size_t wide_scratch_limit() {
    size_t free_b = 0, total_b = 0;
    HIPCHECK(hipMemGetInfo(&free_b, &total_b));
    size_t limit = free_b / 2;
    if (const char* e = std::getenv("HMX_WIDE_SCRATCH_LIMIT")) {
        const long long v = std::atoll(e);
        if (v >= 0) limit = std::min(limit, static_cast<size_t>(v));
    }
    return limit;
}

// Whether a wide pass (32 or 48 columns) can have its scratch, two or three times that
// of 16 columns.  A stream that is being captured gets no new scratch, and where the
// allocation fails or passes the limit above the product runs in narrower passes (the
// same bits).  A lack of memory is remembered until the stream's scratch is released,
// so that not every product tries again.
bool wide_scratch(DeviceOp& op, hipStream_t st, int W) {
    std::lock_guard<std::mutex> g(op.mu);
    auto it = op.scratch.find(static_cast<void*>(st));
    if (it != op.scratch.end()) {
        if (held_scratch(op, it->second, W).S) return true;
        if (W >= it->second.refused) return false;
    }
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    Scratch& sc = stream_scratch(op, st);
    hipError_t e = hipErrorOutOfMemory;
    ScratchW s;
    if (scratch_sizes(op, W).total() <= wide_scratch_limit()) e = alloc_scratch(op, W, st, s);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        if (e == hipErrorOutOfMemory) sc.refused = W;
        return false;
    }
    keep_scratch(op, sc, W, s);
    return true;
}

template <typename TS, typename TIO>
void run_w(DeviceOp& op, const void* X, int64_t ldx, void* Y, int64_t ldy, int nrhs, hipStream_t st) {
    int W = pass_width(nrhs);
    while (W > 16 && !wide_scratch(op, st, W)) W -= 16;
    if (W == 1)
        run<TS, 1, TIO>(op, X, ldx, Y, ldy, nrhs, st);
    else if (W == 4)
        run<TS, 4, TIO>(op, X, ldx, Y, ldy, nrhs, st);
    else if (W == 48)
        run<TS, 48, TIO>(op, X, ldx, Y, ldy, nrhs, st);
    else if (W == 32)
        run<TS, 32, TIO>(op, X, ldx, Y, ldy, nrhs, st);
    else
        run<TS, 16, TIO>(op, X, ldx, Y, ldy, nrhs, st);
}

template <typename TS>
void run_io(DeviceOp& op, const void* X, int64_t ldx, void* Y, int64_t ldy, int nrhs, int io,
            hipStream_t st) {
    if (io == HMX_F64)
        run_w<TS, double>(op, X, ldx, Y, ldy, nrhs, st);
    else
        run_w<TS, float>(op, X, ldx, Y, ldy, nrhs, st);
}

}  // namespace

void device_matvec(HMatrix& h, int storage, const void* X, int64_t ldx, void* Y, int64_t ldy,
                   int nrhs, int io_dtype, void* stream) {
    if (storage < 0 || storage > 2 || !h.dev[storage])
        throw Error(HMX_ERR_STATE, "storage precision not materialised on the device");
    if (io_dtype != HMX_F64 && io_dtype != HMX_F32)
        throw Error(HMX_ERR_ARG, "io_dtype must be HMX_F64 or HMX_F32");
    if (nrhs <= 0) return;
    if (!X || !Y) throw Error(HMX_ERR_ARG, "null X or Y");
    if (ldx < h.n || ldy < h.m) throw Error(HMX_ERR_ARG, "leading dimension smaller than the size");
    DeviceOp& op = *h.dev[storage];
    DeviceGuard guard(op.device);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (storage == HMX_F64)
        run_io<double>(op, X, ldx, Y, ldy, nrhs, io_dtype, st);
    else if (storage == HMX_F32)
        run_io<float>(op, X, ldx, Y, ldy, nrhs, io_dtype, st);
    else
        run_io<bf16s>(op, X, ldx, Y, ldy, nrhs, io_dtype, st);
}

}  // namespace hmx

// ---- product without device allocation -----------------------------------------
// Scratch of hmx_matvec_noalloc: one array per GPU, allocated with the code
// object when the library's kernels are first loaded on that device and held
// until the process ends.  The host-side name is only a symbol: its device
// address is looked up once per device with hipGetSymbolAddress and that
// address is what the kernels receive.
static __device__ __align__(256) unsigned char scratch[hmx::kNoAllocScratchBytes];

namespace hmx {

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_base[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up on the first
// call per device and kept).
void* noalloc_base(int device) {
    if (device < 0 || device >= kMaxDevices) throw Error(HMX_ERR_ARG, "invalid device ordinal");
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    if (!g_noalloc_base[device]) {
        void* p = nullptr;
        HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) throw Error(HMX_ERR_HIP, "hipGetSymbolAddress returned a null scratch address");
        g_noalloc_base[device] = p;
    }
    return g_noalloc_base[device];
}

template <typename TS, int W, typename TIO>
void run_noalloc(DeviceOp& op, const void* X, int64_t ldx, void* Y, int64_t ldy, int nrhs,
                 hipStream_t st, unsigned char* base, const NoAllocPlan& pl) {
    InstDesc one{};
    one.panel = op.panel;
    one.colidx = op.colidx;
    one.S = base + pl.s;
    one.partial = base + pl.p;
    one.lrows = base + pl.lp;
    one.rowsrc = op.rowsrc;
    one.direct = op.direct;
    one.io64 = std::is_same<TIO, double>::value;
    one.m = op.m;
    one.tmap0 = op.tmap0;
    one.inv_smap = op.inv_smap;
    one.smap0 = op.smap0;
    one.colx = op.colx;
    one.X = X;
    one.Y = Y;
    one.ldx = ldx;
    one.ldy = ldy;
    const StagingLayout lay = staging(op, W);
    one.n = op.n;
    one.s0 = op.s0;
    one.s_rows = static_cast<uint32_t>(lay.rows);
    one.nrhs = nrhs;
    zero_staging_tail(base + pl.s, lay, st);
    StageArrays A;
    A.itemsA = op.itemsA;
    A.nA = op.nA;
    A.groups = op.groups;
    A.nG = op.nG;
    A.itemsB = op.itemsB;
    A.nB = op.nB;
    A.gather_n = op.n;
    A.gather_insts = 1;
    A.wide = wide_staging(lay);
    A.xdir = !A.wide && reads_x_in_place<TS, W, TIO>(op, X, Y);
    A.out_m = op.direct ? 0 : op.m;
    for (int rhs0 = 0; rhs0 < nrhs; rhs0 += W) {
        one.rhs0 = rhs0;
        launch_stages<TS, W, TIO, false>(A, one, nullptr, st, nullptr);
    }
    HIPCHECK(hipGetLastError());
}

template <typename TS, typename TIO>
void noalloc_w(DeviceOp& op, const void* X, int64_t ldx, void* Y, int64_t ldy, int nrhs,
               hipStream_t st, size_t limit) {
    int W = pass_width(nrhs);
    if (W > 16 && noalloc_plan(op, W).total > limit) W = 16;
    const NoAllocPlan pl = noalloc_plan(op, W);
    if (pl.total > limit)
        throw Error(HMX_ERR_UNSUPPORTED,
                    "hmx_matvec_noalloc: this product needs " + std::to_string(pl.total) +
                        " bytes of scratch; the static scratch array holds " +
                        std::to_string(limit) + " (use hmx_matvec)");
    unsigned char* base = static_cast<unsigned char*>(noalloc_base(op.device));
    if (W == 1)
        run_noalloc<TS, 1, TIO>(op, X, ldx, Y, ldy, nrhs, st, base, pl);
    else if (W == 4)
        run_noalloc<TS, 4, TIO>(op, X, ldx, Y, ldy, nrhs, st, base, pl);
    else if (W == 48)
        run_noalloc<TS, 48, TIO>(op, X, ldx, Y, ldy, nrhs, st, base, pl);
    else if (W == 32)
        run_noalloc<TS, 32, TIO>(op, X, ldx, Y, ldy, nrhs, st, base, pl);
    else
        run_noalloc<TS, 16, TIO>(op, X, ldx, Y, ldy, nrhs, st, base, pl);
}

}  // namespace

void device_matvec_noalloc(HMatrix& h, int storage, const void* X, int64_t ldx, void* Y,
                           int64_t ldy, int nrhs, int io_dtype, void* stream) {
    if (storage < 0 || storage > 2 || !h.dev[storage])
        throw Error(HMX_ERR_STATE, "storage precision not materialised on the device");
    if (io_dtype != HMX_F64 && io_dtype != HMX_F32)
        throw Error(HMX_ERR_ARG, "io_dtype must be HMX_F64 or HMX_F32");
    if (nrhs <= 0) return;
    if (!X || !Y) throw Error(HMX_ERR_ARG, "null X or Y");
    if (ldx < h.n || ldy < h.m) throw Error(HMX_ERR_ARG, "leading dimension smaller than the size");
    const size_t limit = noalloc_limit();
    DeviceOp& op = *h.dev[storage];
    DeviceGuard guard(op.device);
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto io = [&](auto ts) {
        using TS = decltype(ts);
        if (io_dtype == HMX_F64)
            noalloc_w<TS, double>(op, X, ldx, Y, ldy, nrhs, st, limit);
        else
            noalloc_w<TS, float>(op, X, ldx, Y, ldy, nrhs, st, limit);
    };
    if (storage == HMX_F64)
        io(double{});
    else if (storage == HMX_F32)
        io(float{});
    else
        io(bf16s{});
}

namespace {
std::mutex g_host_product_mu;  // serialises the lazy FP64 materialisation

struct DeviceBuffer {
    void* p = nullptr;
    explicit DeviceBuffer(size_t bytes) { HIPCHECK(hipMalloc(&p, bytes ? bytes : 1)); }
    ~DeviceBuffer() {
        if (p) (void)hipFree(p);
    }
};
}  // namespace

void device_matvec_host(HMatrix& h, const double* x, int64_t ldx, double* y, int64_t ldy,
                        int nrhs) {
    if (nrhs <= 0) return;
    if (!x || !y) throw Error(HMX_ERR_ARG, "null x or y");
    if (ldx < h.n || ldy < h.m) throw Error(HMX_ERR_ARG, "leading dimension smaller than the size");
    {
        std::lock_guard<std::mutex> g(g_host_product_mu);
        if (!h.dev[HMX_F64]) device_build(h, HMX_F64);
    }
    DeviceGuard guard(h.dev[HMX_F64]->device);
    DeviceBuffer dx(static_cast<size_t>(h.n) * nrhs * 8), dy(static_cast<size_t>(h.m) * nrhs * 8);
    HIPCHECK(hipMemcpy2D(dx.p, static_cast<size_t>(h.n) * 8, x, static_cast<size_t>(ldx) * 8,
                         static_cast<size_t>(h.n) * 8, static_cast<size_t>(nrhs),
                         hipMemcpyHostToDevice));
    device_matvec(h, HMX_F64, dx.p, h.n, dy.p, h.m, nrhs, HMX_F64, nullptr);
    // stream-ordered after the product on the null stream; returns when y is filled
    HIPCHECK(hipMemcpy2D(y, static_cast<size_t>(ldy) * 8, dy.p, static_cast<size_t>(h.m) * 8,
                         static_cast<size_t>(h.m) * 8, static_cast<size_t>(nrhs),
                         hipMemcpyDeviceToHost));
}

int64_t device_release_scratch(HMatrix& h, void* stream, bool all_streams) {
    int64_t freed = 0;
    for (auto& d : h.dev) {
        if (!d) continue;
        DeviceGuard guard(d->device);
        std::lock_guard<std::mutex> g(d->mu);
        for (auto it = d->scratch.begin(); it != d->scratch.end();) {
            if (!all_streams && it->first != stream) {
                ++it;
                continue;
            }
            // the stream's products may still be running
            HIPCHECK(hipStreamSynchronize(static_cast<hipStream_t>(it->first)));
            for (auto& w : it->second.w)
                if (w.S) freed++;
            free_scratch(it->second);
            it = d->scratch.erase(it);
        }
    }
    return freed;
}

void device_scratch_usage(const HMatrix& h, int64_t* bytes, int64_t* entries) {
    int64_t b = 0, e = 0;
    for (const auto& d : h.dev) {
        if (!d) continue;
        std::lock_guard<std::mutex> g(d->mu);
        for (const auto& kv : d->scratch) {
            b += static_cast<int64_t>(kv.second.bytes);
            e++;
        }
    }
    *bytes = b;
    *entries = e;
}

void device_profile_enable(HMatrix& h, bool on) {
    for (auto& d : h.dev)
        if (d) d->profiling = on;
}

void device_profile_read(HMatrix& h, double* ms, int64_t* launches, bool reset) {
    for (int k = 0; k < 4; k++) {
        ms[k] = 0;
        launches[k] = 0;
    }
    for (auto& d : h.dev) {
        if (!d) continue;
        DeviceGuard guard(d->device);
        std::lock_guard<std::mutex> g(d->mu);
        for (int k = 0; k < 4; k++) {
            for (auto& pr : d->ev[k]) {
                HIPCHECK(hipEventSynchronize(pr.second));
                float t = 0;
                HIPCHECK(hipEventElapsedTime(&t, pr.first, pr.second));
                d->ms[k] += t;
                d->launches[k] += 1;
                (void)hipEventDestroy(pr.first);
                (void)hipEventDestroy(pr.second);
            }
            d->ev[k].clear();
            ms[k] += d->ms[k];
            launches[k] += d->launches[k];
            if (reset) {
                d->ms[k] = 0;
                d->launches[k] = 0;
            }
        }
    }
}

}  // namespace hmx
