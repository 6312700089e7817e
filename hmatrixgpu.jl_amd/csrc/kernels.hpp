// kernels.hpp -- gfx950 device types and kernels of the H-matrix product and
// of the panel generation.  Included by device.hip (one H-matrix per launch) and
// batch.hip (many H-matrices per launch).  The layout and the stages are
// described in device.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "hmx_host.hpp"

namespace hmx {

#define HIPCHECK(expr)                                                                       \
    do {                                                                                     \
        hipError_t _e = (expr);                                                              \
        if (_e != hipSuccess)                                                                \
            throw ::hmx::Error(HMX_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct bf16s {
    uint16_t u;
};

// One panel work item (rows <= 64).
struct Item {
    int64_t data_off;  // element offset of the panel in the storage array
    int64_t col_off;   // leaf panels: offset into colidx; far-field: first S row
    int64_t out_off;   // leaf panels: first permuted target row; far-field: output row
    int32_t rows;
    int32_t ktiles;
    int32_t ncols;     // far-field generation: valid columns of the chunk
    int32_t inst;      // instance (H-matrix) index in a batched launch
};

// Leaf work item: one or two consecutive row groups (<= 64 rows each) of the
// target order.  The columns both row groups need (blocks whose row range
// covers both) form the shared segment, over one range of column indices; the
// remaining columns of each row group form its private segment.  A row group's
// panel holds its shared and then its private k-tiles back to back, so that one
// pipeline walks both.  A single row group (rows[1] == 0) has only a private
// part.
struct PairItem {
    int64_t out_off[2];  // first permuted target row of each row group
    int64_t data[2];     // panel of each row group: shared, then private k-tiles
    int64_t sh_col;      // colidx offset of the shared columns
    int64_t pr_col[2];   // colidx offset of each private part
    int32_t rows[2];
    int32_t sh_kt;       // k-tiles of the shared segment
    int32_t pr_kt[2];    // k-tiles of each private part
    int32_t inst;        // instance (H-matrix) index in a batched launch
    int64_t part;        // first leaf-result row of this item (or k-range piece of one)
};

// Where the results of one target row lie: nparts leaf-result rows (one per
// k-range piece of its leaf item), from `base`, `stride` rows apart.
struct RowSrc {
    uint32_t base;
    int16_t nparts;
    int16_t stride;
};

struct ReduceGroup {
    int64_t pbase;  // first partial row
    int64_t tbase;  // first T row (S row = s0 + n + tbase)
    int32_t rows;
    int32_t nch;
    int32_t inst;
    int32_t pad;
};

// Per-instance device state of one product launch: the H-matrix operator's
// arrays, its per-stream scratch and the call's X / Y.  Passed by value for a
// single H-matrix, read from a device table for a batch of them.
struct InstDesc {
    const void* panel;
    const int32_t* colidx;
    void* S;                 // source rows from s0: X permuted, then T, then a zero row
    void* partial;           // far-field column-chunk partial sums
    void* lrows;             // leaf results: rows of W, one set per piece of a leaf item
    const RowSrc* rowsrc;    // per original target row: its leaf-result rows
    int64_t m;               // target rows
    const int32_t* tmap0;    // permuted target row -> 0-based original row
    const int32_t* inv_smap; // 0-based original source row -> permuted row
    const int32_t* smap0;    // permuted source row -> 0-based original row
    const int32_t* colx;     // colidx with the X columns by original row (XDIR), or null
    const void* X;
    void* Y;
    int64_t ldx, ldy;
    int64_t n;               // source rows (X rows of S, before T)
    int64_t s0;              // first X row of S (rows before it are unused)
    uint32_t s_rows;         // rows of S (each W elements)
    int32_t nrhs;            // right-hand sides of the call
    int32_t rhs0;            // first right-hand side of this pass
    int16_t io64;            // X and Y are FP64 (else FP32)
    int16_t direct;          // the leaf kernel writes Y itself
};

// ---- element conversions ---------------------------------------------------
__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return static_cast<uint16_t>(u >> 16);
}
__device__ inline float bf2f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

template <typename T>
__device__ inline T from_double(double v);
template <>
__device__ inline double from_double<double>(double v) { return v; }
template <>
__device__ inline float from_double<float>(double v) { return static_cast<float>(v); }
template <>
__device__ inline bf16s from_double<bf16s>(double v) { return bf16s{f2bf(static_cast<float>(v))}; }

template <typename T>
__device__ inline T from_float(float v);
template <>
__device__ inline double from_float<double>(float v) { return v; }
template <>
__device__ inline float from_float<float>(float v) { return v; }
template <>
__device__ inline bf16s from_float<bf16s>(float v) { return bf16s{f2bf(v)}; }

// ---- storage traits ----------------------------------------------------------
// TK: columns per k-tile (64 bytes per row), EPL: elements per lane chunk.
template <typename TS>
struct Store;
template <>
struct Store<double> {
    static constexpr int TK = 8, EPL = 2;
    using acc = double;
};
template <>
struct Store<float> {
    static constexpr int TK = 16, EPL = 4;
    using acc = float;
};
template <>
struct Store<bf16s> {
    static constexpr int TK = 32, EPL = 8;
    using acc = float;
};
// Right-hand sides of a pass: 1 or 4 run on the VALU, multiples of 16 on MFMA as
// kSlices<W> 16-column slices that share each load of the matrix.
template <int W>
constexpr bool kMfma = W >= 16;
template <int W>
constexpr int kSlices = W >= 16 ? W / 16 : 1;
// B-operand (S) element type: MFMA -> its operand type; VALU -> the accumulation type
template <typename TS, int W>
struct SType {
    using type = typename std::conditional<kMfma<W>, TS, typename Store<TS>::acc>::type;
};

constexpr int kWaves = 4;  // waves per workgroup in the panel kernels
constexpr int kPipe = 3;   // k-tiles in flight per wave (panel_accum)
// Exceptions, each measured on the MI355X with the B tiles in LDS: the BF16 far-field
// kernel keeps two (its panels are a few k-tiles long); the leaf kernels with one right-hand
// side and the FP64 ones with 16 keep four (five: FP64 with one 1% faster at N = 50,000 and
// 7% slower at 4,096); the FP32 and BF16 leaf kernels with 16 keep six (N = 100,000: FP32
// 2131 -> 2118 us against five, BF16 1090 -> 1082 against four; seven and eight the same
// or slower); the FP32 and FP64 far kernels with 16 four.  The 4-wide kernels spill from
// five on (FP32, N = 20,011: 188 -> 263 us).  Two and three slices keep three.  The panel
// kernels ask for two waves per SIMD: the compiler then keeps the accumulators in VGPRs
// instead of copying them to and from AGPRs, and the FP64 kernels with three slices fit
// (N = 16,384 with 48 right-hand sides 506 -> 444 us; two k-tiles in flight instead:
// 481 us).  Asking for four makes the VALU kernels spill.
template <typename TS, bool LEAF, int W>
constexpr int pipe_depth() {
    if (!LEAF && std::is_same<TS, bf16s>::value) return 2;
    if (W > 16) return kPipe;
    if (LEAF && W == 16 && !std::is_same<TS, double>::value) return 6;
    if (LEAF && W != 4) return 4;
    if (!LEAF && W == 16) return 4;
    return kPipe;
}
// B tile of one wave and slice: the k-tile's TK rows of S, brought in by one load
// instruction (lane L: LB bytes, chunk L % LPR of row L / LPR) and handed to the lanes
// that need them through LDS.  STRIDE pads a row so that the lane groups of a read hit
// distinct banks: FP32 on MFMA 64 + 16 bytes, FP64 128 + 64, BF16 32 + 8; the VALU
// paths read whole rows, the same one in 16 lanes, and need no padding.  The texture
// unit's load instructions bound these kernels next to HBM: before, only FP32 on MFMA
// went this way, and the others loaded every operand for every lane.  us per product,
// before -> now: N = 20,011 with four right-hand sides FP32 213 -> 188, BF16 163 -> 123,
// FP64 391 -> 350; with one BF16 114 -> 98; N = 4,096 FP64 with one 45 -> 41;
// N = 50,000 BF16 with 16 429 -> 410.
template <typename TS, int W>
struct BTile {
    using s_t = typename SType<TS, W>::type;
    static constexpr int RB = (kMfma<W> ? 16 : W) * static_cast<int>(sizeof(s_t));
    static constexpr int LB = RB < 16 ? RB : 16, LPR = RB / LB;
    static constexpr int LANES = Store<TS>::TK * LPR;
    static constexpr int STRIDE =
        !kMfma<W> ? RB : std::is_same<TS, float>::value ? 80 : std::is_same<TS, double>::value ? 192 : 40;
    static constexpr int BYTES = Store<TS>::TK * STRIDE;
    static_assert(LANES <= 64, "one load per lane");
    // the lane's part of a row, as loaded
    using part_t = typename std::conditional<
        LB == 16, u32x4, typename std::conditional<LB == 8, uint64_t, uint32_t>::type>::type;
};

// ---- the panel kernel ----------------------------------------------------------
// Buffer resources (raw, stride 0): loads past num_records return 0, which masks
// the absent rows of a partial row tile, the padding of the last k-tile and the
// prefetch past the end of a panel without branches.
constexpr int kRsrcWord3 = 0x00020000;  // gfx9-family raw buffer descriptor
// Cache policy of the streamed panel loads: non-temporal, so that the matrix
// stream (read once per product) does not evict the reused source / T rows
// from L2 (measured: 3-10% faster than the default policy at N = 262,144).
constexpr int kPanelPolicy = 2;
constexpr uint32_t kOOB = 0xffffffffu;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes),
                                             kRsrcWord3);
}

// One S row of W values for the VALU paths (W = 1 or 4).
template <typename T, int W>
struct SRow {
    T v[W];
};
// One S (or output) row as a unit of store: W elements, aligned to its size (at most 16
// bytes), so that it is written with row-sized vector stores.
template <typename T, int W>
struct alignas(sizeof(T) * W >= 16 ? 16 : sizeof(T) * W) SRowOut {
    T v[W];
};

// One wave's share of a panel: k-tiles kt0, kt0 + kstep, ... of a `rows` x
// (ktiles * TK) panel at pdata.  B rows come from S: through the column index
// array (LEAF: from colidx + col_off for the first sh_kt k-tiles, from
// colidx + pr_off for the rest) or as the contiguous rows col_off + k masked
// beyond ncols.  The
// accumulated results are handed to emit(row, col, value), row < 64, col < W.
// XDIR (one right-hand side, X of the accumulation type, a small operator): X is read
// from the caller's vector instead of S.  A column index below n then is a row of X
// (LEAF: from the index array; far field: col_off addresses smap0), any other one a row
// of S; each is one load that the other's range check turns into zeros.
// W = 16, 32 and 48 run on MFMA (16 right-hand sides as the N dimension of each of NB
// slices); W = 1 and 4 run on the VALU, lane (row li, k-chunk lg).  CP is the cache
// policy of the streamed A loads.
// Accumulator of one wave for one 16-row tile and slice: MFMA C/D registers, or
// per-lane partial sums (W = 1, 4); acc[rt * NB + slice].
template <typename TS, int W>
using PanelAcc = typename std::conditional<
    kMfma<W>,
    typename std::conditional<std::is_same<typename Store<TS>::acc, double>::value, f64x4,
                              f32x4>::type,
    SRow<typename Store<TS>::acc, W>>::type;

template <typename TS, int W, bool LEAF, int NRT, int CP, bool WIDE, bool XDIR = false>
__device__ __forceinline__ void panel_accum(const TS* pdata, int rows, int ktiles, int64_t col_off,
                                            int ncols, const int32_t* colidx, int sh_kt,
                                            int64_t pr_off,
                                            const typename SType<TS, W>::type* S, uint32_t s_rows,
                                            int kt0, int kstep, int lane, char* btile,
                                            PanelAcc<TS, W>* acc, const void* X = nullptr,
                                            int64_t n = 0) {
    using acc_t = typename Store<TS>::acc;
    using s_t = typename SType<TS, W>::type;
    constexpr int TK = Store<TS>::TK, EPL = Store<TS>::EPL;
    constexpr uint32_t SB = sizeof(s_t), ROWB = W * sizeof(s_t);
    const int li = lane & 15, lg = lane >> 4;
    const uint32_t slab = static_cast<uint32_t>(rows) * 64u;
    const __amdgpu_buffer_rsrc_t Ar = make_rsrc(pdata, slab * ktiles);
    const __amdgpu_buffer_rsrc_t Sr = make_rsrc(S, WIDE ? 0u : s_rows * ROWB);
    // Column indices of both segments, addressed by the k-tile of the whole
    // panel: the private ones from a base moved back by the shared tiles.
    const int32_t* const csh = colidx + (LEAF || XDIR ? col_off : 0);
    const int32_t* const cpr = colidx + (LEAF ? pr_off - static_cast<int64_t>(sh_kt) * TK : 0);
    const __amdgpu_buffer_rsrc_t Csh = make_rsrc(csh, (LEAF ? ktiles * TK : ncols) * 4),
                                 Cpr = LEAF ? make_rsrc(cpr, ktiles * TK * 4) : Csh;
    const __amdgpu_buffer_rsrc_t Xr = make_rsrc(X, static_cast<uint32_t>(n) * ROWB);
    constexpr bool INDEXED = LEAF || XDIR;  // columns come through an index array
    static_assert(!XDIR || (W == 1 && !WIDE), "XDIR: one right-hand side, S below 4 GiB");
    uint32_t aoff[NRT];
    bool aval[NRT];
#pragma unroll
    for (int rt = 0; rt < NRT; rt++) {
        const int rr = min(16, rows - 16 * rt);
        aval[rt] = li < rr;
        aoff[rt] = static_cast<uint32_t>((16 * rt * TK + (rr * lg + li) * EPL) * sizeof(TS));
    }
    constexpr int NB = kSlices<W>;
    const uint32_t bcol = (kMfma<W> ? li : 0) * SB;
    using brow_t = typename std::conditional<kMfma<W>, s_t, SRowOut<s_t, W>>::type;

    // The k-tile's B rows arrive as one load per lane and slice (BTile) instead of one
    // per operand: with four right-hand sides the 16 lanes of a lane group used to load
    // the same rows, 4 KB for 256 B, and held them in registers for every stage.
    using BT = BTile<TS, W>;
    using part_t = typename BT::part_t;
    const int brow = lane / BT::LPR, bpart = lane % BT::LPR;
    const bool bact = lane < BT::LANES;
    struct Stage {
        u32x4 a[NRT];
        part_t b[NB];
    };
    // Column index of the row the lane loads.
    auto load_ix = [&](int kt) {
        const __amdgpu_buffer_rsrc_t Cr = kt < sh_kt ? Csh : Cpr;
        const uint32_t off = bact ? static_cast<uint32_t>((kt * TK + brow) * 4) : kOOB;
        return static_cast<int32_t>(__builtin_amdgcn_raw_buffer_load_b32(Cr, off, 0, 0));
    };
    auto load_stage = [&](int kt, int32_t ix) {
        Stage st;
        const uint32_t base = static_cast<uint32_t>(kt) * slab;
        // A far panel's last k-tile is zero-padded past ncols: a lane whose
        // EPL-column chunk lies wholly in the padding reads nothing (the
        // range check returns the same zeros), which saves those bytes.
        const bool kin = LEAF || kt * TK + lg * EPL < ncols;
#pragma unroll
        for (int rt = 0; rt < NRT; rt++) {
            const uint32_t o = aval[rt] && kin ? base + aoff[rt] : kOOB;
            st.a[rt] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(Ar, o, 0, CP));
        }
        uint32_t row;
        bool ok = bact;
        if constexpr (LEAF) {
            row = static_cast<uint32_t>(ix);
        } else {
            const int k = kt * TK + brow;
            ok = ok && k < ncols;
            row = ok ? static_cast<uint32_t>(col_off + k) : s_rows - 1;
        }
        if constexpr (XDIR) {
            const uint32_t r = static_cast<uint32_t>(LEAF ? row : ix);
            const uint32_t xo = ok && r < static_cast<uint32_t>(n) ? r * ROWB : kOOB;
            const uint32_t so = LEAF && ok && r >= static_cast<uint32_t>(n) ? r * ROWB : kOOB;
            part_t v;
            if constexpr (BT::LB == 8)
                v = __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b64(Xr, xo, 0, 0));
            else
                v = __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b32(Xr, xo, 0, 0));
            if constexpr (LEAF) {  // the one that is out of range reads zeros
                if constexpr (BT::LB == 8)
                    v |= __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b64(Sr, so, 0, 0));
                else
                    v |= __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b32(Sr, so, 0, 0));
            }
            st.b[0] = v;
            return st;
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if constexpr (WIDE) {
                st.b[b] = part_t{};
                if (bact)
                    st.b[b] = *reinterpret_cast<const part_t*>(
                        reinterpret_cast<const char*>(S) + static_cast<uint64_t>(row) * ROWB +
                        b * BT::RB + bpart * BT::LB);
            } else {
                const uint32_t o = ok ? row * ROWB + b * BT::RB + bpart * BT::LB : kOOB;
                if constexpr (BT::LB == 16)
                    st.b[b] = __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b128(Sr, o, 0, 0));
                else if constexpr (BT::LB == 8)
                    st.b[b] = __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b64(Sr, o, 0, 0));
                else
                    st.b[b] = __builtin_bit_cast(part_t, __builtin_amdgcn_raw_buffer_load_b32(Sr, o, 0, 0));
            }
        }
        return st;
    };

    auto compute = [&](const Stage& st) {
        // the lane's B operands: column li of rows lg * EPL + e (MFMA), or those rows
        brow_t bv[NB][EPL];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            // LDS operations of one wave complete in order: the reads see this
            // write, and the next write follows these reads.  The wave barriers
            // keep the compiler from moving them across each other.
            if (BT::LANES == 64 || bact) {
                char* const d = btile + brow * BT::STRIDE + bpart * BT::LB;
                if constexpr (BT::STRIDE % BT::LB == 0) {
                    *reinterpret_cast<part_t*>(d) = st.b[b];
                } else {  // rows aligned to eight bytes only
                    struct Half {
                        uint64_t v[2];
                    };
                    const Half h = __builtin_bit_cast(Half, st.b[b]);
                    reinterpret_cast<uint64_t*>(d)[0] = h.v[0];
                    reinterpret_cast<uint64_t*>(d)[1] = h.v[1];
                }
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int e = 0; e < EPL; e++)
                bv[b][e] = *reinterpret_cast<const brow_t*>(btile + (lg * EPL + e) * BT::STRIDE + bcol);
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int rt = 0; rt < NRT; rt++) {
            const u32x4 raw = st.a[rt];
            PanelAcc<TS, W>* const c = acc + rt * NB;  // the slices' accumulators of this row tile
            if constexpr (kMfma<W>) {
                if constexpr (std::is_same<TS, float>::value) {
                    f32x4 a = __builtin_bit_cast(f32x4, raw);
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int b = 0; b < NB; b++)
                            c[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], bv[b][e], c[b], 0, 0, 0);
                } else if constexpr (std::is_same<TS, double>::value) {
                    typedef double d2 __attribute__((ext_vector_type(2)));
                    d2 a = __builtin_bit_cast(d2, raw);
#pragma unroll
                    for (int e = 0; e < 2; e++)
#pragma unroll
                        for (int b = 0; b < NB; b++)
                            c[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], bv[b][e], c[b], 0, 0, 0);
                } else {
                    bf16x8 a = __builtin_bit_cast(bf16x8, raw);
#pragma unroll
                    for (int b = 0; b < NB; b++) {
                        uint16_t bb[8];
#pragma unroll
                        for (int e = 0; e < 8; e++) bb[e] = bv[b][e].u;
                        bf16x8 bx = __builtin_bit_cast(bf16x8, bb);
                        c[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bx, c[b], 0, 0, 0);
                    }
                }
            } else {
                acc_t av[EPL];
                if constexpr (std::is_same<TS, float>::value) {
                    f32x4 a = __builtin_bit_cast(f32x4, raw);
                    av[0] = a.x; av[1] = a.y; av[2] = a.z; av[3] = a.w;
                } else if constexpr (std::is_same<TS, double>::value) {
                    typedef double d2 __attribute__((ext_vector_type(2)));
                    d2 a = __builtin_bit_cast(d2, raw);
                    av[0] = a.x; av[1] = a.y;
                } else {
                    uint16_t h[8];
                    std::memcpy(h, &raw, 16);
#pragma unroll
                    for (int e = 0; e < 8; e++) av[e] = bf2f(h[e]);
                }
#pragma unroll
                for (int w = 0; w < W; w++) {
                    acc_t s = acc[rt].v[w];
#pragma unroll
                    for (int e = 0; e < EPL; e++) s += av[e] * bv[0][e].v[w];
                    acc[rt].v[w] = s;
                }
            }
        }
    };

    // Software pipeline D = pipe_depth k-tiles deep: D - 1 stages are in
    // flight while one is consumed, and the column indices run two k-tiles
    // ahead of their data.  The loop body is unrolled D times so that every
    // stage index is a constant (no register copies); stage j of an iteration
    // loads k-tile j + D - 1 into the slot consumed at step j - 1, refills the
    // index slot the load two steps later needs, then consumes slot j.  Loads
    // past the end of the panel (kt >= ktiles) fall outside the buffer and
    // return zeros; they are never consumed.  The loop runs over whole
    // groups of D k-tiles and has a single exit, with the 0 .. D - 2
    // remaining k-tiles after it: the accumulators then stay in place across
    // the exit.  (A break inside the unrolled body made the compiler copy
    // just-written FP64 MFMA results at the exit with too few wait states,
    // corrupting their low bits.)
    const int mine = kt0 < ktiles ? (ktiles - kt0 + kstep - 1) / kstep : 0;
    constexpr int D = pipe_depth<TS, LEAF, W>();
    int kt = kt0;
    int32_t ix[D];
    Stage st[D];
    // The prologue issues its loads in the loop's own order (indices, then
    // stages, then the next index), fenced against rescheduling: the wait the
    // compiler puts at the loop header must hold on the entry path as well as
    // on the back edge, and an index load sunk to the end of the prologue
    // would make it wait for every load in flight at each iteration.
#pragma unroll
    for (int d = 0; d < D; d++) {
        ix[d] = 0;
        if constexpr (INDEXED) ix[d] = load_ix(kt + d * kstep);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d + 1 < D; d++) {
        st[d] = load_stage(kt + d * kstep, ix[d]);
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (INDEXED) ix[0] = load_ix(kt + D * kstep);
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
    for (; i + D - 1 < mine; i += D) {
#pragma unroll
        for (int j = 0; j < D; j++) {
            st[(j + D - 1) % D] = load_stage(kt + (j + D - 1) * kstep, ix[(j + D - 1) % D]);
            if constexpr (INDEXED) ix[(j + 1) % D] = load_ix(kt + (j + D + 1) * kstep);
            compute(st[j]);
        }
        kt += D * kstep;
    }
    const int rem = mine - i;
#pragma unroll
    for (int j = 0; j + 1 < D; j++)
        if (j < rem) compute(st[j]);
}

// Hand the accumulated results of slice b (VALU: of all columns) to
// emit(row, col, value), row < 16*nrt, col < min(W, 16).
template <typename TS, int W, typename Emit>
__device__ __forceinline__ void panel_emit(const PanelAcc<TS, W>* acc, int nrt, int b, int lane,
                                           Emit&& emit) {
    using acc_t = typename Store<TS>::acc;
    const int li = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 4; rt++) {
        if (rt >= nrt) break;
        if constexpr (kMfma<W>) {
            // MFMA 16x16 output, column li: f32 accumulators hold rows 4*lg+v of the
            // row tile, the f64 instruction holds rows 4*v+lg.
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = std::is_same<TS, double>::value ? 4 * v + lg : 4 * lg + v;
                emit(16 * rt + row, li, static_cast<acc_t>(acc[rt * kSlices<W> + b][v]));
            }
        } else {
#pragma unroll
            for (int w = 0; w < W; w++) {
                acc_t v = acc[rt].v[w];
                v += __shfl_xor(v, 16);
                v += __shfl_xor(v, 32);
                if (lg == 0) emit(16 * rt + li, w, v);
            }
        }
    }
}

template <typename F>
__device__ __forceinline__ void dispatch_nrt(int rows, F&& f) {
    switch ((rows + 15) >> 4) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    default: f(std::integral_constant<int, 4>{}); break;
    }
}

template <bool BATCH>
__device__ __forceinline__ const InstDesc& inst_of(const InstDesc& one, const InstDesc* insts,
                                                   int idx) {
    if constexpr (BATCH)
        return insts[idx];
    else
        return one;
}

// Leaf item: for a pair of row groups, waves 0-1 own row group 0 and waves 2-3
// row group 1; the two waves of a row group split the k-tiles of its panel (the
// shared, then the private ones), keeping one set of accumulators and one
// pipeline: with a pipeline per segment, every piece of an item paid two fills.  Waves 0 and 2
// (1 and 3) walk the same shared k-tiles at the same time, so each shared B
// row is fetched once per workgroup and served to the second wave from L1.  A
// single row group is split over all four waves.  Partial sums are reduced
// through LDS and written as whole leaf-result rows, which k_finish sums and
// scatters; the items of a small operator, none of them cut, write Y directly.
template <typename TS, int W, int CP, bool BATCH, bool WIDE, bool XDIR = false>
__global__ __launch_bounds__(kWaves * 64, 2) void k_leaf(const PairItem* __restrict__ items,
                                                      const InstDesc one,
                                                      const InstDesc* __restrict__ insts) {
    using acc_t = typename Store<TS>::acc;
    using s_t = typename SType<TS, W>::type;
    const PairItem it = items[blockIdx.x];
    const InstDesc& I = inst_of<BATCH>(one, insts, it.inst);
    // The wave index is uniform across the wave; readfirstlane tells the
    // compiler so, which keeps every per-wave panel pointer and buffer
    // descriptor in SGPRs (a VGPR descriptor wraps each load in a loop).
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const bool pair = it.rows[1] > 0;
    const int g = pair ? wave >> 1 : 0;
    const int kt0 = pair ? (wave & 1) : wave, kstep = pair ? 2 : 4;
    // per-row-group fields by select, not by a runtime index into the item
    const int rows = g ? it.rows[1] : it.rows[0];
    const int64_t data = g ? it.data[1] : it.data[0];
    const int64_t pr_col = g ? it.pr_col[1] : it.pr_col[0];
    const int pr_kt = g ? it.pr_kt[1] : it.pr_kt[0];
    constexpr int NB = kSlices<W>, WS = W / NB;  // columns of a slice
    __shared__ acc_t red[kWaves][64][WS];
    __shared__ alignas(16) char btile[kWaves][BTile<TS, W>::BYTES];
    const TS* panel = static_cast<const TS*>(I.panel);
    const s_t* S = static_cast<const s_t*>(I.S);
    PanelAcc<TS, W> acc[4 * NB];
#pragma unroll
    for (int q = 0; q < 4 * NB; q++) acc[q] = PanelAcc<TS, W>{};
    dispatch_nrt(rows, [&](auto nrt) {
        constexpr int NRT = decltype(nrt)::value;
        panel_accum<TS, W, true, NRT, CP, WIDE, XDIR>(panel + data, rows, it.sh_kt + pr_kt, it.sh_col,
                                                      0, XDIR ? I.colx : I.colidx, it.sh_kt, pr_col, S,
                                                      I.s_rows, kt0, kstep, lane, btile[wave], acc,
                                                      I.X, I.n);
    });
    acc_t* lrows = static_cast<acc_t*>(I.lrows);
    const int r0 = it.rows[0], total = r0 + it.rows[1];
#pragma unroll
    for (int b = 0; b < NB; b++) {  // one slice at a time through LDS
        if (b) __syncthreads();
        panel_emit<TS, W>(acc, (rows + 15) >> 4, b, lane,
                          [&](int row, int j, acc_t v) { red[wave][row][j] = v; });
        __syncthreads();
        for (int t = threadIdx.x; t < total * WS; t += kWaves * 64) {
            const int rr = t / WS, j = t % WS, c = b * WS + j;
            const int gg = rr < r0 ? 0 : 1, r = rr - gg * r0;
            acc_t s;
            if (pair) {
                s = red[2 * gg][r][j] + red[2 * gg + 1][r][j];
            } else {
                s = red[0][r][j];
#pragma unroll
                for (int w = 1; w < kWaves; w++) s += red[w][r][j];
            }
            if (!I.direct) {
                lrows[(it.part + rr) * W + c] = s;
            } else if (I.rhs0 + c < I.nrhs) {
                const int64_t y = I.tmap0[(gg ? it.out_off[1] : it.out_off[0]) + r] +
                                  static_cast<int64_t>(I.rhs0 + c) * I.ldy;
                if (I.io64)
                    static_cast<double*>(I.Y)[y] = static_cast<double>(s);
                else
                    static_cast<float*>(I.Y)[y] = static_cast<float>(s);
            }
        }
    }
}

// Y[i, rhs0 + j] = sum over the pieces of row i, in piece order, for the pass's
// columns (instance = blockIdx.y, slice = blockIdx.z).  One thread per original
// target row and kFinCols<W> columns: the loads of eight pieces are in flight together (the
// sum itself stays in order), and a wave writes 64 consecutive rows of each
// column of Y.
// Bound by the latency of its scattered row reads.  One launch in place of a
// piece sum with one workgroup per leaf item (128 rows in one workgroup, the
// pieces in a serial loop) and an unpermute.
template <int W>
constexpr int kFinCols = W < 4 ? W : 4;
template <int W>
constexpr int kFinRows = kMfma<W> ? 64 : 256;  // target rows of a workgroup

template <typename TS, int W, typename TIO, bool BATCH>
__global__ __launch_bounds__(256) void k_finish(const InstDesc one,
                                                const InstDesc* __restrict__ insts) {
    using acc_t = typename Store<TS>::acc;
    constexpr int C = kFinCols<W>, G = W / C, ROWS = kFinRows<W>;
    const InstDesc& I = inst_of<BATCH>(one, insts, blockIdx.y);
    if (BATCH && I.direct) return;
    const int c0 = (threadIdx.x / ROWS) * C + 16 * blockIdx.z;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * ROWS + threadIdx.x % ROWS;
    if (i >= I.m || I.rhs0 + c0 >= I.nrhs) return;
    const RowSrc rs = I.rowsrc[i];
    using row_t = SRowOut<acc_t, C>;
    const row_t* src = static_cast<const row_t*>(I.lrows) + static_cast<int64_t>(rs.base) * G + c0 / C;
    const int64_t step = static_cast<int64_t>(rs.stride) * G;
    row_t s = src[0];
    for (int p = 1; p < rs.nparts; p += 8) {
        row_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (p + u < rs.nparts) v[u] = src[(p + u) * step];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (p + u < rs.nparts)
#pragma unroll
                for (int j = 0; j < C; j++) s.v[j] += v[u].v[j];
    }
    TIO* Y = static_cast<TIO*>(I.Y);
#pragma unroll
    for (int j = 0; j < C; j++)
        if (I.rhs0 + c0 + j < I.nrhs)
            Y[i + static_cast<int64_t>(I.rhs0 + c0 + j) * I.ldy] = static_cast<TIO>(s.v[j]);
}

// Far-field work item: up to kWaves consecutive 64-row groups of the stacked V
// rows of one source cluster over one column chunk.  With three or four row groups
// wave w owns row group w and walks every k-tile of the chunk; the waves read the same S
// rows (the cluster's X rows), so the B operand is fetched once per workgroup and shared
// through the L1 cache.  With one or two, four or two waves share a row group's
// k-tiles and are summed through LDS: one wave alone walked the whole chunk while the
// others had nothing to do, which set the time of small operators (and of the last
// item of a cluster).  N = 12,000 on a circle, FP64: far kernel 68 -> 24 us; N = 4,000
// FP64 with 40 right-hand sides 21 -> 16 us.
struct FarItem {
    int64_t data_off;  // panel of row group 0; group g at + g*64*ktiles*TK
    int64_t col_off;   // first S row of the chunk
    int64_t out_off;   // output row of row 0 of group 0 (group g: + 64*g)
    int32_t ktiles;
    int32_t ncols;
    int32_t rows_last;  // rows of the last group (the others have 64)
    int16_t nrg;        // number of row groups (<= kWaves)
    int16_t to_T;       // 1: write T rows of S, 0: write partial rows
    int32_t inst;
    int32_t pad;
};

template <typename TS, int W, int CP, bool BATCH, bool WIDE, bool XDIR = false>
__global__ __launch_bounds__(kWaves * 64, 2) void k_far(const FarItem* __restrict__ items,
                                                     const InstDesc one,
                                                     const InstDesc* __restrict__ insts) {
    using acc_t = typename Store<TS>::acc;
    using s_t = typename SType<TS, W>::type;
    constexpr int TK = Store<TS>::TK;
    const FarItem it = items[blockIdx.x];
    const InstDesc& I = inst_of<BATCH>(one, insts, it.inst);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));  // uniform
    const int split = it.nrg == 1 ? 4 : it.nrg == 2 ? 2 : 1;  // waves per row group
    const int g = wave / split;
    if (g >= it.nrg) return;  // three row groups: no barrier below
    constexpr int NB = kSlices<W>, WS = W / NB;
    __shared__ alignas(16) char btile[kWaves][BTile<TS, W>::BYTES];
    __shared__ acc_t red[kWaves][64][WS];
    const int rows = g == it.nrg - 1 ? it.rows_last : 64;
    const TS* pd = static_cast<const TS*>(I.panel) + it.data_off +
                   static_cast<int64_t>(g) * 64 * it.ktiles * TK;
    s_t* S = static_cast<s_t*>(I.S);
    acc_t* partial = static_cast<acc_t*>(I.partial);
    // result of row `row` of the item, column c
    auto store = [&](int row, int c, acc_t v) {
        const int64_t o = it.out_off + row;
        if (it.to_T)
            S[(I.s0 + I.n + o) * W + c] = from_double<s_t>(static_cast<double>(v));
        else
            partial[o * W + c] = v;
    };
    PanelAcc<TS, W> acc[4 * NB];
#pragma unroll
    for (int q = 0; q < 4 * NB; q++) acc[q] = PanelAcc<TS, W>{};
    dispatch_nrt(rows, [&](auto nrt) {
        panel_accum<TS, W, false, decltype(nrt)::value, CP, WIDE, XDIR>(
            pd, rows, it.ktiles, it.col_off, it.ncols, XDIR ? I.smap0 : nullptr, 0, 0, S, I.s_rows,
            wave % split, split, lane, btile[wave], acc, I.X, I.n);
    });
    if (split == 1) {
#pragma unroll
        for (int b = 0; b < NB; b++)
            panel_emit<TS, W>(acc, (rows + 15) >> 4, b, lane, [&](int row, int j, acc_t v) {
                if (row < rows) store(64 * g + row, WS * b + j, v);
            });
        return;
    }
    const int total = 64 * (it.nrg - 1) + it.rows_last;
#pragma unroll
    for (int b = 0; b < NB; b++) {  // one slice at a time through LDS
        if (b) __syncthreads();
        panel_emit<TS, W>(acc, (rows + 15) >> 4, b, lane,
                          [&](int row, int j, acc_t v) { red[wave][row][j] = v; });
        __syncthreads();
        for (int t = threadIdx.x; t < total * WS; t += kWaves * 64) {
            const int row = t / WS, j = t % WS, w0 = row / 64 * split;
            acc_t v = red[w0][row % 64][j];
            for (int w = 1; w < split; w++) v += red[w0 + w][row % 64][j];
            store(row, WS * b + j, v);
        }
    }
}

// Sum the column-chunk partials of far-field row groups in a fixed order.
template <typename TS, int W, bool BATCH>
__global__ __launch_bounds__(256) void k_reduce(const ReduceGroup* __restrict__ groups,
                                                const InstDesc one,
                                                const InstDesc* __restrict__ insts) {
    using acc_t = typename Store<TS>::acc;
    using s_t = typename SType<TS, W>::type;
    const ReduceGroup g = groups[blockIdx.x];
    const InstDesc& I = inst_of<BATCH>(one, insts, g.inst);
    const acc_t* partial = static_cast<const acc_t*>(I.partial);
    s_t* S = static_cast<s_t*>(I.S);
    for (int t = threadIdx.x; t < g.rows * W; t += blockDim.x) {
        const int r = t / W, j = t % W;
        acc_t s = 0;
        for (int c = 0; c < g.nch; c++) s += partial[(g.pbase + static_cast<int64_t>(c) * g.rows + r) * W + j];
        S[(I.s0 + I.n + g.tbase + r) * W + j] = from_double<s_t>(static_cast<double>(s));
    }
}

// S[s0 + p][j] = X[smap[p], rhs0 + j]  (zero for j beyond nrhs); thread per original
// source index, instance = blockIdx.y.  Reads are coalesced per column of X;
// each thread writes its S row whole.
template <typename TS, int W, typename TIO, bool BATCH>
__global__ __launch_bounds__(256) void k_gather(const InstDesc one, const InstDesc* __restrict__ insts) {
    using s_t = typename SType<TS, W>::type;
    const InstDesc& I = inst_of<BATCH>(one, insts, blockIdx.y);
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= I.n) return;
    const TIO* X = static_cast<const TIO*>(I.X);
    const int64_t p = I.inv_smap[t];
    SRowOut<s_t, W> row;
#pragma unroll
    for (int j = 0; j < W; j++) {
        const int c = I.rhs0 + j;
        const double v = c < I.nrhs ? static_cast<double>(X[t + static_cast<int64_t>(c) * I.ldx]) : 0.0;
        row.v[j] = from_double<s_t>(v);
    }
    reinterpret_cast<SRowOut<s_t, W>*>(I.S)[I.s0 + p] = row;
}

// Zero n16 16-byte words.
static __global__ __launch_bounds__(256) void k_zero16(uint4* __restrict__ p, int64_t n16) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n16) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// ---- build-time panel generation ------------------------------------------------
// Column descriptors of the leaf panels: kind 0 = built-in kernel entry
// (base = 0-based original source index), 1 = U payload, 2 = dense payload (callback
// kernels), 3 = padding.  Buffer element (row r) = base + r * stride.
struct ColDesc {
    int64_t base;
    int32_t stride;
    int32_t kind;
};

__device__ inline double kernel_entry(int kid, const double* a, const double* b) {
#pragma clang fp contract(off)
    if (kid == HMX_KERNEL_LAPLACE) {
        const double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
        double d2 = dx * dx + dy * dy;
        d2 = d2 + dz * dz;
        const double d = sqrt(d2);
        return d == 0.0 ? 0.0 : 1.0 / d;
    }
    // HMX_KERNEL_LOG2D: generic_norm2 branch without scaling (scaling only
    // triggers for |r| < 1e-154, where the entry is 1.0 anyway).
    const double r0 = a[0] - b[0], r1 = a[1] - b[1], r2 = a[2] - b[2];
    double s = r0 * r0;
    s += r1 * r1;
    s += r2 * r2;
    const double d = sqrt(s);
    return d < 1e-12 ? 1.0 : (-0.5 / 3.141592653589793) * log(d);
}

// dipolar_tensor_xx / _xy of examples/hmatrix_vector.jl:12-28 (same operation
// order as the host and the reference)
__device__ inline double dip_xx(double x, double y, double z) {
#pragma clang fp contract(off)
    const double R = x * x + y * y + z * z;
    if (R == 0) return 0.0;
    return -(2 * x * x - y * y - z * z) / (R * R * sqrt(R)) / (4 * 3.141592653589793);
}
__device__ inline double dip_xy(double x, double y, double z) {
#pragma clang fp contract(off)
    const double R = x * x + y * y + z * z;
    if (R == 0) return 0.0;
    return -3 * x * y / (R * R * sqrt(R)) / (4 * 3.141592653589793);
}

// Component (ca, cb) of the dipolar tensor at r = (x, y, z) (hmatrix_vector.jl:30-51).
__device__ inline double dip_component(int ca, int cb, double x, double y, double z) {
    if (ca == cb) return ca == 0 ? dip_xx(x, y, z) : ca == 1 ? dip_xx(y, x, z) : dip_xx(z, y, x);
    const int s = ca + cb;  // 1: xy, 2: xz, 3: yz
    return s == 1 ? dip_xy(x, y, z) : s == 2 ? dip_xy(x, z, y) : dip_xy(y, z, x);
}

// Entry of a built-in kernel between original target index i and source index
// j: points for the scalar kernels, degrees of freedom 3p + a for the dipole
// tensor.
__device__ inline double kernel_entry_ij(int kid, const double* xt, const double* xs, int64_t i,
                                         int64_t j) {
#pragma clang fp contract(off)
    if (kid == HMX_KERNEL_DIPOLE) {
        const double* a = xt + 3 * (i / 3);
        const double* b = xs + 3 * (j / 3);
        return dip_component(static_cast<int>(i % 3), static_cast<int>(j % 3), a[0] - b[0],
                             a[1] - b[1], a[2] - b[2]);
    }
    return kernel_entry(kid, xt + 3 * i, xs + 3 * j);
}

// Element (row r, column k) of an item, at tile position q (16-byte chunks).
template <typename TS>
__device__ inline void chunk_coords(int q, int rows, int& kt, int& r, int& k0) {
    constexpr int TK = Store<TS>::TK, EPL = Store<TS>::EPL;
    const int per_slab = rows * 4;
    kt = q / per_slab;
    const int c = q % per_slab;
    const int rt = c / 64;
    const int rr = min(16, rows - 16 * rt);
    const int w = c % 64;
    const int g = w / rr, i = w % rr;
    r = 16 * rt + i;
    k0 = kt * TK + g * EPL;
}

template <typename TS>
__global__ __launch_bounds__(256) void k_gen_leaf(const Item* __restrict__ items, TS* __restrict__ panel,
                                                  const ColDesc* __restrict__ cols,
                                                  const int32_t* __restrict__ tmap0,
                                                  const double* __restrict__ xt,
                                                  const double* __restrict__ xs,
                                                  const double* __restrict__ Ubuf,
                                                  const double* __restrict__ Dbuf, int kid) {
    constexpr int EPL = Store<TS>::EPL;
    const Item it = items[blockIdx.x];
    const int nchunks = it.ktiles * it.rows * 4;
    for (int q = threadIdx.x; q < nchunks; q += blockDim.x) {
        int kt, r, k0;
        chunk_coords<TS>(q, it.rows, kt, r, k0);
        const int64_t trow = it.out_off + r;
        const int64_t ti = tmap0[trow];  // original target index
        TS vals[EPL];
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const ColDesc cd = cols[it.col_off + k0 + e];
            double v = 0.0;
            if (cd.kind == 0)
                v = kernel_entry_ij(kid, xt, xs, ti, cd.base);
            else if (cd.kind == 1)
                v = Ubuf[cd.base + static_cast<int64_t>(r) * cd.stride];
            else if (cd.kind == 2)
                v = Dbuf[cd.base + static_cast<int64_t>(r) * cd.stride];
            vals[e] = from_double<TS>(v);
        }
        // chunk q of the item sits at data_off + q*EPL (chunk-major tiles)
        std::memcpy(panel + it.data_off + static_cast<int64_t>(q) * EPL, vals, sizeof(vals));
    }
}

// Far-field panels: element (r, k) = V[vrow[vbase + r] + kc0 + k] for k < ncols.
struct GenA {
    int64_t vbase;  // first entry of vrow for this item's rows
    int64_t kc0;    // first column of the chunk inside the source cluster
};

template <typename TS>
__global__ __launch_bounds__(256) void k_gen_far(const Item* __restrict__ items,
                                                 const GenA* __restrict__ gens, TS* __restrict__ panel,
                                                 const int64_t* __restrict__ vrow,
                                                 const double* __restrict__ Vbuf) {
    constexpr int EPL = Store<TS>::EPL;
    const Item it = items[blockIdx.x];
    const GenA g = gens[blockIdx.x];
    const int nchunks = it.ktiles * it.rows * 4;
    for (int q = threadIdx.x; q < nchunks; q += blockDim.x) {
        int kt, r, k0;
        chunk_coords<TS>(q, it.rows, kt, r, k0);
        const int64_t vb = vrow[g.vbase + r] + g.kc0;
        TS vals[EPL];
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const int k = k0 + e;
            vals[e] = from_double<TS>(k < it.ncols ? Vbuf[vb + k] : 0.0);
        }
        std::memcpy(panel + it.data_off + static_cast<int64_t>(q) * EPL, vals, sizeof(vals));
    }
}

}  // namespace hmx
