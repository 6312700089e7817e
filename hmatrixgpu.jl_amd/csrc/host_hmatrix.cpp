// host_hmatrix.cpp -- H-matrix construction on the host.
//
//   build_hmatrix    HMatrix(K, X, Y; eta, eps, svd_recompress), hmatrix.jl:72-148
//                    with build_matrices, hmatrix.jl:170-217, and the flattened
//                    reference layout of hmatrix.jl:95-147
//   EntrySource      the user-matrix getindex contract (hmatrix.jl:183,195-196,209)
//                    plus native built-in kernels
//
// Low-rank blocks are compressed in parallel (one block per task); each task is
// a deterministic sequential FP64 computation, so the result does not depend on
// the thread count.  Compiled with -ffp-contract=off.
#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>

#include "hmx_host.hpp"

#include <sys/mman.h>

namespace hmx {

int default_threads() {
    for (const char* var : {"HMX_NUM_THREADS", "OMP_NUM_THREADS"}) {
        const char* s = std::getenv(var);
        if (s && std::atoi(s) > 0) return std::atoi(s);
    }
    unsigned hc = std::thread::hardware_concurrency();
    return hc ? static_cast<int>(hc) : 1;
}

void parallel_for(int64_t n, int threads, const std::function<void(int64_t)>& f) {
    if (threads <= 1 || n <= 1) {
        for (int64_t i = 0; i < n; i++) f(i);
        return;
    }
    std::atomic<int64_t> next{0};
    std::exception_ptr err;
    std::mutex mu;
    auto work = [&]() {
        for (;;) {
            int64_t i = next.fetch_add(1);
            if (i >= n) return;
            try {
                f(i);
            } catch (...) {
                std::lock_guard<std::mutex> g(mu);
                if (!err) err = std::current_exception();
                next.store(n);
                return;
            }
        }
    };
    int t = static_cast<int>(std::min<int64_t>(threads, n));
    std::vector<std::thread> pool;
    for (int i = 1; i < t; i++) pool.emplace_back(work);
    work();
    for (auto& th : pool) th.join();
    if (err) std::rethrow_exception(err);
}

// ---- entries ---------------------------------------------------------------
namespace {
// dipolar_tensor_xx / _xy of examples/hmatrix_vector.jl:12-28, same operation
// order (R is summed from the arguments as passed)
double dip_xx(double x, double y, double z) {
    const double R = x * x + y * y + z * z;
    if (R == 0) return 0.0;
    return -(2 * x * x - y * y - z * z) / (R * R * std::sqrt(R)) / (4 * 3.141592653589793);
}
double dip_xy(double x, double y, double z) {
    const double R = x * x + y * y + z * z;
    if (R == 0) return 0.0;
    return -3 * x * y / (R * R * std::sqrt(R)) / (4 * 3.141592653589793);
}
// component (a, b) of dipolar_tensor(x, y, z) (hmatrix_vector.jl:30-51)
double dipole(int a, int b, double x, double y, double z) {
    if (a == b) return a == 0 ? dip_xx(x, y, z) : a == 1 ? dip_xx(y, x, z) : dip_xx(z, y, x);
    const int s = a + b;  // 1: xy, 2: xz, 3: yz
    return s == 1 ? dip_xy(x, y, z) : s == 2 ? dip_xy(x, z, y) : dip_xy(y, z, x);
}
}  // namespace

double EntrySource::entry(int64_t i, int64_t j) const {
    if (kernel_id == HMX_KERNEL_DIPOLE) {  // degrees of freedom 3p + a, 3q + b
        const double* a = xt + 3 * (i / 3);
        const double* b = xs + 3 * (j / 3);
        return dipole(static_cast<int>(i % 3), static_cast<int>(j % 3), a[0] - b[0], a[1] - b[1],
                      a[2] - b[2]);
    }
    const double* a = xt + 3 * i;
    const double* b = xs + 3 * j;
    if (kernel_id == HMX_KERNEL_LAPLACE) {
        const double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
        double d2 = dx * dx + dy * dy;
        d2 = d2 + dz * dz;
        const double d = std::sqrt(d2);
        return d == 0.0 ? 0.0 : 1.0 / d;
    }
    // HMX_KERNEL_LOG2D
    double r[3] = {a[0] - b[0], a[1] - b[1], a[2] - b[2]};
    const double d = norm3(r);
    return d < 1e-12 ? 1.0 : (-0.5 / 3.141592653589793) * std::log(d);
}

void EntrySource::block(const int64_t* rows, int64_t nr, const int64_t* cols, int64_t nc,
                        double* out) const {
    if (kernel_id != HMX_KERNEL_CALLBACK) {
        for (int64_t j = 0; j < nc; j++)
            for (int64_t i = 0; i < nr; i++) out[i + j * nr] = entry(rows[i], cols[j]);
        return;
    }
    // The callback receives 1-based indices (Julia getindex).
    std::vector<int64_t> r1(rows, rows + nr), c1(cols, cols + nc);
    for (auto& v : r1) v += 1;
    for (auto& v : c1) v += 1;
    int rc = fill(ctx, r1.data(), nr, c1.data(), nc, out);
    if (rc != 0) throw Error(HMX_ERR_CALLBACK, "entry callback returned " + std::to_string(rc));
}

// ---- H-matrix ----------------------------------------------------------------
void advise_huge_pages(void* p, size_t bytes) {
    const uintptr_t huge = uintptr_t(2) << 20;
    const uintptr_t a = (reinterpret_cast<uintptr_t>(p) + huge - 1) & ~(huge - 1);
    const uintptr_t e = (reinterpret_cast<uintptr_t>(p) + bytes) & ~(huge - 1);
    if (p && e > a) (void)madvise(reinterpret_cast<void*>(a), e - a, MADV_HUGEPAGE);
}

void HMatrix::ensure_dense_payload() {
    if (D_ready) return;
    D.resize(static_cast<size_t>(dlen));  // every element is written below
    advise_huge_pages(D.data(), D.size() * sizeof(double));
    const int threads = src.thread_safe() ? default_threads() : 1;
    parallel_for(static_cast<int64_t>(dense.size()), threads, [&](int64_t b) {
        const DenseBlock& d = dense[b];
        const int64_t mm = d.r1 - d.r0 + 1, nn = d.c1 - d.c0 + 1;
        std::vector<int64_t> rows(mm), cols(nn);
        for (int64_t i = 0; i < mm; i++) rows[i] = tmap[d.r0 - 1 + i] - 1;
        for (int64_t j = 0; j < nn; j++) cols[j] = smap[d.c0 - 1 + j] - 1;
        std::vector<double> cm(mm * nn);
        src.block(rows.data(), mm, cols.data(), nn, cm.data());
        double* out = D.data() + d.off;  // vec(D'): row-major
        for (int64_t i = 0; i < mm; i++)
            for (int64_t j = 0; j < nn; j++) out[i * nn + j] = cm[i + j * mm];
    });
    D_ready = true;
}

namespace {

// Eigenvalues of a symmetric 3 x 3 matrix (cyclic Jacobi), largest first.
void sym3_eigenvalues(double a[3][3], double ev[3]) {
    for (int sweep = 0; sweep < 12; sweep++) {
        const double off = a[0][1] * a[0][1] + a[0][2] * a[0][2] + a[1][2] * a[1][2];
        const double diag = a[0][0] * a[0][0] + a[1][1] * a[1][1] + a[2][2] * a[2][2];
        if (off <= 1e-30 * diag || off == 0.0) break;
        for (int p = 0; p < 2; p++)
            for (int q = p + 1; q < 3; q++) {
                if (a[p][q] == 0.0) continue;
                const double th = (a[q][q] - a[p][p]) / (2.0 * a[p][q]);
                const double t = (th >= 0 ? 1.0 : -1.0) / (std::fabs(th) + std::sqrt(th * th + 1.0));
                const double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
                for (int k = 0; k < 3; k++) {  // columns p, q
                    const double akp = a[k][p], akq = a[k][q];
                    a[k][p] = c * akp - s * akq;
                    a[k][q] = s * akp + c * akq;
                }
                for (int k = 0; k < 3; k++) {  // rows p, q
                    const double apk = a[p][k], aqk = a[q][k];
                    a[p][k] = c * apk - s * aqk;
                    a[q][k] = s * apk + c * aqk;
                }
            }
    }
    ev[0] = a[0][0];
    ev[1] = a[1][1];
    ev[2] = a[2][2];
    std::sort(ev, ev + 3, [](double x, double y) { return x > y; });
}

// Principal-axis shape of every cluster: 0.5 log(l2 / l1) and 0.5 log(l3 / l1)
// for the eigenvalues l1 >= l2 >= l3 of the covariance of its points (ratios
// clamped at 1e-8; 0 for a cluster of coincident points or without
// coordinates).  (0, 0) is an isotropic volume, (0, -inf) a flat patch,
// (-inf, -inf) a line: the geometry that sets how fast the kernel's singular
// values decay, independent of the cluster's scale and orientation.
std::vector<std::array<float, 2>> cluster_shapes(const ClusterTree& T, const double* x,
                                                 int threads) {
    const int64_t nn = static_cast<int64_t>(T.nodes.size());
    std::vector<std::array<float, 2>> out(static_cast<size_t>(nn), {0.f, 0.f});
    if (!x) return out;
    parallel_for(nn, threads, [&](int64_t id) {
        const ClusterNode& c = T.nodes[id];
        double s1[3] = {0, 0, 0}, s2[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        const int64_t cnt = c.end - c.start;
        if (cnt <= 0) return;
        for (int64_t p = c.start - 1; p < c.end - 1; p++) {
            const double* q = x + 3 * ((T.index_map[p] - 1) / T.dims);
            const double d[3] = {q[0] - c.center[0], q[1] - c.center[1], q[2] - c.center[2]};
            for (int i = 0; i < 3; i++) {
                s1[i] += d[i];
                for (int j = 0; j < 3; j++) s2[i][j] += d[i] * d[j];
            }
        }
        double cov[3][3];
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++)
                cov[i][j] = s2[i][j] / cnt - (s1[i] / cnt) * (s1[j] / cnt);
        double ev[3];
        sym3_eigenvalues(cov, ev);
        if (!(ev[0] > 0.0)) return;
        auto half_log = [&](double l) {
            return static_cast<float>(0.5 * std::log(std::max(l / ev[0], 1e-8)));
        };
        out[id] = {half_log(ev[1]), half_log(ev[2])};
    });
    return out;
}

// Rank-predictor inputs of an admissible block (rankpred.hip), chosen to be
// invariant under a change of length scale: ACA+ stops on an absolute step
// size (aca.jl:96-100) while a kernel of decay order p (K(s x, s y) =
// s^-p K(x, y): p = 1 for 1/r, 3 for the dipole tensor) scales the block by
// s^-p, so tol * dist^p is the tolerance relative to the block's entries.
//   0, 1  log(diam_s / dist), log(diam_t / dist)
//   2     log(tol * dist^p)
//   3, 4  log n_s, log n_t
//   5..8  cluster_shapes of s, then of t
void block_features(const ClusterNode& t, const ClusterNode& s, double tol, int decay,
                    const std::array<float, 2>& shape_t, const std::array<float, 2>& shape_s,
                    float* f) {
    auto lg = [](double x) { return std::log(std::max(x, 1e-300)); };
    // ratios clamped to [e^-14, e^14]: a cluster of coincident points has
    // diameter 0, and such clusters may also coincide (distance 0)
    auto lratio = [&](double a, double b) {
        return static_cast<float>(std::min(14.0, std::max(-14.0, lg(a) - lg(b))));
    };
    const double d[3] = {t.center[0] - s.center[0], t.center[1] - s.center[1],
                         t.center[2] - s.center[2]};
    const double dist = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    const double ld = lg(dist);
    f[0] = lratio(2.0 * s.radius, dist);
    f[1] = lratio(2.0 * t.radius, dist);
    f[2] = static_cast<float>(lg(tol) + decay * ld);
    f[3] = static_cast<float>(lg(static_cast<double>(s.end - s.start)));
    f[4] = static_cast<float>(lg(static_cast<double>(t.end - t.start)));
    f[5] = shape_s[0];
    f[6] = shape_s[1];
    f[7] = shape_t[0];
    f[8] = shape_t[1];
}

}  // namespace

std::unique_ptr<HMatrix> build_hmatrix(const ClusterTree& T, const ClusterTree& S,
                                       const EntrySource& src, double eta, double eps, bool svd,
                                       int nthreads, const BuildOptions* opt) {
    const BuildOptions defaults;
    if (!opt) opt = &defaults;
    auto t0 = std::chrono::steady_clock::now();
    auto h = std::make_unique<HMatrix>();
    h->src = src;
    h->m = static_cast<int64_t>(T.index_map.size());
    h->n = static_cast<int64_t>(S.index_map.size());
    h->tmap = T.index_map;
    h->smap = S.index_map;
    h->target_dims = T.dims;
    h->source_dims = S.dims;

    auto bt = build_block_tree(T, S, eta);  // hmatrix.jl:74
    merge_dense(*bt);                       // :75
    std::vector<std::pair<int64_t, int64_t>> direct, approx;
    traverse(*bt, &direct, &approx);        // :78
    bt.reset();

    // Compress every admissible block (ACA+ at eps/10, then SVD at eps).
    const int threads = src.thread_safe() ? (nthreads > 0 ? nthreads : default_threads()) : 1;

    const int64_t na = static_cast<int64_t>(approx.size());
    h->approx_stats.assign(static_cast<size_t>(na), HMatrix::ApproxStat{});
    {
        const int cpu_threads = nthreads > 0 ? nthreads : default_threads();
        const auto shape_t = cluster_shapes(T, src.xt, cpu_threads);
        const auto shape_s = &S == &T && src.xs == src.xt ? shape_t
                                                          : cluster_shapes(S, src.xs, cpu_threads);
        const int decay = src.kernel_id == HMX_KERNEL_LAPLACE  ? 1
                          : src.kernel_id == HMX_KERNEL_DIPOLE ? 3
                                                               : 0;
        for (int64_t b = 0; b < na; b++)
            block_features(T.nodes[approx[b].first], S.nodes[approx[b].second], eps, decay,
                           shape_t[approx[b].first], shape_s[approx[b].second],
                           h->approx_stats[b].feat);
    }
    std::vector<LowRank> lr(approx.size());
    std::vector<std::unique_ptr<FactorSlab>> slabs;  // recompressed on the GPU (lr stays empty)
    std::mutex slab_mu;
    std::vector<int64_t> rank(approx.size(), 0);
    if (opt->aca_device == 1) {
        // batched ACA+ on the GPU with a rank capacity per block; recompressed there
        // too, or (for a tolerance below zero, which the device does not take) on host
        // threads as blocks come back
        std::vector<AcaBlock> blocks(static_cast<size_t>(na));
        std::vector<int32_t> caps(static_cast<size_t>(na), std::max(1, opt->initial_rank));
        for (int64_t b = 0; b < na; b++) {
            const ClusterNode& a = T.nodes[approx[b].first];
            const ClusterNode& s = S.nodes[approx[b].second];
            blocks[b] = AcaBlock{a.start - 1, s.start - 1, a.end - a.start, s.end - s.start};
        }
        std::vector<float> X(static_cast<size_t>(na) * kRankFeatures);
        for (int64_t b = 0; b < na; b++)
            std::copy(h->approx_stats[b].feat, h->approx_stats[b].feat + kRankFeatures,
                      X.begin() + b * kRankFeatures);
        // capacity = ceil((1 + margin) * predicted rank)
        auto predict_caps = [&](const RankPredictor& p, std::vector<int32_t>& out,
                                const std::vector<char>* skip) {
            std::vector<float> z(static_cast<size_t>(na));
            rankpred_predict(p, X.data(), na, z.data());
            for (int64_t b = 0; b < na; b++) {
                if (skip && (*skip)[b]) continue;
                const double r = std::expm1(static_cast<double>(z[b]));
                const double c = std::ceil((1.0 + opt->cap_margin) * std::max(r, 0.0));
                out[b] = static_cast<int32_t>(std::min<double>(std::max(c, 1.0), 1 << 30));
            }
        };
        if (opt->predictor && na > 0) predict_caps(*opt->predictor, caps, nullptr);
        auto record_caps = [&](const std::vector<char>* skip) {
            for (int64_t b = 0; b < na; b++)
                if (!skip || !(*skip)[b])
                    h->approx_stats[b].cap = static_cast<int32_t>(
                        aca_round_cap(caps[b], std::min(blocks[b].m, blocks[b].n)));
        };
        record_caps(nullptr);
        // Probe phase: an evenly spaced sample of the admissible blocks (DFS
        // order, so every level and region is represented) runs first; a copy
        // of the predictor is fine-tuned on their ACA+ ranks and predicts the
        // capacities of the remaining blocks.
        std::vector<int64_t> probe;
        std::vector<char> in_probe;
        AcaRefine refine;
        if (opt->predictor && opt->refine_samples > 0 && na >= 4 * int64_t(opt->refine_samples)) {
            const int64_t step = na / opt->refine_samples;
            in_probe.assign(static_cast<size_t>(na), 0);
            for (int64_t b = 0; b < na; b += step) {
                probe.push_back(b);
                in_probe[b] = 1;
            }
            refine = [&](const std::vector<int64_t>& ids, const std::vector<int32_t>& ranks,
                         std::vector<int32_t>& c) {
                std::unique_ptr<RankPredictor, void (*)(RankPredictor*)> q(
                    rankpred_clone(*opt->predictor), rankpred_destroy);
                std::vector<float> Xs(ids.size() * kRankFeatures), zs(ids.size());
                for (size_t i = 0; i < ids.size(); i++) {
                    std::copy(X.begin() + ids[i] * kRankFeatures,
                              X.begin() + (ids[i] + 1) * kRankFeatures, Xs.begin() + i * kRankFeatures);
                    zs[i] = static_cast<float>(std::log1p(static_cast<double>(ranks[i])));
                }
                rankpred_train(*q, Xs.data(), zs.data(), static_cast<int64_t>(ids.size()),
                               opt->refine_epochs, 256, 3e-3f, 0x5eedULL, nullptr);
                predict_caps(*q, c, &in_probe);
                caps = c;
                record_caps(&in_probe);
            };
        }
        h->device = opt->device;
        gpu_aca(*h, blocks, caps, eps / 10.0, svd ? eps : -1.0, threads, opt->stats,
                [&](int64_t b, int64_t aca_k, LowRank&& f) {
                    h->approx_stats[b].aca_rank = static_cast<int32_t>(aca_k);
                    lr[b] = svd ? svd_recompress(f, eps) : std::move(f);
                    rank[b] = lr[b].k;
                },
                [&](std::unique_ptr<FactorSlab> s) {
                    for (const FactorSlab::Part& p : s->parts) {
                        h->approx_stats[p.block].aca_rank = static_cast<int32_t>(p.aca_k);
                        rank[p.block] = p.k;
                    }
                    std::lock_guard<std::mutex> g(slab_mu);
                    slabs.push_back(std::move(s));
                },
                probe, refine);
    } else
    parallel_for(static_cast<int64_t>(approx.size()), threads, [&](int64_t b) {
        const ClusterNode& a = T.nodes[approx[b].first];
        const ClusterNode& s = S.nodes[approx[b].second];
        const int64_t mm = a.end - a.start, nn = s.end - s.start;
        std::vector<int64_t> rows(mm), cols(nn);
        for (int64_t i = 0; i < mm; i++) rows[i] = T.index_map[a.start - 1 + i] - 1;
        for (int64_t j = 0; j < nn; j++) cols[j] = S.index_map[s.start - 1 + j] - 1;
        RowFn rowf, colf;
        if (src.kernel_id != HMX_KERNEL_CALLBACK) {
            rowf = [&](int64_t I, double* out) {
                for (int64_t j = 0; j < nn; j++) out[j] = src.entry(rows[I], cols[j]);
            };
            colf = [&](int64_t J, double* out) {
                for (int64_t i = 0; i < mm; i++) out[i] = src.entry(rows[i], cols[J]);
            };
        } else {
            rowf = [&](int64_t I, double* out) { src.block(&rows[I], 1, cols.data(), nn, out); };
            colf = [&](int64_t J, double* out) { src.block(rows.data(), mm, &cols[J], 1, out); };
        }
        LowRank f = aca_plus(mm, nn, rowf, colf, eps / 10.0, 0);  // hmatrix.jl:194-196
        h->approx_stats[b].aca_rank = static_cast<int32_t>(f.k);
        if (svd) f = svd_recompress(f, eps);                       // :197-199
        rank[b] = f.k;
        lr[b] = std::move(f);
    });
    for (int64_t b = 0; b < na; b++) h->approx_stats[b].rank = static_cast<int32_t>(rank[b]);

    // Storage test (m+n)k < mn, else the block is stored dense after all direct
    // blocks, in approx order (hmatrix.jl:202-213).
    int64_t off = 0;
    auto add_dense = [&](const ClusterNode& a, const ClusterNode& s) {
        DenseBlock d{a.start, a.end - 1, s.start, s.end - 1, off};
        off += (a.end - a.start) * (s.end - s.start);
        h->dense.push_back(d);
    };
    for (auto& [ti, si] : direct) add_dense(T.nodes[ti], S.nodes[si]);
    int64_t ulen = 0, vlen = 0, vx = 0;
    std::vector<int64_t> keep;
    for (size_t b = 0; b < approx.size(); b++) {
        const ClusterNode& a = T.nodes[approx[b].first];
        const ClusterNode& s = S.nodes[approx[b].second];
        const int64_t mm = a.end - a.start, nn = s.end - s.start, k = rank[b];
        if (mm * k + k * nn < mm * nn) {
            LowRankBlock L{a.start, a.end - 1, s.start, s.end - 1, k, ulen, vlen, vx,
                           approx[b].second};
            h->lowrank.push_back(L);
            keep.push_back(static_cast<int64_t>(b));
            ulen += mm * k;
            vlen += nn * k;
            vx += k;
        } else {
            add_dense(a, s);
            lr[b] = LowRank();
        }
    }
    h->dlen = off;
    h->R = vx;
    h->U.resize(static_cast<size_t>(ulen));
    h->V.resize(static_cast<size_t>(vlen));
    advise_huge_pages(h->U.data(), h->U.size() * sizeof(double));
    advise_huge_pages(h->V.data(), h->V.size() * sizeof(double));
    std::vector<int64_t> pos(slabs.empty() ? 0 : approx.size(), -1);  // block -> h->lowrank
    if (!slabs.empty())
        for (size_t q = 0; q < keep.size(); q++) pos[keep[q]] = static_cast<int64_t>(q);
    parallel_for(static_cast<int64_t>(slabs.size()), threads, [&](int64_t s) {
        const FactorSlab& S = *slabs[s];
        for (const FactorSlab::Part& p : S.parts) {
            if (pos[p.block] < 0) continue;  // stored dense
            const LowRankBlock& L = h->lowrank[pos[p.block]];
            const double* src = S.data.data() + p.off;
            double* U = h->U.data() + L.uoff;  // vec(U'): U row-major m x k
            for (int64_t i = 0; i < p.m; i++)
                for (int64_t c = 0; c < p.k; c++) U[i * p.k + c] = src[i + c * p.m];
            std::copy(src + p.k * p.m, src + p.k * (p.m + p.n), h->V.data() + L.voff);
        }
        slabs[s].reset();
    });
    parallel_for(slabs.empty() ? static_cast<int64_t>(keep.size()) : 0, threads, [&](int64_t q) {
        LowRank& f = lr[keep[q]];
        const LowRankBlock& L = h->lowrank[q];
        double* U = h->U.data() + L.uoff;  // vec(U'): U row-major m x k
        for (int64_t i = 0; i < f.m; i++)
            for (int64_t c = 0; c < f.k; c++) U[i * f.k + c] = f.U[i + c * f.m];
        double* V = h->V.data() + L.voff;  // vec(V'): V row-major k x n
        for (int64_t c = 0; c < f.k; c++)
            for (int64_t j = 0; j < f.n; j++) V[c * f.n + j] = f.V[c + j * f.k];
        f = LowRank();  // release the column-major factors as soon as they are copied
    });
    for (int64_t l : T.leaves) h->target_leaf_start.push_back(T.nodes[l].start - 1);
    h->target_leaf_start.push_back(h->m);
    if (src.kernel_id == HMX_KERNEL_CALLBACK) h->ensure_dense_payload();
    h->build_seconds =
        std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return h;
}

// ---- sparsify_hmatrix (hmatrix.jl:234-274) ------------------------------------------
// Every entry of the merged dense blocks of the block tree, as a CSR matrix in
// the original index spaces (0-based, columns sorted within a row).  Rows are
// owned by exactly one target leaf, so leaves are filled in parallel.
CsrMatrix sparsify(const ClusterTree& T, const ClusterTree& S, const EntrySource& src, double eta,
                   int nthreads) {
    auto bt = build_block_tree(T, S, eta);  // hmatrix.jl:236
    merge_dense(*bt);                       // :237
    std::vector<std::pair<int64_t, int64_t>> direct, approx;
    traverse(*bt, &direct, &approx);        // :239
    bt.reset();
    CsrMatrix out;
    out.m = static_cast<int64_t>(T.index_map.size());
    out.n = static_cast<int64_t>(S.index_map.size());
    // dense blocks covering each target leaf (a block's rows are a union of leaves)
    const int64_t nl = static_cast<int64_t>(T.leaves.size());
    std::vector<int64_t> leaf_start(nl);
    for (int64_t l = 0; l < nl; l++) leaf_start[l] = T.nodes[T.leaves[l]].start;
    std::vector<std::vector<int32_t>> blocks_of(nl);
    for (size_t d = 0; d < direct.size(); d++) {
        const ClusterNode& a = T.nodes[direct[d].first];
        const int64_t l0 = std::lower_bound(leaf_start.begin(), leaf_start.end(), a.start) -
                           leaf_start.begin();
        for (int64_t l = l0; l < nl && leaf_start[l] < a.end; l++)
            blocks_of[l].push_back(static_cast<int32_t>(d));
    }
    auto leaf_rows = [&](int64_t l) {  // permuted positions [r0, r1) of leaf l (node
        const ClusterNode& L = T.nodes[T.leaves[l]];  // ranges are in index-map units)
        return std::make_pair(L.start - 1, L.end - 1);
    };
    std::vector<int64_t> row_nnz(static_cast<size_t>(out.m), 0);
    for (int64_t l = 0; l < nl; l++) {
        int64_t w = 0;
        for (int32_t d : blocks_of[l]) {
            const ClusterNode& b = S.nodes[direct[d].second];
            w += b.end - b.start;
        }
        auto [r0, r1] = leaf_rows(l);
        for (int64_t p = r0; p < r1; p++) row_nnz[T.index_map[p] - 1] = w;
    }
    out.rowptr.assign(static_cast<size_t>(out.m + 1), 0);
    for (int64_t r = 0; r < out.m; r++) out.rowptr[r + 1] = out.rowptr[r] + row_nnz[r];
    const int64_t nnz = out.rowptr[out.m];
    out.col.resize(static_cast<size_t>(nnz));
    out.val.resize(static_cast<size_t>(nnz));
    const int threads = src.thread_safe() ? (nthreads > 0 ? nthreads : default_threads()) : 1;
    parallel_for(nl, threads, [&](int64_t l) {
        auto [r0, r1] = leaf_rows(l);
        const int64_t nr = r1 - r0;
        std::vector<int64_t> rows(static_cast<size_t>(nr)), cols;
        for (int64_t i = 0; i < nr; i++) rows[i] = T.index_map[r0 + i] - 1;
        std::vector<int64_t> cursor(static_cast<size_t>(nr));
        for (int64_t i = 0; i < nr; i++) cursor[i] = out.rowptr[rows[i]];
        std::vector<double> blk;
        for (int32_t d : blocks_of[l]) {
            const ClusterNode& b = S.nodes[direct[d].second];
            const int64_t c0 = b.start - 1, nc = b.end - b.start;
            cols.resize(static_cast<size_t>(nc));
            for (int64_t j = 0; j < nc; j++) cols[j] = S.index_map[c0 + j] - 1;
            blk.resize(static_cast<size_t>(nr * nc));
            src.block(rows.data(), nr, cols.data(), nc, blk.data());  // K[target_ids, source_ids]
            for (int64_t i = 0; i < nr; i++)
                for (int64_t j = 0; j < nc; j++) {
                    out.col[cursor[i]] = cols[j];
                    out.val[cursor[i]] = blk[i + j * nr];
                    cursor[i]++;
                }
        }
        // sort each row by column (the blocks' columns are disjoint ranges)
        std::vector<std::pair<int64_t, double>> tmp;
        for (int64_t i = 0; i < nr; i++) {
            const int64_t a = out.rowptr[rows[i]], e = out.rowptr[rows[i] + 1];
            tmp.resize(static_cast<size_t>(e - a));
            for (int64_t q = a; q < e; q++) tmp[q - a] = {out.col[q], out.val[q]};
            std::sort(tmp.begin(), tmp.end(),
                      [](const auto& x, const auto& y) { return x.first < y.first; });
            for (int64_t q = a; q < e; q++) {
                out.col[q] = tmp[q - a].first;
                out.val[q] = tmp[q - a].second;
            }
        }
    });
    return out;
}

}  // namespace hmx
