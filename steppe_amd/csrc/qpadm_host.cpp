// steppe_amd/csrc/qpadm_host.cpp — host side of the batched qpAdm fit
// (HipBackend::qpadm_batch).
//
// Mirrors the reference's batched entry (ComputeBackend::fit_models_batched,
// src/device/cuda/cuda_backend_qpadm_fit.cu:623-960 and run_qpadm_search,
// src/core/qpadm/model_search.cpp:30-218): survivor blocks are found once for the
// tensor, models are validated and grouped by the size of their largest normal
// matrix, and each stage of the fit is one launch per group; results come back in input
// order.  The f2 slab is first transposed to pair-major, survivor-only order so a
// model's f4 basis reads each f2 series contiguously.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <vector>

#include "chunks.hpp"
#include "engine.hpp"
#include "qpadm.hpp"

namespace stp {

namespace {

struct ModelShape {
    int nl, nr;
};

// The normal-matrix bucket of a model: rank sweeps and LOO fits run at ranks up to
// nl - 1, so the largest systems are nl*(nl-1) (A-step) and (nl-1)*nr (B-step).
// Models the batched kernel fits: one f4 entry per lane, one normal-matrix row per lane.
bool fits_batched(int nl, int nr) { return nl * nr <= kMaxQpadmM && nr <= kMaxQpadmNr; }

// Largest normal system of a large model's fits (rank sweep and refits up to nl - 1).
int large_t(int nl, int nr, int rank) {
    const int rmax = std::max(nl - 1, rank);
    return std::max({nl * rmax, rmax * nr, nl});
}

int bucket_of(int nl, int nr, int rank) {
    const int rmax = std::max(nl - 1, rank);
    const int t = std::max({nl * rmax, rmax * nr, nl});
    if (t <= 16) return 16;
    if (t <= 32) return 32;
    if (t <= 48) return 48;
    return 64;
}

// Work on a second stream between a fork from the main one and a join with it.  Without a
// second stream it all runs on the main one.  Left by an exception, it waits for the second
// stream, so that nothing still runs on the workspaces of the failed call.
class Beside {
public:
    Beside(hipStream_t side, hipStream_t main, hipEvent_t (&ev)[2]) : side_(side), main_(main), ev_(ev) {
        if (!side_) return;
        STP_HIP(hipEventRecord(ev_[0], main_));
        STP_HIP(hipStreamWaitEvent(side_, ev_[0], 0));
    }
    ~Beside() {
        if (side_) (void)hipStreamSynchronize(side_);
    }
    Beside(const Beside&) = delete;
    Beside& operator=(const Beside&) = delete;
    hipStream_t stream() const { return side_ ? side_ : main_; }
    void join() {
        if (!side_) return;
        STP_HIP(hipEventRecord(ev_[1], side_));
        STP_HIP(hipStreamWaitEvent(main_, ev_[1], 0));
        side_ = nullptr;
    }

private:
    hipStream_t side_, main_;
    hipEvent_t (&ev_)[2];
};

}  // namespace

hipStream_t HipBackend::side_stream() {
    if (!side_stream_) {
        for (hipEvent_t& e : side_ev_)
            if (!e) STP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        STP_HIP(hipStreamCreateWithFlags(&side_stream_, hipStreamNonBlocking));
    }
    return side_stream_;
}

void HipBackend::qpadm_batch(const F2Blocks& h, int n_models, const std::int32_t* target,
                             const std::int32_t* left_off, const std::int32_t* left, const std::int32_t* right_off,
                             const std::int32_t* right, const stp_qpadm_options& opt, stp_qpadm_result* out) {
    activate();
    STP_REQUIRE(n_models >= 0, "qpadm: n_models must be non-negative");
    if (n_models == 0) return;
    STP_REQUIRE(target && left_off && left && right_off && right && out, "qpadm: null model arena or output");
    STP_REQUIRE(opt.als_iterations >= 0, "qpadm: als_iterations must be non-negative");
    STP_REQUIRE(opt.jackknife >= 0 && opt.jackknife <= 2, "qpadm: jackknife must be 0, 1 or 2");
    STP_REQUIRE(opt.rank >= -1 && opt.rank < STP_QPADM_MAX_RANK, "qpadm: rank out of range");
    const int P = h.P, nb = h.n_block;

    // ---- validate models ----
    std::vector<ModelShape> shape(n_models);
    int total_left = 0, total_right = 0;
    for (int i = 0; i < n_models; ++i) {
        const int nl = left_off[i + 1] - left_off[i];
        const int nr = right_off[i + 1] - right_off[i] - 1;
        const std::string tag = "qpadm: model " + std::to_string(i) + ": ";
        STP_REQUIRE(left_off[i] == total_left && right_off[i] == total_right, tag + "offsets are not cumulative");
        STP_REQUIRE(nl >= 1, tag + "needs at least one source population");
        STP_REQUIRE(nr >= 1, tag + "needs at least two right populations");
        STP_REQUIRE(nl <= STP_QPADM_MAX_NL, tag + "more than " + std::to_string(STP_QPADM_MAX_NL) + " sources");
        // The reference seeds the rank nl - 1 fit from nl - 1 right singular vectors of the
        // nl x nr f4 matrix (seed_AB, cpu_backend.cpp:2738-2744), which exist for nl <= nr + 1.
        STP_REQUIRE(nl <= nr + 1, tag + "needs at least sources - 1 right populations beyond the first");
        STP_REQUIRE(opt.rank < nl, tag + "rank must be below the number of sources");
        if (!fits_batched(nl, nr)) {
            STP_REQUIRE(nl * nr <= kQpLargeMaxM && nr <= kQpLargeMaxNr && large_t(nl, nr, opt.rank) <= kQpLargeMaxT,
                        tag + "model too large (sources x (right - 1) must be <= " + std::to_string(kQpLargeMaxM) +
                            ", right - 1 <= " + std::to_string(kQpLargeMaxNr) + ")");
        }
        STP_REQUIRE(target[i] >= 0 && target[i] < P, tag + "target index out of range");
        for (int k = left_off[i]; k < left_off[i + 1]; ++k)
            STP_REQUIRE(left[k] >= 0 && left[k] < P, tag + "left index out of range");
        for (int k = right_off[i]; k < right_off[i + 1]; ++k)
            STP_REQUIRE(right[k] >= 0 && right[k] < P, tag + "right index out of range");
        total_left += nl;
        total_right += nr + 1;
        shape[i] = ModelShape{nl, nr};
    }
    STP_REQUIRE(left_off[n_models] == total_left && right_off[n_models] == total_right,
                "qpadm: offsets are not cumulative");

    // ---- survivor blocks ----
    STP_REQUIRE(h.tier == kTierResident,
                "qpadm: the f2 tensor is held in host memory or on disk; fits need it resident in HBM");
    const std::int64_t slab = static_cast<std::int64_t>(P) * P;
    qp_keep_.ensure(static_cast<std::size_t>(nb));
    launch_survivors(h.vpair.get(), slab, nb, qp_keep_.get(), stream_);
    std::vector<std::int32_t> keep(nb);
    STP_HIP(hipMemcpyAsync(keep.data(), qp_keep_.get(), nb * sizeof(std::int32_t), hipMemcpyDeviceToHost, stream_));
    STP_HIP(hipStreamSynchronize(stream_));
    std::vector<std::int32_t> surv, bsz;
    double n_total = 0.0;
    for (int b = 0; b < nb; ++b)
        if (keep[b]) {
            surv.push_back(b);
            bsz.push_back(h.block_sizes[b]);
            n_total += static_cast<double>(h.block_sizes[b]);
        }
    const int nbs = static_cast<int>(surv.size());
    STP_REQUIRE(nbs >= 1, "qpadm: no jackknife block survives (every block has partially missing pairs)");
    for (int s : bsz) STP_REQUIRE(s > 0, "qpadm: surviving blocks must have positive sizes");

    // ---- device arena: survivors, sizes, models ----
    std::vector<int> small, large;
    for (int i = 0; i < n_models; ++i) (fits_batched(shape[i].nl, shape[i].nr) ? small : large).push_back(i);
    std::vector<std::int32_t> arena;
    auto put = [&](const std::int32_t* p, std::size_t n) {
        const std::size_t off = arena.size();
        arena.insert(arena.end(), p, p + n);
        return off;
    };
    const std::size_t o_surv = put(surv.data(), surv.size());
    const std::size_t o_bsz = put(bsz.data(), bsz.size());
    const std::size_t o_tgt = put(target, n_models);
    const std::size_t o_left = put(left, total_left);
    const std::size_t o_right = put(right, total_right);
    qp_i32_.ensure(arena.size());
    STP_HIP(hipMemcpyAsync(qp_i32_.get(), arena.data(), arena.size() * sizeof(std::int32_t), hipMemcpyHostToDevice,
                           stream_));

    // ---- survivor-transposed f2 ----
    qpT_.ensure(static_cast<std::size_t>(slab) * nbs);
    launch_transpose_survivors(h.f2.get(), slab, qp_i32_.get() + o_surv, nbs, qpT_.get(), stream_);

    // ---- the fits ----
    qp_out_.ensure(static_cast<std::size_t>(n_models));
    STP_HIP(hipMemsetAsync(qp_out_.get(), 0, static_cast<std::size_t>(n_models) * sizeof(stp_qpadm_result), stream_));
    mark_begin(kQpadm);
    auto model_of = [&](int mi) {
        QpLargeModel md{};
        md.mi = mi;
        md.l0 = left_off[mi];
        md.nl = shape[mi].nl;
        md.r0 = right_off[mi];
        md.nr = shape[mi].nr;
        md.m = md.nl * md.nr;
        md.rank = opt.rank < 0 ? md.nl - 1 : opt.rank;
        return md;
    };
    if (!small.empty()) {
        QpFitArgs a{};
        a.f2T = qpT_.get();
        a.bsz = qp_i32_.get() + o_bsz;
        a.P = P;
        a.nbs = nbs;
        a.n_total = n_total;
        a.target = qp_i32_.get() + o_tgt;
        a.left = qp_i32_.get() + o_left;
        a.right = qp_i32_.get() + o_right;
        a.fudge = opt.fudge;
        a.iters = opt.als_iterations;
        a.jackknife = opt.jackknife;
        a.se_require_p = opt.se_require_p;
        a.p_se_threshold = opt.p_se_threshold;
        std::vector<QpLargeModel> sm;
        for (int mi : small) sm.push_back(model_of(mi));
        qpadm_small(a, std::move(sm), opt);
    }
    if (!large.empty()) {
        QpLargeArgs a{};
        a.f2T = qpT_.get();
        a.bsz = qp_i32_.get() + o_bsz;
        a.P = P;
        a.nbs = nbs;
        a.n_total = n_total;
        a.target = qp_i32_.get() + o_tgt;
        a.left = qp_i32_.get() + o_left;
        a.right = qp_i32_.get() + o_right;
        a.out = qp_out_.get();
        a.fudge = opt.fudge;
        a.iters = opt.als_iterations;
        a.alpha = opt.rank_alpha;
        a.jackknife = opt.jackknife;
        a.se_require_p = opt.se_require_p;
        a.p_se_threshold = opt.p_se_threshold;
        std::vector<QpLargeModel> lm;
        for (int mi : large) lm.push_back(model_of(mi));
        qpadm_large(a, lm, opt.rank);
    }
    mark_end(kQpadm);
    STP_HIP(hipMemcpyAsync(out, qp_out_.get(), static_cast<std::size_t>(n_models) * sizeof(stp_qpadm_result),
                           hipMemcpyDeviceToHost, stream_));
    sync();
}

// Models whose fits hold a matrix row per lane: chunks of models whose setup results and
// refit weights fit a fixed budget, or what is free beside a large resident tensor; per chunk
// the models are ordered by kernel instance and each stage is one launch per instance.
void HipBackend::qpadm_small(QpFitArgs a, std::vector<QpLargeModel> models, const stp_qpadm_options& opt) {
    constexpr std::size_t kBudget = std::size_t{1} << 29;        // doubles (4 GiB): setup results and weights
    constexpr std::size_t kMaxChunk = 16384;                     // models
    const int nbs = a.nbs;
    // STEPPE_QPADM_REFITS=wave takes every refit with a wavefront a fit (tests).
    const char* form = std::getenv("STEPPE_QPADM_REFITS");
    const bool rows = !(form && std::strcmp(form, "wave") == 0);
    auto cls = [&](const QpLargeModel& md) {
        return rows && qpadm_rows_fit(md.nl, md.nr, md.rank, a.iters) ? qpadm_rows_class(md.nl, md.nr) : 0;
    };
    auto bucket = [&](const QpLargeModel& md) { return bucket_of(md.nl, md.nr, opt.rank); };
    // largest systems first: the launches that end in a few long fits come first
    std::stable_sort(models.begin(), models.end(), [&](const QpLargeModel& x, const QpLargeModel& y) {
        if (bucket(x) != bucket(y)) return bucket(x) > bucket(y);
        if (cls(x) != cls(y)) return cls(x) > cls(y);
        return x.m > y.m;
    });
    const bool refits = a.jackknife != 0 && nbs >= 2;
    const std::size_t weights = refits ? static_cast<std::size_t>(STP_QPADM_MAX_NL) * nbs : 0;   // of a model
    // Models per chunk; STEPPE_QPADM_CHUNK lowers it (tests).
    std::size_t max_chunk = kMaxChunk;
    if (const char* env = std::getenv("STEPPE_QPADM_CHUNK")) {
        const long long v = std::strtoll(env, nullptr, 10);
        if (v > 0) max_chunk = std::min<std::size_t>(max_chunk, static_cast<std::size_t>(v));
    }
    int m_max = 0;   // of the chunk
    auto reserve = [&](std::size_t i0, std::size_t i1) {
        std::size_t setup = 0;
        m_max = 0;
        for (std::size_t i = i0; i < i1; ++i) {
            models[i].base = static_cast<std::int64_t>(setup);
            setup += qp_setup_doubles(models[i].m, nbs);
            m_max = std::max(m_max, models[i].m);
        }
        try {
            ql_models_.ensure(i1 - i0);
            ql_tables_.ensure(i1 - i0);
            ql_setup_.ensure(setup);
            ql_wm_.ensure((i1 - i0) * weights);
        } catch (const OomError&) {
            if (i1 - i0 == 1) throw;
            (void)hipGetLastError();   // or the next launch's check would report it
            ql_setup_.release();
            ql_wm_.release();
            return false;
        }
        return true;
    };
    auto run = [&](std::size_t i0, std::size_t i1) {
        const int nm = static_cast<int>(i1 - i0);
        STP_HIP(hipMemcpyAsync(ql_models_.get(), models.data() + i0, nm * sizeof(QpLargeModel), hipMemcpyHostToDevice,
                               stream_));
        launch_zero_u32(reinterpret_cast<unsigned*>(ql_tables_.get()),
                        static_cast<int>(nm * sizeof(QpLargeTables) / sizeof(unsigned)), stream_);
        a.models = ql_models_.get();
        a.tables = ql_tables_.get();
        a.setup = ql_setup_.get();
        a.wm = ql_wm_.get();
        launch_qpadm_setup(a, nm, m_max, stream_);
        // runs of models that share a kernel instance
        auto runs = [&](auto key, auto launch) {
            for (int s = 0; s < nm;) {
                int e = s, mm = 0, nn = 0;
                for (; e < nm && key(models[i0 + e]) == key(models[i0 + s]); ++e) {
                    mm = std::max(mm, models[i0 + e].m);
                    nn = std::max(nn, models[i0 + e].nr);
                }
                QpFitArgs r = a;
                r.models += s;
                r.tables += s;
                r.slot0 = s;
                launch(r, models[i0 + s], e - s, mm, nn);
                s = e;
            }
        };
        // With standard errors for every model the refits wait for nothing in the fit tables,
        // which are few long fits: those run beside them on a second stream, and the records
        // wait for both: one model of 2 sources 577 -> 470 us, 1000 mixed models 166 -> 157 ms.
        // (A model whose main fit fails is then refitted for nothing.)
        a.all_refits = refits && a.jackknife == 2;
        Beside beside(a.all_refits ? side_stream() : nullptr, stream_, side_ev_);
        runs(bucket, [&](const QpFitArgs& r, const QpLargeModel& md, int n, int mm, int nn) {
            launch_qpadm_fits(bucket(md), r, false, n, mm, nn, beside.stream());
        });
        if (refits)
            runs([&](const QpLargeModel& md) { return 128 * bucket(md) + cls(md); },
                 [&](const QpFitArgs& r, const QpLargeModel& md, int n, int mm, int nn) {
                     if (cls(md)) launch_qpadm_rows(r, cls(md), n, mm, stream_);
                     else launch_qpadm_fits(bucket(md), r, true, n, mm, nn, stream_);
                 });
        beside.join();
        launch_qpadm_finish(a, nm, opt.rank_alpha, qp_out_.get(), stream_);
        sync();   // the models (host memory) must outlive their copy, the buffers this chunk
    };
    for_chunks(
        models.size(), max_chunk, kBudget,
        [&](std::size_t i) { return qp_setup_doubles(models[i].m, nbs) + weights; }, reserve, run);
}

// Models beyond the batched kernel: chunks of models whose setup scratch fits a fixed
// budget; per chunk the setup kernel, the fit-table fits, the leave-one-block-out refits
// and the record kernel, each one launch.
void HipBackend::qpadm_large(QpLargeArgs a, const std::vector<QpLargeModel>& large, int rank_opt) {
    constexpr std::size_t kSetupBudget = std::size_t{1} << 29;   // doubles (4 GiB)
    constexpr std::size_t kFitBudget = std::size_t{1} << 28;     // doubles (2 GiB)
    const int nbs = a.nbs;
    std::size_t i0 = 0;
    while (i0 < large.size()) {
        // ---- the chunk's models and their setup scratch ----
        std::vector<QpLargeModel> models;
        std::size_t setup = 0;
        int m_max = 0, nr_max = 0, t_max = 0;
        for (; i0 < large.size(); ++i0) {
            QpLargeModel md = large[i0];
            const int nl = md.nl, nr = md.nr, m = md.m;
            const std::size_t need = qpadm_large_setup_doubles(m, nbs);
            if (!models.empty() && (setup + need > kSetupBudget || models.size() >= 4096)) break;
            md.base = static_cast<std::int64_t>(setup);
            models.push_back(md);
            setup += need;
            m_max = std::max(m_max, m);
            nr_max = std::max(nr_max, nr);
            t_max = std::max(t_max, large_t(nl, nr, rank_opt));
        }
        const int nm = static_cast<int>(models.size());
        // ---- fit tasks: every model's fit table, then its leave-one-block-out refits ----
        std::vector<QpLargeTask> tasks;
        for (int sl = 0; sl < nm; ++sl) {
            const int nl = models[sl].nl, nr = models[sl].nr, rank = models[sl].rank;
            const int nrows = nl >= 2 ? nl + 1 : 1;
            for (int k = 0; k < nrows; ++k) {
                const int nlr = k == 0 ? nl : nl - 1;
                const int rmax = std::min(nlr, nr) - 1, rf = nlr - 1;
                for (int rr = 0; rr <= rmax; ++rr) tasks.push_back({sl, k, rr, -1});
                if (rf > rmax) tasks.push_back({sl, k, rf, -1});
                if (k == 0 && rank > rmax && rank != rf) tasks.push_back({sl, 0, rank, -1});
            }
        }
        const int n_table = static_cast<int>(tasks.size());
        if (a.jackknife != 0 && nbs >= 2)
            for (int sl = 0; sl < nm; ++sl)
                for (int b = 0; b < nbs; ++b) tasks.push_back({sl, 0, 0, b});
        const int n_loo = static_cast<int>(tasks.size()) - n_table;

        ql_models_.ensure(static_cast<std::size_t>(nm));
        STP_HIP(hipMemcpyAsync(ql_models_.get(), models.data(), nm * sizeof(QpLargeModel), hipMemcpyHostToDevice,
                               stream_));
        ql_tasks_.ensure(tasks.size());
        STP_HIP(hipMemcpyAsync(ql_tasks_.get(), tasks.data(), tasks.size() * sizeof(QpLargeTask),
                               hipMemcpyHostToDevice, stream_));
        ql_tables_.ensure(static_cast<std::size_t>(nm));
        launch_zero_u32(reinterpret_cast<unsigned*>(ql_tables_.get()),
                        static_cast<int>(nm * sizeof(QpLargeTables) / sizeof(unsigned)), stream_);
        ql_setup_.ensure(setup);
        ql_wm_.ensure(static_cast<std::size_t>(nm) * nbs * STP_QPADM_MAX_NL);
        const std::size_t per_wave = qpadm_large_fit_doubles(m_max, nr_max, t_max);
        const int waves_per_wg = qpadm_large_fit_waves();
        int n_wg = std::min<int>(2 * n_cu_, static_cast<int>(ceil_div(std::max(n_table, n_loo), waves_per_wg)));
        n_wg = std::max(1, std::min<int>(n_wg, static_cast<int>(kFitBudget / (per_wave * waves_per_wg))));
        ql_fit_.ensure(per_wave * waves_per_wg * n_wg);
        counter_.ensure(64);

        a.models = ql_models_.get();
        a.n_models = nm;
        a.tables = ql_tables_.get();
        a.setup = ql_setup_.get();
        a.fit = ql_fit_.get();
        a.fit_stride = static_cast<std::int64_t>(per_wave);
        a.m_max = m_max;
        a.nr_max = nr_max;
        a.t_max = t_max;
        a.wm = ql_wm_.get();
        a.counter = counter_.get() + 30;
        launch_qpadm_large_setup(a, stream_);
        a.tasks = ql_tasks_.get();
        a.n_tasks = n_table;
        launch_zero_u32(a.counter, 1, stream_);
        launch_qpadm_large_fits(a, n_wg, stream_);
        if (n_loo > 0) {
            a.tasks = ql_tasks_.get() + n_table;
            a.n_tasks = n_loo;
            launch_zero_u32(a.counter, 1, stream_);
            launch_qpadm_large_fits(a, n_wg, stream_);
        }
        QpFitArgs f{};
        f.models = a.models;
        f.tables = a.tables;
        f.nbs = nbs;
        f.wm = a.wm;
        f.jackknife = a.jackknife;
        f.se_require_p = a.se_require_p;
        f.p_se_threshold = a.p_se_threshold;
        launch_qpadm_finish(f, nm, a.alpha, a.out, stream_);
        // the chunk's task list (host memory) must outlive its copy
        sync();
    }
}

}  // namespace stp
