// steppe_amd/csrc/qpadm.hpp — launch interface of the batched qpAdm kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "stp_qpadm_result.h"

namespace stp {

// Every model runs as four launches over all models of a call: setup (f4 basis, jackknife
// covariance and its inverse, a workgroup per model), the fit table (rank sweeps of the full
// model and of each popdrop row), the leave-one-block-out refits, and the record; so one
// model's refits spread over the whole device, and many models fill it.
//
// Model shape limits of the fits with one f4 entry per lane (m = nl*nr <= 64) and one
// normal-matrix row per lane (nl*r, r*nr <= 64).
constexpr int kMaxQpadmM = 64;
constexpr int kMaxQpadmNr = 32;

// ---- models beyond the batched kernel (qpadm_large.hip) -----------------------------
// Largest f4 basis (sources x (right - 1)), right set and normal system of the large path.
constexpr int kQpLargeMaxM = 1024;
constexpr int kQpLargeMaxNr = 128;
constexpr int kQpLargeMaxT = 1024;

struct QpLargeModel {
    int mi;                // model index (result record)
    int l0, nl, r0, nr;    // arena offsets and sizes (nr excludes the base)
    int m, rank;
    std::int64_t base;     // offset of the model's setup scratch (doubles)
};

// One fit of a large model: (popdrop row k, rank rr) of its fit table when b < 0, else
// the leave-one-block-out refit without surviving block b.
struct QpLargeTask {
    int slot, k, rr, b;
};

// Per-model fit tables (row k = 0 the full model, then each source dropped).
struct QpLargeTables {
    double chisq[STP_QPADM_MAX_NL + 1][STP_QPADM_MAX_NL + 1];
    int ok[STP_QPADM_MAX_NL + 1][STP_QPADM_MAX_NL + 1];
    double wrf[STP_QPADM_MAX_NL + 1][STP_QPADM_MAX_NL];
    double wmain[STP_QPADM_MAX_NL];
    int cov_ok, pad;
};

struct QpLargeArgs {
    const double* f2T = nullptr;
    const std::int32_t* bsz = nullptr;
    int P = 0, nbs = 0;
    double n_total = 0.0;
    const std::int32_t* target = nullptr;
    const std::int32_t* left = nullptr;
    const std::int32_t* right = nullptr;
    const QpLargeModel* models = nullptr;
    int n_models = 0;
    const QpLargeTask* tasks = nullptr;
    int n_tasks = 0;
    unsigned* counter = nullptr;
    QpLargeTables* tables = nullptr;
    double* setup = nullptr;       // per-model setup scratch
    double* fit = nullptr;         // per-wavefront fit scratch
    std::int64_t fit_stride = 0;
    int m_max = 0, nr_max = 0, t_max = 0;
    double* wm = nullptr;          // leave-one-block-out weights: slot s, block b at (s*nbs + b)*8
    stp_qpadm_result* out = nullptr;
    double fudge = 1e-4;
    int iters = 20;
    double alpha = 0.05;
    int jackknife = 2;
    int se_require_p = 0;
    double p_se_threshold = 0.05;
};

// ---- models within the limits above (qpadm.hip, qpadm_rows.hip) -----------------------
// QpLargeModel and QpLargeTables describe them too; models[0 .. n_models) of a launch share
// a kernel instance.  slot0 is the index of models[0] among the chunk's models.
struct QpFitArgs {
    const double* f2T = nullptr;
    const std::int32_t* bsz = nullptr;
    int P = 0, nbs = 0;
    double n_total = 0.0;
    const std::int32_t* target = nullptr;
    const std::int32_t* left = nullptr;
    const std::int32_t* right = nullptr;
    const QpLargeModel* models = nullptr;
    QpLargeTables* tables = nullptr;
    double* setup = nullptr;       // per-model setup results (qp_setup)
    double* wm = nullptr;          // leave-one-block-out weights: slot s, block b at (s*nbs + b)*8
    double fudge = 1e-4;
    int iters = 20;
    int jackknife = 2;             // 0 none, 1 feasible-only, 2 all
    int se_require_p = 0;
    double p_se_threshold = 0.05;
    int slot0 = 0;
    bool all_refits = false;       // refit every model: the fit tables may still be running
};

// A model's setup results: tau and the leave-one-out values [m][nbs], Qinv [m][m], totals.
struct QpSetup {
    double *X, *LOO, *Qi, *xtot, *totline;
};
__host__ __device__ inline QpSetup qp_setup(double* setup, const QpLargeModel& md, int nbs) {
    const std::int64_t mn = static_cast<std::int64_t>(md.m) * nbs;
    QpSetup p;
    p.X = setup + md.base;
    p.LOO = p.X + mn;
    p.Qi = p.LOO + mn;
    p.xtot = p.Qi + md.m * md.m;
    p.totline = p.xtot + md.m;
    return p;
}
inline std::size_t qp_setup_doubles(int m, int nbs) {
    return 2 * static_cast<std::size_t>(m) * nbs + static_cast<std::size_t>(m) * m + 2 * m;
}

void launch_qpadm_setup(const QpFitArgs& g, int n_models, int m_max, hipStream_t st);
// The fits of one system-size bucket T by wavefronts with a matrix row per lane: each
// model's fit table, or (refits) its leave-one-block-out refits.
void launch_qpadm_fits(int T, const QpFitArgs& g, bool refits, int n_models, int m_max, int nr_max, hipStream_t st);
// Leave-one-block-out refits with eight or sixteen lanes a fit: whether a model's take that
// form, the kernel instance, and the launch over models of one instance (g.models and g.tables
// at its first model, g.wm at the chunk's first).
bool qpadm_rows_fit(int nl, int nr, int rank, int iters);
int qpadm_rows_class(int nl, int nr);
void launch_qpadm_rows(const QpFitArgs& g, int cls, int n_models, int m_max, hipStream_t st);
// The result records, for models of either path.
void launch_qpadm_finish(const QpFitArgs& g, int n_models, double alpha, stp_qpadm_result* out, hipStream_t st);

std::size_t qpadm_large_setup_doubles(int m, int nbs);
std::size_t qpadm_large_fit_doubles(int m_max, int nr_max, int t_max);
int qpadm_large_fit_waves();
void launch_qpadm_large_setup(const QpLargeArgs& g, hipStream_t st);
void launch_qpadm_large_fits(const QpLargeArgs& g, int n_workgroups, hipStream_t st);

void launch_survivors(const double* vpair, std::int64_t slab, int n_block, std::int32_t* keep, hipStream_t st);
void launch_transpose_survivors(const double* f2, std::int64_t slab, const std::int32_t* surv, int nbs, double* f2T,
                                hipStream_t st);

}  // namespace stp
