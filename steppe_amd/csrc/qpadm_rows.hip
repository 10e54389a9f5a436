// steppe_amd/csrc/qpadm_rows.hip — leave-one-block-out qpAdm refits, one fit per group of 16
// or 8 lanes (four or eight fits per wavefront).
//
// A model with jackknife standard errors is refitted nb (hundreds of) times on the same
// Qinv: nearly all of a qpAdm call.  A fit is a chain of small systems (t = nl r and r nr
// unknowns); a wavefront that works on one fit with a matrix row per lane keeps t of its 64
// lanes and spends two lane reads per element of every elimination step.  Here lane j of a
// 16- or 8-lane group owns column j of the f4 matrix (right population j + 1) of one fit:
//
//   B-step  lane j holds the r rows (p, j) of the normal matrix in registers, so an element of
//           Qinv read from LDS serves every p, A is the same in all its lanes, and the
//           matrix is built without any exchange.
//   A-step  lane j forms W[(i, j), (i', p')] = sum_j' Qinv[(i, j), (i', j')] B[p', j'] and
//           leaves it in LDS; lane a then sums its rows of the normal matrix over j.
//   LU      the pivot (the largest entry, ties to the first row) by a 4- or 3-stage reduction
//           over the group; its owner writes the pivot row to LDS and every lane reads it.
//   Seed    one-sided Jacobi on the columns: the rotations of the (p, q) loops that share
//           p + q touch different columns and run at once, lane j with lane p + q - j.
//
// The estimator is als_fit's (qpadm.hip) operation for operation: the sums of a fit keep their
// order, products are rounded before they are added (no contraction), pivots and divisions are
// the same, so the refits are als_fit's to the bit, also for sources that can hardly be told
// apart (compared over all shapes, up to 500 blocks).  Only the seed's stopping sum is added
// per lane first: it falls by orders of magnitude from sweep to sweep, and where it met 1e-30
// to within its rounding the seed could take a sweep more or less.  (A form with eliminations that need no
// exchanges, contracted sums and Jacobi on the nl rows is twice as fast again, but its
// standard errors differ by the rounding that near-degenerate models magnify: 1e-5.)
//
// Bound by VALU issue (the eliminations' multiply-subtracts, a third of them on lanes past
// nr) and, for the small systems, by the pivot reductions.  On MI355X with 744 blocks: 1000
// models of 2-5 sources and 6-12 right populations 1,061 ms as a workgroup per model and a
// wavefront per fit, 165 ms so (the whole call; 204 ms with 16 lanes for every fit, which
// leaves half of them idle up to 8 columns); a rotation of 1330 models of 2-3 sources against
// 8 right populations 242 -> 31.5 ms (51; without the garbage collections of its 1330 result
// dicts, which add up to 45 ms to a call now and then); one model of 2 sources 43.5 -> 0.58 ms.  Columns
// padded to 6, 8, 10, 12 with straight-line sums instead of a test per column: the same time
// at 3 sources, 2.3 times slower at 5 (spills).

#include <climits>
#include <cmath>

#include "common.hpp"
#include "qpadm.hpp"
#include "qpadm_record.hpp"
#include "wave_linalg.hpp"

namespace stp {

namespace {

using namespace wl;

// Bodies over register arrays must be inlined however large they are, or the arrays go to
// scratch.
#define STP_INLINE __attribute__((always_inline))

constexpr int kWaves = 4;

__device__ inline double lane_perm(int byte_index, double v) {
    return __hiloint2double(__builtin_amdgcn_ds_bpermute(byte_index, __double2hiint(v)),
                            __builtin_amdgcn_ds_bpermute(byte_index, __double2loint(v)));
}

// Lanes a fit: eight where they hold its columns.
constexpr int lanes_of(int nr) { return nr <= 8 ? 8 : 16; }

template <int NL, int NR>
struct RowShape {
    static constexpr int G = lanes_of(NR), kFits = kWaves * 64 / G;   // lanes a fit, fits of a workgroup
    static constexpr int R = NL - 1, TA = NL * R, RA = (TA + G - 1) / G;
    // LDS doubles of a fit: W of one i' [R][m], y [m], B [R][NR], a pivot row with its
    // right-hand side
    static constexpr int kRow = (TA > NR * R ? TA : NR * R) + 2;
    static constexpr int slice(int m) { return (R + 1) * m + R * NR + kRow + (((R + 1) * m + R * NR + kRow) & 1); }
};

// (key, pos) of the larger key, the smaller position at equal keys.
template <int CTRL>
__device__ inline void best_stage(long long& key, int& pos) {
    const long long k2 = __double_as_longlong(dpp<CTRL>(__longlong_as_double(key)));
    const int p2 = __builtin_amdgcn_mov_dpp(pos, CTRL, 0xF, 0xF, true);
    const bool take = k2 > key || (k2 == key && p2 < pos);
    key = take ? k2 : key;
    pos = take ? p2 : pos;
}

// LU solve with partial pivoting of one system per group of G lanes, as lu_solve_rows: each
// lane holds ROWS matrix rows (M, right-hand side b, logical position pos; -1 for a row that
// is none).  Storage column c is unknown order(c) when it is one of the system's (order
// ascending with c, the same in all lanes; negative otherwise).  buf: COLS + 2 doubles of the
// fit's LDS, 16-byte aligned.  found(c, x) receives each unknown in every lane; false for an
// exactly zero pivot.
template <int G, int ROWS, int COLS, class Order, class Found>
__device__ __forceinline__ bool row_solve(double (&M)[ROWS][COLS], double (&b)[ROWS], int (&pos)[ROWS], double* buf,
                                          Order&& order, Found&& found) {
    bool ok = true;
    static_for<COLS>([&](auto kc) STP_INLINE {
        constexpr int k = decltype(kc)::value;
        const int kk = order(kc);
        if (kk >= 0) {
            long long key = -1;
            int at = INT_MAX;
#pragma unroll
            for (int p = 0; p < ROWS; ++p) {
                const long long mine = pos[p] >= kk ? __double_as_longlong(fabs(M[p][k])) : -1;
                const bool take = mine > key || (mine == key && pos[p] < at);
                key = take ? mine : key;
                at = take ? pos[p] : at;
            }
            if constexpr (G == 16) best_stage<kRowMirror>(key, at);
            best_stage<kHalfMirror>(key, at);
            best_stage<kQuadMirror>(key, at);
            best_stage<kQuadSwap>(key, at);
            ok = ok && key != 0;
            constexpr int k0 = k & ~1;
#pragma unroll
            for (int p = 0; p < ROWS; ++p) {
                if (pos[p] == at) {
#pragma unroll
                    for (int c = k0; c < COLS; c += 2)
                        *reinterpret_cast<double2*>(buf + c) =
                            double2{M[p][c], c + 1 < COLS ? M[p][c + 1 < COLS ? c + 1 : c] : 0.0};
                    buf[COLS + (COLS & 1)] = b[p];
                }
                pos[p] = pos[p] == at ? kk : (pos[p] == kk ? at : pos[p]);
            }
            __builtin_amdgcn_wave_barrier();
            const double rp = 1.0 / buf[k], bk = buf[COLS + (COLS & 1)];
            double f[ROWS];
#pragma unroll
            for (int p = 0; p < ROWS; ++p) {
                f[p] = pos[p] > kk ? M[p][k] * rp : 0.0;
                b[p] -= f[p] * bk;
            }
            static_for<COLS - 1 - k>([&](auto cc) STP_INLINE {
                constexpr int c = k + 1 + decltype(cc)::value;
                if (order(std::integral_constant<int, c>{}) >= 0) {
                    const double u = buf[c];
#pragma unroll
                    for (int p = 0; p < ROWS; ++p) M[p][c] -= f[p] * u;
                }
            });
            __builtin_amdgcn_wave_barrier();
        }
    });
    static_for<COLS>([&](auto kc) STP_INLINE {
        constexpr int k = COLS - 1 - decltype(kc)::value;
        const std::integral_constant<int, k> ck{};
        const int kk = order(ck);
        if (kk >= 0) {
            double bs = b[0], us = M[0][k];
            bool own = pos[0] == kk;
#pragma unroll
            for (int p = 1; p < ROWS; ++p) {
                const bool me = pos[p] == kk;
                double bp = b[p], up = M[p][k];
                asm("" : "+v"(bp), "+v"(up));   // select values, not addresses (which would put M in scratch)
                bs = me ? bp : bs;
                us = me ? up : us;
                own = own || me;
            }
            const double xo = bs / us;
            if (own) buf[0] = xo;
            __builtin_amdgcn_wave_barrier();
            const double x = buf[0];
            __builtin_amdgcn_wave_barrier();
            found(ck, x);
#pragma unroll
            for (int p = 0; p < ROWS; ++p) {
                const double nb = b[p] - M[p][k] * x;
                b[p] = pos[p] < kk ? nb : b[p];
            }
        }
    });
    return ok;
}

// One fit in each group of lanes: x[i] is the f4 entry (i, lane), Q the model's Qinv in LDS
// (leading dimension ldq), sl the fit's slice of LDS.  Lanes past nr run on row 0's values,
// hold no matrix row and are never read.  Returns ok; w is the same in the
// group's lanes.
template <int NL, int NR>
__device__ __forceinline__ bool row_fit(const double* Q, int ldq, int nr, int iters, double fudge,
                                        const double (&x)[NL], double* sl, double (&w)[NL]) {
    using S = RowShape<NL, NR>;
    constexpr int G = S::G, R = S::R, TA = S::TA, RA = S::RA;
    const int j = lane_id() & (G - 1);
    const bool act = j < nr;
    const int ja = act ? j : 0;
    const double* Qj = Q + ja * ldq;   // row (0, j); row (i, j) is i * nr * ldq further
    const int qi = nr * ldq, m = NL * nr;
    double* const sW = sl + ((S::kRow + 1) & ~1);
    double* const sY = sW + R * m;
    double* const sB = sY + m;

    // y = Qinv^T x at (i, j)
    double y[NL] = {};
#pragma unroll
    for (int ii = 0; ii < NL; ++ii)
        static_for<NR>([&](auto jc) STP_INLINE {
            constexpr int jj = decltype(jc)::value;
            if (jj < nr) {
                const double xv = group_bcast<G, jj>(x[ii]);
                const double* q = Q + ii * qi + jj * ldq + ja;
#pragma unroll
                for (int i = 0; i < NL; ++i) y[i] += q[i * nr] * xv;
            }
        });
    if (act)
#pragma unroll
        for (int i = 0; i < NL; ++i) sY[i * nr + j] = y[i];

    // ---- seed: one-sided Jacobi SVD on the columns of x, lane j holding column j ----
    double B[R];
    {
        double ws[NL], V[NR];
#pragma unroll
        for (int i = 0; i < NL; ++i) ws[i] = x[i];
#pragma unroll
        for (int e = 0; e < NR; ++e) V[e] = e == j ? 1.0 : 0.0;
        bool done = false;
        const int lane0 = lane_id() & ~(G - 1);
        for (int sweep = 0; sweep < 60 && __ballot(!done); ++sweep) {
            double off = 0.0;
            for (int s = 1; s <= 2 * nr - 3; ++s) {
                const int o = s - j;
                const bool pair = act && o >= 0 && o < nr && o != j, low = j < o;
                const int from = 4 * (lane0 + (pair ? o : j));
                double ot[NL], al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
                for (int i = 0; i < NL; ++i) {
                    ot[i] = lane_perm(from, ws[i]);
                    const double wp = low ? ws[i] : ot[i], wq = low ? ot[i] : ws[i];
                    al += wp * wp;
                    be += wq * wq;
                    ga += wp * wq;
                }
                if (pair && low) off += ga * ga;
                const bool rot = pair && !done && !(fabs(ga) <= 1e-15 * sqrt(al * be) || ga == 0.0);
                if (__ballot(rot) == 0) continue;
                const double zeta = (be - al) / (2.0 * ga);
                const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
                const double c = 1.0 / sqrt(1.0 + t * t);
                const double sn = low ? -(c * t) : c * t;
#pragma unroll
                for (int i = 0; i < NL; ++i) {
                    const double v = c * ws[i] + sn * ot[i];
                    ws[i] = rot ? v : ws[i];
                }
#pragma unroll
                for (int e = 0; e < NR; ++e)
                    if (e < nr) {
                        const double v = c * V[e] + sn * lane_perm(from, V[e]);
                        V[e] = rot ? v : V[e];
                    }
            }
            done = done || group_sum<G>(off) < 1e-30;
        }
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < NL; ++i) ss += ws[i] * ws[i];
        const double sig = sqrt(ss);
        // exchange sort on descending sigma; positions 0..r-1 are final after r outer passes
        double sv[NR];
        int so[NR];
        static_for<NR>([&](auto ec) STP_INLINE {
            constexpr int e = decltype(ec)::value;
            sv[e] = group_bcast<G, e>(sig);
            so[e] = e;
        });
#pragma unroll
        for (int p = 0; p < R; ++p) {
            if constexpr (R <= NR) {
#pragma unroll
                for (int e = p + 1; e < NR; ++e)
                    if (e < nr) {
                        const bool sw = sv[e] > sv[p];
                        const double s1 = sv[e], s0 = sv[p];
                        const int o1 = so[e], o0 = so[p];
                        sv[p] = sw ? s1 : s0;
                        sv[e] = sw ? s0 : s1;
                        so[p] = sw ? o1 : o0;
                        so[e] = sw ? o0 : o1;
                    }
            }
            B[p] = 0.0;
#pragma unroll
            for (int e = 0; e < NR; ++e)
                if (e < nr) {
                    const double v = lane_perm(4 * (lane0 + so[p]), V[e]);
                    B[p] = e == j ? v : B[p];
                }
        }
    }

    double A[NL][R];
    for (int it = 0; it < iters; ++it) {
        // ---- A-step: unknowns A[i][p] at i R + p, lane a holding rows a, G + a, ... ----
        {
            double bb[R][NR];
            static_for<NR>([&](auto jc) STP_INLINE {
                constexpr int jj = decltype(jc)::value;
#pragma unroll
                for (int p = 0; p < R; ++p) bb[p][jj] = group_bcast<G, jj>(B[p]);
            });
            if (act)
#pragma unroll
                for (int p = 0; p < R; ++p) sB[p * NR + j] = B[p];
            __builtin_amdgcn_wave_barrier();
            double M[RA][TA], b[RA], bl[RA][NR], dg[RA];
            int pos[RA], ro[RA];
#pragma unroll
            for (int q = 0; q < RA; ++q) {
                const int a = j + G * q, ac = min(a, TA - 1), ia = ac / R, pa = ac - ia * R;
                pos[q] = a < TA ? a : -1;
                ro[q] = ia * nr;
                b[q] = 0.0;
                dg[q] = 0.0;
#pragma unroll
                for (int jj = 0; jj < NR; ++jj) bl[q][jj] = jj < nr ? sB[pa * NR + jj] : 0.0;
#pragma unroll
                for (int jj = 0; jj < NR; ++jj)
                    if (jj < nr) b[q] += bl[q][jj] * sY[ro[q] + jj];
            }
            static_for<NL>([&](auto ic) STP_INLINE {
                constexpr int i2 = decltype(ic)::value;
                double Z[NL][R] = {};
#pragma unroll
                for (int jj = 0; jj < NR; ++jj)
                    if (jj < nr) {
#pragma unroll
                        for (int i = 0; i < NL; ++i) {
                            const double q = Qj[i * qi + i2 * nr + jj];
#pragma unroll
                            for (int p = 0; p < R; ++p) Z[i][p] += q * bb[p][jj];
                        }
                    }
                if (act)
#pragma unroll
                    for (int p = 0; p < R; ++p)
#pragma unroll
                        for (int i = 0; i < NL; ++i) sW[p * m + i * nr + j] = Z[i][p];
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int q = 0; q < RA; ++q)
#pragma unroll
                    for (int p = 0; p < R; ++p) {
                        double s = 0.0;
#pragma unroll
                        for (int jj = 0; jj < NR; ++jj)
                            if (jj < nr) s += bl[q][jj] * sW[p * m + ro[q] + jj];
                        M[q][i2 * R + p] = s;
                        dg[q] = pos[q] == i2 * R + p ? s : dg[q];
                    }
                __builtin_amdgcn_wave_barrier();
            });
            double tr = 0.0;
            static_for<TA>([&](auto cc) STP_INLINE {
                constexpr int c = decltype(cc)::value;
                tr += group_bcast<G, c % G>(dg[c / G]);
            });
            const double ft = fudge * tr;
            static_for<TA>([&](auto cc) STP_INLINE {
                constexpr int c = decltype(cc)::value;
                const double v = M[c / G][c] + ft;
                M[c / G][c] = j == c % G ? v : M[c / G][c];
            });
            const bool ok = row_solve<G, RA, TA>(
                M, b, pos, sl, [](auto cc) STP_INLINE { return decltype(cc)::value; },
                [&](auto cc, double v) STP_INLINE {
                    constexpr int c = decltype(cc)::value;
                    A[c / R][c % R] = v;
                });
#pragma unroll
            for (int i = 0; i < NL; ++i)
#pragma unroll
                for (int p = 0; p < R; ++p) A[i][p] = ok ? A[i][p] : 0.0;
        }
        // ---- B-step: unknowns B[p][j] at p nr + j, lane j holding rows (p, j) ----
        {
            double M[R][R * NR], b[R], dg[R];
            int pos[R];
#pragma unroll
            for (int p = 0; p < R; ++p) {
                b[p] = 0.0;
#pragma unroll
                for (int i = 0; i < NL; ++i) b[p] += A[i][p] * y[i];
                pos[p] = act ? p * nr + j : -1;
                dg[p] = 0.0;
            }
            static_for<NR>([&](auto jc) STP_INLINE {
                constexpr int jj = decltype(jc)::value;
                if (jj < nr) {
                    double W[NL][R] = {};
#pragma unroll
                    for (int i2 = 0; i2 < NL; ++i2)
#pragma unroll
                        for (int i = 0; i < NL; ++i) {
                            const double q = Qj[i * qi + i2 * nr + jj];
#pragma unroll
                            for (int p2 = 0; p2 < R; ++p2) W[i][p2] += q * A[i2][p2];
                        }
#pragma unroll
                    for (int p = 0; p < R; ++p) {
#pragma unroll
                        for (int p2 = 0; p2 < R; ++p2) {
                            double s = 0.0;
#pragma unroll
                            for (int i = 0; i < NL; ++i) s += A[i][p] * W[i][p2];
                            M[p][p2 * NR + jj] = s;
                        }
                        dg[p] = j == jj ? M[p][p * NR + jj] : dg[p];
                    }
                } else {
#pragma unroll
                    for (int p = 0; p < R; ++p)
#pragma unroll
                        for (int p2 = 0; p2 < R; ++p2) M[p][p2 * NR + jj] = 0.0;
                }
            });
            double tr = 0.0;
#pragma unroll
            for (int p = 0; p < R; ++p)
                static_for<NR>([&](auto jc) STP_INLINE {
                    constexpr int jj = decltype(jc)::value;
                    if (jj < nr) tr += group_bcast<G, jj>(dg[p]);
                });
            const double ft = fudge * tr;
            static_for<NR>([&](auto jc) STP_INLINE {
                constexpr int jj = decltype(jc)::value;
#pragma unroll
                for (int p = 0; p < R; ++p) {
                    const double v = M[p][p * NR + jj] + ft;
                    M[p][p * NR + jj] = j == jj ? v : M[p][p * NR + jj];
                }
            });
            const bool ok = row_solve<G, R, R * NR>(
                M, b, pos, sl,
                [&](auto cc) STP_INLINE {
                    constexpr int c = decltype(cc)::value;
                    return c % NR < nr ? c / NR * nr + c % NR : -1;
                },
                [&](auto cc, double v) STP_INLINE {
                    constexpr int c = decltype(cc)::value;
                    B[c / NR] = j == c % NR ? v : B[c / NR];
                });
#pragma unroll
            for (int p = 0; p < R; ++p) B[p] = ok ? B[p] : 0.0;
        }
    }
    // ---- weights: (Xa Xa^T) w = Xa[:, r], Xa = [A, 1], normalised to sum 1 ----
    double M[1][NL], b[1] = {1.0};
    int pos[1] = {j < NL ? j : -1};
    double al[R];
#pragma unroll
    for (int p = 0; p < R; ++p) {
        al[p] = A[0][p];
#pragma unroll
        for (int i = 1; i < NL; ++i) al[p] = j == i ? A[i][p] : al[p];
    }
#pragma unroll
    for (int c = 0; c < NL; ++c) {
        double s = 0.0;
#pragma unroll
        for (int p = 0; p < R; ++p) s += al[p] * A[c][p];
        s += 1.0 * 1.0;
        M[0][c] = s;
    }
    const bool ok = row_solve<G, 1, NL>(
        M, b, pos, sl, [](auto cc) STP_INLINE { return decltype(cc)::value; },
        [&](auto cc, double v) STP_INLINE { w[decltype(cc)::value] = v; });
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < NL; ++i) sum += w[i];
#pragma unroll
    for (int i = 0; i < NL; ++i) w[i] = ok ? w[i] / sum : 0.0;
    return ok;
}

// Registers bound the wavefronts per SIMD: the B-step's normal matrix takes 2 r^2 NR of them
// per lane.
template <int NL, int NR>
constexpr int row_waves() {
    constexpr int regs = 2 * (NL - 1) * (NL - 1) * NR;
    return regs <= 32 ? 4 : regs <= 64 ? 3 : regs <= 130 ? 2 : 1;
}

// Workgroup (part, model): kFits consecutive blocks of one model.
template <int NL, int NR>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(row_waves<NL, NR>())))
void qpadm_rows_kernel(QpFitArgs g, int n_parts) {
    extern __shared__ __attribute__((aligned(16))) double lds[];
    const int tid = threadIdx.x;
    const int slot = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) / n_parts);
    const int part = static_cast<int>(blockIdx.x) - slot * n_parts;
    const QpLargeModel md = g.models[slot];
    const QpLargeTables* tb = g.tables + slot;
    if (!tb->cov_ok) return;
    const int nr = __builtin_amdgcn_readfirstlane(md.nr), m = NL * nr, nbs = g.nbs;
    const double* wmain = md.rank == NL - 1 ? tb->wrf[0] : tb->wmain;
    if (!g.all_refits && !qpadm_do_se(tb->ok[0][md.rank] != 0, nbs, g.jackknife, wmain, NL, g.se_require_p != 0,
                                      tb->chisq[0][md.rank], dof_of(NL, nr, md.rank), g.p_se_threshold))
        return;
    const QpSetup sp = qp_setup(g.setup, md, nbs);
    const int ldq = m | 1;
    for (int e = tid; e < m * m; e += 64 * kWaves) {
        const int a = e / m;
        lds[a * ldq + (e - a * m)] = sp.Qi[e];
    }
    __syncthreads();
    using S = RowShape<NL, NR>;
    const int fit = tid / S::G, j = tid & (S::G - 1);
    const int b = part * S::kFits + fit;
    if (__ballot(b < nbs) == 0) return;          // a wavefront past the last block
    double x[NL], w[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i)
        x[i] = sp.LOO[static_cast<std::int64_t>(i * nr + min(j, nr - 1)) * nbs + min(b, nbs - 1)];
    const int q_lds = (m * ldq + 1) & ~1;
    row_fit<NL, NR>(lds, ldq, nr, g.iters, g.fudge, x, lds + q_lds + fit * S::slice(m), w);
    if (b >= nbs) return;
    double* wm = g.wm + (static_cast<std::int64_t>(g.slot0 + slot) * nbs + b) * STP_QPADM_MAX_NL;
#pragma unroll
    for (int i = 0; i < NL; ++i)
        if (j == i) wm[i] = w[i];
}

}  // namespace

bool qpadm_rows_fit(int nl, int nr, int rank, int iters) {
    // the instances below; with no iterations the weights come from a seed of A that this
    // kernel does not form
    return nl >= 2 && nl <= 5 && nr <= 16 && rank == nl - 1 && iters >= 1;
}

int qpadm_rows_class(int nl, int nr) { return 8 * nl + (nr <= 8 ? 0 : nr <= 12 ? 1 : 2); }

template <int NL, int NR>
static void launch_rows(const QpFitArgs& g, int n_models, int m_max, hipStream_t st) {
    using S = RowShape<NL, NR>;
    const int n_parts = static_cast<int>(ceil_div(g.nbs, S::kFits));
    const std::size_t lds =
        (static_cast<std::size_t>((m_max * (m_max | 1) + 1) & ~1) + S::kFits * S::slice(m_max)) * sizeof(double);
    if (lds > 64 * 1024)
        STP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(qpadm_rows_kernel<NL, NR>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    qpadm_rows_kernel<NL, NR><<<static_cast<unsigned>(n_models * n_parts), 64 * kWaves, lds, st>>>(g, n_parts);
    STP_LAUNCH_CHECK();
}

void launch_qpadm_rows(const QpFitArgs& g, int cls, int n_models, int m_max, hipStream_t st) {
    if (n_models <= 0) return;
    switch (cls) {
        case 8 * 2: return launch_rows<2, 8>(g, n_models, m_max, st);
        case 8 * 2 + 1: return launch_rows<2, 12>(g, n_models, m_max, st);
        case 8 * 2 + 2: return launch_rows<2, 16>(g, n_models, m_max, st);
        case 8 * 3: return launch_rows<3, 8>(g, n_models, m_max, st);
        case 8 * 3 + 1: return launch_rows<3, 12>(g, n_models, m_max, st);
        case 8 * 3 + 2: return launch_rows<3, 16>(g, n_models, m_max, st);
        case 8 * 4: return launch_rows<4, 8>(g, n_models, m_max, st);
        case 8 * 4 + 1: return launch_rows<4, 12>(g, n_models, m_max, st);
        case 8 * 4 + 2: return launch_rows<4, 16>(g, n_models, m_max, st);
        case 8 * 5: return launch_rows<5, 8>(g, n_models, m_max, st);
        case 8 * 5 + 1: return launch_rows<5, 12>(g, n_models, m_max, st);
        default: throw ArgError("qpadm: unsupported row-fit class " + std::to_string(cls));
    }
}

}  // namespace stp
