// Batched FP64 Newton solver for the synchronous fixpoints of Kuramoto-type power
// grids (swing / first-order load vertices, AntiSymmetric K*sin lines): one workgroup
// per grid, all grids in one launch.
//
// A state with omega = 0 is a fixpoint of the swing and load models iff
//     F_i(theta) = P_i + sum_j K_ij sin(theta_j - theta_i) = 0   for every vertex,
// the condition find_fixpoint solves through NonlinearSolve (initialization.jl:73-144).
// Jacobian: dF/dtheta = -L_w, the Laplacian with weights w_ij = K_ij cos(theta_j - theta_i),
// singular along the global phase.  Each Newton step solves L_w d = F (so theta + d
// is the Newton update) with Jacobi-preconditioned conjugate gradients on the
// mean-zero subspace, then backtracks (halving) until the max-norm of the scaled
// residual F_i / scale_i decreases.  Converged when max_i |F_i / scale_i| <= tol.
//
// Layout: the rows (a vertex's lines) are taken in order of decreasing length and stored in
// slices of 64, column by column: entry j of the slice's 64 rows is one contiguous column of
// 64, padded to the slice's longest row (a few per cent after the sort).  Every read of a
// column is one contiguous access of its wave, and all columns' reads are independent.  Rows that
// would widen their slice for the other 63 (hubs; long_row_count chooses) are stored apart, entries
// 64 j .. 64 j + 63 in one column, and a whole wave evaluates them, adding in order.
//
// Who does what: thread t sums the rows at positions t, t + 512, ... of that order and hands
// each result over through LDS to the thread that owns the vertex; vertices t, t + 512, ...
// belong to thread t in the caller's order.  Vector updates and all reductions run in that
// order, so a solve does not depend on how rows are stored.
//
// On chip: two vectors of the grid in LDS (theta or the CG search vector for the neighbour
// gathers, and the row results); the first columns' weights and neighbours in the LDS that is
// left (all of them up to about 2000 vertices), the other columns' in memory; the per-vertex CG
// vectors in registers (V vertices per thread).
//
// What bounds it: a CG iteration on 5000 vertices (30000 entries) is four block barriers and
// a gather of 8 random bytes per entry from LDS, between loads of the columns that are not
// in LDS whose latency two waves per SIMD hide in part: 8.4 us an iteration, vector units 41 %
// busy (450 vertices: 2.6 us).  With a row per thread read entry by entry it took 29 us.
// Whole solves of 256 grids of 500 to 5000 vertices: 59 -> 19 ms.  Sixteen waves (the upper
// eight only summing rows) were slower: 14.9 us, the 128 registers a wave then has spill.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include "nd_block.h"
#include "nd_internal.h"
#include "nd_math.h"

namespace {

constexpr int kWave = 64;
constexpr int kThreads = 512;
constexpr int kColBytes = kWave * (sizeof(double) + sizeof(uint16_t));   // one column in LDS

struct GridDesc {
    int32_t n, ncol;     // vertices, columns of all slices and long rows
    int32_t nlong, pad_; // long rows
    int64_t voff;        // vertex offset (theta, P, scale, perm)
    int64_t coff;        // column offset
    int64_t soff;        // slice offset
};

struct NewtonArgs {
    const GridDesc* grid;
    const int2* slice;       // per slice of 64 positions: {first column, columns}; then per long row: {first
                             // column, entries}
    const uint16_t* perm;    // vertex of each row position, the long rows' last
    const uint16_t* nbr;     // per entry: 8 x the neighbour (padding: 8 x the row's own vertex)
    const int32_t* slot_edge;// global edge index per entry, -1 for padding
    double* w;               // weight per entry (columns that do not fit LDS)
    double* theta;
    const double* P;
    const double* scale;
    const double* K;         // per edge
    nd_newton_stat* stats;   // original grid order
    const int32_t* order;    // launch position -> grid index
    double tol, cg_rtol, eta_max;
    int32_t max_newton, cg_maxiter;
    int32_t linearized, inexact;
    int32_t first, lds;      // dynamic LDS of the launch
};

using namespace nd;

// a / b from y = 1.0 / b, both correctly rounded: one correction of the rounded product
// a * y by its remainder gives the rounded quotient (Markstein 1990), with three operations
// in place of a division's dozen.  The same bits as a division where a, b, y and the quotient
// are normal numbers and the remainder does not underflow (|a| > 2^-960); not finite where y
// or the quotient overflows or b is infinite (the caller divides there).
__device__ __forceinline__ double quotient(double a, double b, double y) {
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

// A quotient that is not finite makes the sum rz = r . z not finite, so one test finds every z to be
// divided out
template <int V>
__device__ __forceinline__ double divide_out(double rz, const double (&r)[V], const double (&dg)[V], double (&z)[V]) {
    if (__builtin_expect(!(fabs(rz) <= 0x1.fffffffffffffp+1023), 0)) {
        rz = 0.0;
#pragma unroll
        for (int k = 0; k < V; ++k) {
            z[k] = r[k] / dg[k];
            rz += r[k] * z[k];
        }
    }
    return rz;
}

// acc + x of lane 0, + x of lane 1, ... of the first count lanes and of the others up to a multiple
// of 8, where x is 0
__device__ __forceinline__ double add_in_order(double acc, double x, int count) {
    const long long b = __double_as_longlong(x);
    const int lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
    for (int i = 0; i < count; i += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned l = static_cast<unsigned>(__builtin_amdgcn_readlane(lo, i + j));
            const unsigned h = static_cast<unsigned>(__builtin_amdgcn_readlane(hi, i + j));
            acc += __longlong_as_double((static_cast<long long>(h) << 32) | l);
        }
    }
    return acc;
}

// LONG: some grid of the launch has long rows (their code costs the others 2 to 3 %)
template <int V, bool LONG>
__global__ void __launch_bounds__(kThreads) k_newton(NewtonArgs a) {
    constexpr int T = kThreads, WPB = kThreads / kWave;
    const int t = static_cast<int>(threadIdx.x), lane = t & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(t / kWave);
    const int g = a.first + static_cast<int>(blockIdx.x);
    const GridDesc G = a.grid[g];
    const int n = G.n, nr = LONG ? n - G.nlong : n;   // nr: rows in slices
    extern __shared__ double sm[];
    double* buf = sm;                          // theta or the CG search vector
    double* rowv = buf + n;                    // row results: F, the Jacobi diagonal, L_w p
    BlockRedN<kThreads / kWave> red{rowv + n, 0, 32};
    // the first columns' weights and neighbours, as many as fit
    const int cols_lds = min((a.lds - 8 * (2 * n + 64)) / kColBytes, G.ncol);
    double* wl = rowv + n + 64 + lane;
    uint16_t* nl = reinterpret_cast<uint16_t*>(rowv + n + 64 + cols_lds * kWave) + lane;
    const int2* sl = a.slice + G.soff;
    const uint16_t* nb = a.nbr + G.coff * kWave + lane;
    const int32_t* se = a.slot_edge + G.coff * kWave + lane;
    double* wg = a.w + G.coff * kWave + lane;
    auto at = [&](int bytes) { return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(buf) + bytes); };

    for (int c = wv; c < cols_lds; c += WPB) nl[c * kWave] = nb[c * kWave];
    // slice k of this wave, kept on lane k: {first column, columns}, columns < 0 in memory
    static_assert(V <= kWave, "a slice per lane");
    int2 mine = make_int2(0, 0);
    if (lane < V && lane * T + wv * kWave < nr) mine = sl[lane * WPB + wv];
    if (mine.x + mine.y > cols_lds) mine.y = -mine.y;
    auto slice_of = [&](int k) {
        return make_int2(__builtin_amdgcn_readlane(mine.x, k), __builtin_amdgcn_readlane(mine.y, k));
    };
    // neighbours and weights of the columns c .. c + 3 of a slice, past its last column c1 that one
    auto fetch = [&](bool mem, int c, int c1, int (&jn)[4], double (&ws)[4]) {
        if (mem) {
#pragma unroll
            for (int u = 0; u < 4; ++u) jn[u] = nb[min(c + u, c1) * kWave];
#pragma unroll
            for (int u = 0; u < 4; ++u) ws[u] = wg[min(c + u, c1) * kWave];
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) jn[u] = nl[min(c + u, c1) * kWave];
#pragma unroll
            for (int u = 0; u < 4; ++u) ws[u] = wl[min(c + u, c1) * kWave];
        }
    };
    double* th = a.theta + G.voff;             // the accepted theta (read and written by its owners)
    double d[V], r[V], dg[V], dgi[V];
    int row[V];                                // vertex of the thread's rows, -1 beyond the last
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        row[k] = v < nr ? a.perm[G.voff + v] : -1;
        if (v < n) buf[v] = th[v];
    }
    __syncthreads();

    // term(column, weight, theta_j - theta_i) for the entries of the thread's row k, in row
    // order, at the theta in buf.  The next entry's loads are on their way meanwhile.
    auto row_terms = [&](int k, double own, auto term) {
        const int2 S = slice_of(k);
        const int c0 = S.x, nc = abs(S.y);
        int e1 = nc > 0 ? se[c0 * kWave] : -1;
        int j1 = nc > 0 ? nb[c0 * kWave] : 0;
        double k1 = e1 >= 0 ? a.K[e1] : 0.0;
#pragma unroll 1
        for (int j = 0; j < nc; ++j) {
            const int jn = j1;
            const double kv = k1;
            // padding adds 0 whatever the row's own angle is: a vertex without lines has no equation
            const bool pad = e1 < 0;
            if (j + 1 < nc) {
                e1 = se[(c0 + j + 1) * kWave];
                j1 = nb[(c0 + j + 1) * kWave];
                k1 = e1 >= 0 ? a.K[e1] : 0.0;
            }
            term(c0 + j, kv, pad ? 0.0 : at(jn) - own);
        }
    };

    // f(vertex, first column, entries) for the long rows of this wave, and the sum of a lane's
    // f(column) over a row's entries in order
    auto long_rows = [&](auto f) {
        if constexpr (!LONG) return;
        for (int j = wv; j < G.nlong; j += WPB) {
            const int2 S = sl[(nr + kWave - 1) / kWave + j];
            f(static_cast<int>(a.perm[G.voff + nr + j]), __builtin_amdgcn_readfirstlane(S.x), __builtin_amdgcn_readfirstlane(S.y));
        }
    };
    auto long_sum = [&](int c0, int len, auto f) {
        double acc = 0.0;
        for (int e = 0; e < len; e += kWave) {
            const double x = e + lane < len ? f(c0 + e / kWave) : 0.0;
            acc = add_in_order(acc, x, min(len - e, kWave));
        }
        return acc;
    };
    auto in_lds = [&](int c0, int len) { return c0 + (len + kWave - 1) / kWave <= cols_lds; };

    // F(theta) of every vertex into rowv, from the theta in buf; returns max |F/scale| over the
    // grid.  The library sin and cos, called out of line: a handful of evaluations per solve,
    // whose registers the CG loop needs.
    auto residual = [&]() {
        double m = 0.0;
        long_rows([&](int v, int c0, int len) {
            const double own = buf[v];
            const double acc = long_sum(c0, len, [&](int c) {
                const double kv = a.K[se[c * kWave]], D = at(nb[c * kWave]) - own;
                return a.linearized ? kv * D : kv * sin_far(D);
            });
            const double F = a.P[G.voff + v] + acc;
            if (lane == 0) rowv[v] = F;
            m = MaxNanOp{}(m, fabs(F / a.scale[G.voff + v]));
        });
#pragma unroll 1
        for (int k = 0; k < V; ++k) {
            if (k * T + wv * kWave >= nr) break;
            const int i = t + k * T;
            if (i < nr) {
                const int v = a.perm[G.voff + i];
                double acc = 0.0;
                if (a.linearized) row_terms(k, buf[v], [&](int, double kv, double D) { acc += kv * D; });
                else row_terms(k, buf[v], [&](int, double kv, double D) { acc += kv * sin_far(D); });
                const double F = a.P[G.voff + v] + acc;
                rowv[v] = F;
                m = MaxNanOp{}(m, fabs(F / a.scale[G.voff + v]));
            }
        }
        return red.max_nan(m);
    };

    double res = residual();
    int it = 0, cg_total = 0, retcode = 0;
    while (res > a.tol) {
        if (it >= a.max_newton) { retcode = 1; break; }
        ++it;
        double fmean = 0.0;
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int v = t + k * T;
            r[k] = v < n ? rowv[v] : 0.0;
            fmean += r[k];
        }
        fmean = red.sum(fmean) / n;                 // its barrier: rowv may be written again
        // weights and Jacobi diagonal at the current theta
        long_rows([&](int v, int c0, int len) {
            const double own = buf[v];
            const bool lds = in_lds(c0, len);
            const double dsum = long_sum(c0, len, [&](int c) {
                const double kv = a.K[se[c * kWave]], D = at(nb[c * kWave]) - own;
                const double ws = a.linearized ? kv : kv * cos_far(D);
                if (lds) wl[c * kWave] = ws;
                else wg[c * kWave] = ws;
                return ws;
            });
            if (lane == 0) rowv[v] = dsum > 0.0 ? dsum : 1.0;
        });
#pragma unroll 1
        for (int k = 0; k < V; ++k) {
            if (k * T + wv * kWave >= nr) break;
            const int i = t + k * T;
            if (i < nr) {
                const int v = a.perm[G.voff + i];
                double dsum = 0.0;
                const bool mem = slice_of(k).y < 0;
                row_terms(k, buf[v], [&](int c, double kv, double D) {
                    const double ws = a.linearized ? kv : kv * cos_far(D);
                    if (!mem) wl[c * kWave] = ws;
                    else wg[c * kWave] = ws;
                    dsum += ws;
                });
                rowv[v] = dsum > 0.0 ? dsum : 1.0;
            }
        }
        __syncthreads();
        // CG for L_w d = F, d mean-zero (F sums to zero when P is balanced)
        double rz = 0.0, rr0 = 0.0, z[V];
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int v = t + k * T;
            d[k] = 0.0;
            r[k] = v < n ? r[k] - fmean : 0.0;
            dg[k] = v < n ? rowv[v] : 1.0;
            dgi[k] = 1.0 / dg[k];
            z[k] = quotient(r[k], dg[k], dgi[k]);
            rz += r[k] * z[k];
            rr0 += r[k] * r[k];
        }
        rz = divide_out(rz, r, dg, z);
#pragma unroll
        for (int k = 0; k < V; ++k)
            if (t + k * T < n) buf[t + k * T] = z[k];
        red.sum2(rz, rr0);
        const double eta = a.inexact ? fmax(a.cg_rtol, fmin(a.eta_max, res)) : a.cg_rtol;
        const double stop2 = eta * eta * rr0;
        double rr = rr0;
        int cg = 0;
        while (rr > stop2 && cg < a.cg_maxiter) {
            ++cg;
            // L_w p of the thread's rows, two rows and four columns of each at a time: eight
            // neighbours and weights are on their way together.  Columns past a row's last
            // repeat it and are not added.
            long_rows([&](int v, int c0, int len) {
                const double own = buf[v];
                const bool lds = in_lds(c0, len);
                const double sum = long_sum(c0, len, [&](int c) {
                    const double ws = lds ? wl[c * kWave] : wg[c * kWave];
                    return ws * (own - at(lds ? nl[c * kWave] : nb[c * kWave]));
                });
                if (lane == 0) rowv[v] = sum;
            });
#pragma unroll
            for (int k = 0; k < V; k += 2) {
                if (k * T + wv * kWave < nr) {       // whole waves without rows do nothing
                    const int2 Sa = slice_of(k), Sb = slice_of(k + 1);    // empty beyond the last slice
                    const int na = abs(Sa.y), nb_ = abs(Sb.y), ca = Sa.x + na - 1, cb = Sb.x + nb_ - 1;
                    const double oa = buf[max(row[k], 0)], ob = buf[max(row[k + 1], 0)];
                    double sa = 0.0, sb = 0.0;
                    for (int j = 0; j < max(na, nb_); j += 4) {
                        int ja[4], jb[4];
                        double wa[4], wb[4], pa[4], pb[4];
                        if (j < na) fetch(Sa.y < 0, Sa.x + j, ca, ja, wa);
                        if (j < nb_) fetch(Sb.y < 0, Sb.x + j, cb, jb, wb);
                        if (j < na) {
#pragma unroll
                            for (int u = 0; u < 4; ++u) pa[u] = at(ja[u]);
                        }
                        if (j < nb_) {
#pragma unroll
                            for (int u = 0; u < 4; ++u) pb[u] = at(jb[u]);
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (j + u < na) sa += wa[u] * (oa - pa[u]);
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (j + u < nb_) sb += wb[u] * (ob - pb[u]);
                    }
                    if (row[k] >= 0) rowv[row[k]] = sa;
                    if (row[k + 1] >= 0) rowv[row[k + 1]] = sb;
                }
            }
            __syncthreads();
            double q[V], pi[V], pq = 0.0;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const int v = t + k * T;
                pi[k] = v < n ? buf[v] : 0.0;
                q[k] = v < n ? rowv[v] : 0.0;
                pq += pi[k] * q[k];
            }
            pq = red.sum(pq);
            const double alpha = rz / pq;
            double rzn = 0.0, rrn = 0.0;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                d[k] += alpha * pi[k];
                r[k] -= alpha * q[k];
                q[k] = quotient(r[k], dg[k], dgi[k]);
                rzn += r[k] * q[k];
                rrn += r[k] * r[k];
            }
            rzn = divide_out(rzn, r, dg, q);
            red.sum2(rzn, rrn);
            rr = rrn;
            const double beta = rzn / rz;
            rz = rzn;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const int v = t + k * T;
                pi[k] = q[k] + beta * pi[k];
                if (v < n) buf[v] = pi[k];
            }
            __syncthreads();
        }
        cg_total += cg;
        // backtracking on the residual max-norm
        double step = 1.0, nres = res;
        for (int ls = 0; ls < 30; ++ls) {
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const int v = t + k * T;
                if (v < n) buf[v] = th[v] + step * d[k];
            }
            __syncthreads();
            nres = residual();
            if (nres < res || ls == 29) break;
            step *= 0.5;
        }
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int v = t + k * T;
            if (v < n) th[v] = th[v] + step * d[k];
        }
        if (!(nres < res)) { res = nres; retcode = 2; break; }
        res = nres;
    }
    if (!(res == res)) retcode = 3;         // a NaN residual never counts as converged
    if (t == 0) {
        nd_newton_stat s;
        s.residual = res;
        s.newton_iters = it;
        s.cg_iters = cg_total;
        s.retcode = retcode;
        s.pad_ = 0;
        a.stats[a.order[g]] = s;
    }
}

// How many of a grid's rows, given by decreasing length, are long rows.  Modelled cost of a product
// in cycles: the wave with the widest slices, kColumn per column, and the long rows over 8 waves.
// Solves of 64 stars of 1500 / 5000 vertices: 7.5 / 28 ms with every row in a slice, 0.54 / 1.6 so (4.6 /
// 15.4 with a thread per row and nothing padded); 256 preferential attachment grids of 500 to 2000 / 2100
// to 5000 vertices: 1.96 / 4.3 ms, 0.98 / 1.7 (2.5 / 4.9).  A wide first slice also left no room in
// LDS for those after it.
constexpr int kLongRow = 32;        // no shorter row is one
int64_t long_row_count(const std::vector<int32_t>& len) {
    constexpr int64_t kColumn = 100, kRow = 300, kEntry = 25;
    const int64_t n = static_cast<int64_t>(len.size());
    int64_t best = 0, cost = INT64_MAX, rows = 0;
    for (int64_t m = 0; m <= n; ++m) {
        int64_t c = rows / (kThreads / kWave);
        for (int64_t i = m; i < n; i += kThreads) c += kColumn * len[static_cast<size_t>(i)];
        if (c < cost) {
            cost = c;
            best = m;
        }
        if (m == n || len[static_cast<size_t>(m)] <= kLongRow) break;
        rows += kRow + kEntry * len[static_cast<size_t>(m)];
    }
    return best;
}

int herr(hipError_t e, const char* w) {
    return e == hipSuccess ? ND_OK : nd::set_error(ND_ERR_DEVICE, "%s: %s", w, hipGetErrorString(e));
}

}  // namespace

struct nd_fixpoint {
    int device = 0;
    int32_t ngrid = 0;
    std::vector<GridDesc> grids;
    std::vector<int32_t> small, large;      // grid indices by class (V = 4 / V = 10)
    std::vector<void*> allocs;
    GridDesc* d_grid = nullptr;
    int2* d_slice = nullptr;
    uint16_t *d_perm = nullptr, *d_nb = nullptr;
    int32_t *d_se = nullptr, *d_order = nullptr;
    double* d_w = nullptr;
    int lds_max = 0;
    int32_t lds[2] = {0, 0};                // dynamic LDS of the two classes' launches
    bool has_long[2] = {false, false};      // whether a grid of the class has long rows
    int64_t total_vertices = 0, total_edges = 0;
    // the two size classes run on their own streams, forked from and joined back to the
    // caller's stream with events, so the large grids start while small ones still run
    hipStream_t cls_stream[2] = {};
    hipEvent_t ev_fork = nullptr, ev_join[2] = {};
    ~nd_fixpoint() {
        for (void* p : allocs) (void)hipFree(p);
        for (auto& x : cls_stream) if (x) (void)hipStreamDestroy(x);
        for (auto& x : ev_join) if (x) (void)hipEventDestroy(x);
        if (ev_fork) (void)hipEventDestroy(ev_fork);
    }
};

namespace {
template <typename T>
int upv(nd_fixpoint* f, const std::vector<T>& h, T** d) {
    *d = nullptr;
    if (h.empty()) return ND_OK;
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, h.size() * sizeof(T));
    if (e != hipSuccess) return nd::set_error(ND_ERR_ALLOC, "hipMalloc: %s", hipGetErrorString(e));
    f->allocs.push_back(p);
    e = hipMemcpy(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess) return herr(e, "hipMemcpy");
    *d = static_cast<T*>(p);
    return ND_OK;
}
}  // namespace

extern "C" {

int nd_fixpoint_create(int32_t ngrid, const int64_t* nv, const int64_t* ne, const int64_t* src, const int64_t* dst,
                       nd_fixpoint** out) {
    nd::clear_error();
    if (!out || ngrid < 1 || !nv || !ne) return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    *out = nullptr;
    nd_fixpoint* f = new (std::nothrow) nd_fixpoint;
    if (!f) return nd::set_error(ND_ERR_ALLOC, "allocation failed");
    (void)hipGetDevice(&f->device);
    f->ngrid = ngrid;
    int lds_max = 0;
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, f->device) != hipSuccess || lds_max <= 0)
        lds_max = 64 * 1024;
    f->lds_max = lds_max;
    std::vector<int2> slices;
    std::vector<uint16_t> perm, nb;
    std::vector<int32_t> sedge;
    int64_t voff = 0, eoff = 0;
    for (int32_t gi = 0; gi < ngrid; ++gi) {
        const int64_t n = nv[gi], m = ne[gi];
        if (n < 1 || n > 10 * kThreads || m < 0) {
            delete f;
            return nd::set_error(ND_ERR_UNSUPPORTED, "grid %d: %lld vertices (supported 1..%d)", gi, (long long)n, 10 * kThreads);
        }
        GridDesc G{};
        G.n = static_cast<int32_t>(n);
        G.voff = voff;
        G.coff = static_cast<int64_t>(nb.size()) / kWave;
        G.soff = static_cast<int64_t>(slices.size());
        std::vector<int32_t> deg(static_cast<size_t>(n) + 1, 0);
        for (int64_t e = 0; e < m; ++e) {
            const int64_t s = src[eoff + e] - 1, d = dst[eoff + e] - 1;
            if (s < 0 || s >= n || d < 0 || d >= n) { delete f; return nd::set_error(ND_ERR_ARGUMENT, "grid %d: bad edge", gi); }
            deg[s + 1]++;
            deg[d + 1]++;
        }
        for (int64_t v = 0; v < n; ++v) deg[v + 1] += deg[v];
        // rows by decreasing length (ties in vertex order), in slices of 64
        int32_t longest = 0;
        for (int64_t v = 0; v < n; ++v) longest = std::max(longest, deg[v + 1] - deg[v]);
        std::vector<int32_t> first(static_cast<size_t>(longest) + 2, 0), pos(static_cast<size_t>(n));
        for (int64_t v = 0; v < n; ++v) first[longest - (deg[v + 1] - deg[v]) + 1]++;
        for (size_t l = 1; l < first.size(); ++l) first[l] += first[l - 1];
        const size_t p0 = perm.size();
        perm.resize(p0 + static_cast<size_t>(n));
        for (int32_t v = 0; v < static_cast<int32_t>(n); ++v) {
            pos[v] = first[longest - (deg[v + 1] - deg[v])]++;
            perm[p0 + pos[v]] = static_cast<uint16_t>(v);
        }
        // the longest rows that are better off apart go behind the others
        std::vector<int32_t> len(static_cast<size_t>(n));
        for (size_t i = 0; i < len.size(); ++i) len[i] = deg[perm[p0 + i] + 1] - deg[perm[p0 + i]];
        const int32_t nlong = static_cast<int32_t>(long_row_count(len)), nr = static_cast<int32_t>(n) - nlong;
        std::rotate(perm.begin() + p0, perm.begin() + p0 + nlong, perm.end());
        for (int32_t i = 0; i < static_cast<int32_t>(n); ++i) pos[perm[p0 + i]] = i;
        int32_t col = 0;
        const size_t s0 = slices.size(), e0 = nb.size();
        for (int32_t i = 0; i < nr; i += kWave) {
            const int32_t v = perm[p0 + i], width = deg[v + 1] - deg[v];
            slices.push_back(make_int2(col, width));
            col += width;
        }
        const size_t l0 = slices.size();
        for (int32_t i = nr; i < static_cast<int32_t>(n); ++i) {
            const int32_t v = perm[p0 + i], entries = deg[v + 1] - deg[v];
            slices.push_back(make_int2(col, entries));
            col += (entries + kWave - 1) / kWave;
        }
        nb.resize(e0 + static_cast<size_t>(col) * kWave);
        sedge.resize(nb.size(), -1);
        for (size_t s = s0; s < l0; ++s)
            for (int32_t l = 0; l < kWave; ++l) {
                const size_t i = (s - s0) * kWave + l;
                const uint16_t own = static_cast<uint16_t>(8 * (i < static_cast<size_t>(nr) ? perm[p0 + i] : 0));
                for (int32_t j = 0; j < slices[s].y; ++j) nb[e0 + static_cast<size_t>(slices[s].x + j) * kWave + l] = own;
            }
        std::vector<int32_t> fill(static_cast<size_t>(n), 0);
        auto entry = [&](int64_t v, int64_t other, int64_t e) {
            const int32_t i = pos[v], f = fill[v]++;
            const size_t k = i < nr ? e0 + static_cast<size_t>(slices[s0 + i / kWave].x + f) * kWave + i % kWave
                                    : e0 + static_cast<size_t>(slices[l0 + i - nr].x) * kWave + f;
            nb[k] = static_cast<uint16_t>(8 * other);
            sedge[k] = static_cast<int32_t>(eoff + e);
        };
        for (int64_t e = 0; e < m; ++e) {
            const int64_t s = src[eoff + e] - 1, d = dst[eoff + e] - 1;
            entry(s, d, e);
            entry(d, s, e);
        }
        G.ncol = col;
        G.nlong = nlong;
        // the vectors, the reduction buffers and as many columns of weights as there is room for
        const int cls = n <= 4 * kThreads ? 0 : 1;
        f->has_long[cls] = f->has_long[cls] || nlong > 0;
        f->lds[cls] = std::max(f->lds[cls], static_cast<int32_t>(std::min<int64_t>(lds_max, 8 * (2 * n + 64) + static_cast<int64_t>(kColBytes) * col)));
        f->grids.push_back(G);
        (n <= 4 * kThreads ? f->small : f->large).push_back(gi);
        voff += n;
        eoff += m;
    }
    f->total_vertices = voff;
    f->total_edges = eoff;
    // one launch per class: order = small grids then large grids, each by decreasing size
    auto bysize = [&](std::vector<int32_t>& v) {
        std::sort(v.begin(), v.end(), [&](int32_t x, int32_t y) { return f->grids[x].n > f->grids[y].n; });
    };
    bysize(f->small);
    bysize(f->large);
    std::vector<GridDesc> ordered;
    for (int32_t x : f->small) ordered.push_back(f->grids[x]);
    for (int32_t x : f->large) ordered.push_back(f->grids[x]);
    std::vector<int32_t> order(f->small);
    order.insert(order.end(), f->large.begin(), f->large.end());
    int rc = upv(f, ordered, &f->d_grid);
    rc = rc ? rc : upv(f, order, &f->d_order);
    rc = rc ? rc : upv(f, slices, &f->d_slice);
    rc = rc ? rc : upv(f, perm, &f->d_perm);
    rc = rc ? rc : upv(f, nb, &f->d_nb);
    rc = rc ? rc : upv(f, sedge, &f->d_se);
    if (!rc && !nb.empty()) {
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, nb.size() * sizeof(double));
        if (e != hipSuccess) rc = nd::set_error(ND_ERR_ALLOC, "hipMalloc(w): %s", hipGetErrorString(e));
        else { f->allocs.push_back(p); f->d_w = static_cast<double*>(p); }
    }
    if (rc) { delete f; return rc; }
    *out = f;
    return ND_OK;
}

void nd_fixpoint_destroy(nd_fixpoint* f) { delete f; }

int nd_fixpoint_solve(nd_fixpoint* f, double* theta, const double* P, const double* scale, const double* K,
                      const nd_newton_opts* o, nd_newton_stat* stats, void* stream) {
    if (!f || !theta || !P || !scale || !o || !stats) return nd::set_error(ND_ERR_ARGUMENT, "NULL argument");
    if (f->total_edges > 0 && !K) return nd::set_error(ND_ERR_ARGUMENT, "NULL K");
    int dev = -1;
    (void)hipGetDevice(&dev);
    if (dev != f->device) return nd::set_error(ND_ERR_ARGUMENT, "solver lives on device %d", f->device);
    NewtonArgs a{};
    a.grid = f->d_grid;
    a.slice = f->d_slice;
    a.perm = f->d_perm;
    a.nbr = f->d_nb;
    a.slot_edge = f->d_se;
    a.w = f->d_w;
    a.theta = theta;
    a.P = P;
    a.scale = scale;
    a.K = K;
    a.stats = stats;
    a.order = f->d_order;
    a.tol = o->tol > 0 ? o->tol : 1e-10;
    a.cg_rtol = o->cg_rtol > 0 ? o->cg_rtol : 1e-12;
    a.eta_max = o->eta_max > 0 ? o->eta_max : 1e-2;
    a.max_newton = o->max_newton > 0 ? o->max_newton : 50;
    a.cg_maxiter = o->cg_maxiter > 0 ? o->cg_maxiter : 20000;
    a.linearized = o->linearized ? 1 : 0;
    a.inexact = o->inexact ? 1 : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t ns = f->small.size(), nl = f->large.size();
    int rc = ND_OK;
    if (!f->ev_fork) rc = herr(hipEventCreateWithFlags(&f->ev_fork, hipEventDisableTiming), "hipEventCreate");
    for (int c = 0; c < 2 && !rc; ++c) {
        if (!f->cls_stream[c]) rc = herr(hipStreamCreateWithFlags(&f->cls_stream[c], hipStreamNonBlocking), "hipStreamCreate");
        if (!rc && !f->ev_join[c]) rc = herr(hipEventCreateWithFlags(&f->ev_join[c], hipEventDisableTiming), "hipEventCreate");
    }
    if (rc) return rc;
    const auto small_kernel = f->has_long[0] ? k_newton<4, true> : k_newton<4, false>;
    const auto large_kernel = f->has_long[1] ? k_newton<10, true> : k_newton<10, false>;
    size_t lds_s = 0, lds_l = 0;
    if (ns) {
        lds_s = static_cast<size_t>(f->lds[0]);
        rc = herr(hipFuncSetAttribute(reinterpret_cast<const void*>(small_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds_s)), "hipFuncSetAttribute");
    }
    if (!rc && nl) {
        lds_l = static_cast<size_t>(f->lds[1]);
        rc = herr(hipFuncSetAttribute(reinterpret_cast<const void*>(large_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds_l)), "hipFuncSetAttribute");
    }
    rc = rc ? rc : herr(hipEventRecord(f->ev_fork, s), "hipEventRecord");
    if (rc) return rc;
    // large grids first: they take longest
    if (nl) {
        hipStream_t cs = f->cls_stream[1];
        rc = herr(hipStreamWaitEvent(cs, f->ev_fork, 0), "hipStreamWaitEvent");
        if (rc) return rc;
        a.first = static_cast<int32_t>(ns);
        a.lds = f->lds[1];
        hipLaunchKernelGGL(large_kernel, dim3(static_cast<unsigned>(nl)), dim3(kThreads), lds_l, cs, a);
        rc = herr(hipGetLastError(), "newton launch");
        rc = rc ? rc : herr(hipEventRecord(f->ev_join[1], cs), "hipEventRecord");
        rc = rc ? rc : herr(hipStreamWaitEvent(s, f->ev_join[1], 0), "hipStreamWaitEvent");
        if (rc) return rc;
    }
    if (ns) {
        hipStream_t cs = f->cls_stream[0];
        rc = herr(hipStreamWaitEvent(cs, f->ev_fork, 0), "hipStreamWaitEvent");
        if (rc) return rc;
        a.first = 0;
        a.lds = f->lds[0];
        hipLaunchKernelGGL(small_kernel, dim3(static_cast<unsigned>(ns)), dim3(kThreads), lds_s, cs, a);
        rc = herr(hipGetLastError(), "newton launch");
        rc = rc ? rc : herr(hipEventRecord(f->ev_join[0], cs), "hipEventRecord");
        rc = rc ? rc : herr(hipStreamWaitEvent(s, f->ev_join[0], 0), "hipStreamWaitEvent");
    }
    return rc;
}

}  // extern "C"
