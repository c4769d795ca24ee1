// Batched ensemble integrator: thousands of independent (uneven) networks, one
// workgroup per instance, whole trajectory in one launch per size class.
//
// Per instance everything a stage touches is on-chip:
//   registers  per-vertex state y and the Runge-Kutta stage derivatives (up to V
//              vertices per thread);
//   LDS        stage vertex outputs theta[n], edge parameters, the edge outputs in row order
//              (each vertex's entries consecutive, in whole pairs) and the edge table.
// A stage: write theta, barrier; evaluate each edge once, four consecutive ones per thread,
// and store its output at both endpoints' places in their rows, barrier; each vertex sums its
// row in the reference order (increasing output index), kChunk entries at a time, and applies
// its model.  Rows longer than kRowMax are summed by chunks spread over the block first.
//
// What bounds it: vector instruction issue.  One network of 1000 vertices and 4000 edges
// (first-order Kuramoto, RK4, 16 waves of one CU) takes 2.47 us per evaluation with the vector
// units 67 % busy and the LDS 60 %; with an index list per row entry, a bound on every entry
// and the longer sine it took 3.61 us.  1024 swing networks of 100 to 2000 vertices (Tsit5 to
// t = 10, default classes) take 39.1 ms, against 66.7 ms; at four vertices per thread the
// vector units are 60 % busy with two waves per SIMD.
//
// Methods: Tsit5 (Tsitouras 2011) with the PI step-size controller of
// OrdinaryDiffEq (beta1 = 7/50, beta2 = 2/25, qmin = 1/5, qmax = 10, gamma = 9/10,
// error norm sqrt(mean((err / (abstol + reltol*max(|y|,|ynew|)))^2))), and fixed-step
// classic RK4.  Step acceptance is block-uniform, so every wave leaves the loop
// together.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "nd_block.h"
#include "nd_internal.h"
#include "nd_models.h"

namespace {

using namespace nd;
constexpr int kWave = 64;
constexpr int kChunk = 8;          // destination-list entries summed together
constexpr int kRowMax = 16;        // longest row one thread sums by itself
constexpr uint32_t kRowHub = 0x80000000u;
constexpr int kSideStreams = 3;    // with the caller's stream, as many as a process has hardware queues
// Consecutive edges one thread evaluates together (their LDS reads and sines overlap, and
// table records and parameters are read 16 bytes at a time); the table is padded to a
// multiple of this with edges of no effect, so no lane of a batch needs a bound
constexpr int kEdgeBatch = 4;
// after an instance's row pairs: pairs that stay zero (read past a row's end) and one that the
// padding edges write to
constexpr int kZeroPairs = kRowMax / 2, kDumpPairs = 1;
__host__ __device__ constexpr int pad_edges(int ne) { return (ne + kEdgeBatch - 1) & ~(kEdgeBatch - 1); }
__host__ __device__ constexpr int pad2(int n) { return (n + 1) & ~1; }

// LDS of the crossing location: a second phase buffer and three bytes per edge, whole 16 bytes
__host__ __device__ constexpr int32_t locate_bytes(int32_t n, int32_t ne) { return (8 * n + 3 * ne + 15) & ~15; }

struct InstDesc {
    int32_t n, ne, nhc;           // vertices, edges, chunks of the rows longer than kRowMax
    int32_t npair;                // pairs of row entries, without the zeros and the dump
    int64_t uoff, poff, eoff, toff, voff, hoff;   // eoff: edges before this instance, toff: table records
    int32_t lds_bytes, tab_bytes; // dynamic LDS without the tables, and the tables'
    int32_t limit_bytes;          // the figure an instance's size is limited by (nd_ensemble_create)
    int32_t cls, vper;
};

struct SolveArgs {
    const InstDesc* inst;
    const int32_t* order;
    const uint2* tab;             // per edge, padded to a multiple of kEdgeBatch per instance: {src | dst << 16, row
                                  // position of the src entry | of the dst entry << 16}; src and dst in bytes of theta
    const uint32_t* row;          // per vertex: first pair of entries | pairs << 16, or for a row longer than kRowMax
                                  // kRowHub | first chunk | chunks << 16
    const uint32_t* hc;           // per chunk of the long rows: first pair of entries | pairs << 16
    int32_t lds_max;              // tab and hc go to LDS where they fit as well
    double* u;
    double* p;                    // written only where a line trips (line_limit set)
    const double* limit;          // per edge (instance order), or null: no line tripping
    const double* event_t;        // per instance: preset trip time, or null
    const int32_t* event_e;       // per instance: the edge it trips (local index, -1 none)
    nd_ensemble_stat* stats;
    double t0, t1, dt0, reltol, abstol, dtmax, dtmin;
    double ss_abstol, ss_reltol;  // steady-state termination (ss != 0)
    int64_t maxiters;
    int32_t first, count;
    int32_t ss;
};


// Dynamic LDS in this order (16-byte alignment up to the edge table): the vertex outputs, the
// edge outputs in row order, the edge parameters, the reduction buffers, the crossing
// location's arrays, the edge table (tab_lds), the long rows' chunk sums and chunks (tab_lds).
struct Lds {
    double* theta;
    double* fslot;                // edge outputs in row order: each vertex's entries are consecutive, in whole pairs
    double* epar;                 // padded with zeros to pad_edges
    BlockRed red;
    const uint2* tab;             // edge table in LDS, or
    const uint2* tab_g;           // in memory
    double* partial;              // sums of the long rows' chunks
    const uint32_t* hc;           // those chunks in LDS, or
    const uint32_t* hc_g;         // in memory
    uint32_t zero_pair;           // first of the pairs that stay zero
    bool tab_lds;                 // the tables are in LDS
};

// loads from the LDS or the memory copy of a table.  The typed pointers keep the two apart
// (a select of generic pointers would make both of them flat loads)
template <typename T>
__device__ __forceinline__ T table_load(bool lds, const void* l, const void* g, int i) {
    typedef const __attribute__((address_space(3))) T lds_t;
    typedef const __attribute__((address_space(1))) T mem_t;
    T r;
    if (lds) r = ((lds_t*)l)[i];
    else r = ((mem_t*)g)[i];
    return r;
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// the table records of the N consecutive edges from e (a multiple of N)
template <int N>
__device__ __forceinline__ void edge_recs(const Lds& L, int e, uint2 (&rec)[N]) {
    static_assert(N % 2 == 0, "records in pairs");
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const u32x4 r = table_load<u32x4>(L.tab_lds, L.tab, L.tab_g, e / 2 + i);
        rec[2 * i] = make_uint2(r.x, r.y);
        rec[2 * i + 1] = make_uint2(r.z, r.w);
    }
}
__device__ __forceinline__ uint2 edge_rec(const Lds& L, int e) {
    const u32x2 r = table_load<u32x2>(L.tab_lds, L.tab, L.tab_g, e);
    return make_uint2(r.x, r.y);
}
__device__ __forceinline__ double theta_at(const double* th, uint32_t bytes) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(th) + bytes);
}

// The same value, opaque to the optimiser (FRESH): what is derived from it is computed where it is
// used.  Otherwise every address derived from a thread's rows and index is kept in registers
// across the whole integration and spilled (100 registers at four vertices per thread)
template <bool FRESH, typename T>
__device__ __forceinline__ T fresh(T x) {
    if constexpr (FRESH) asm volatile("" : "+v"(x));
    return x;
}
// where registers are short; elsewhere keeping the addresses is 5 % faster
template <int V, int LB>
constexpr bool kFresh = V >= 3 || (V == 2 && LB > 512);

// the step controller's powers, out of line: inlined, their polynomial's constants occupy
// registers across the whole integration
__device__ __noinline__ double step_pow(double x, double y) { return pow(x, y); }
// x^a and y^b in one evaluation, on the even and the odd lanes of the wave
__device__ __forceinline__ void step_pow2(double x, double a, double y, double b, double& xa, double& yb) {
    const bool odd = threadIdx.x & 1;
    const double r = step_pow(odd ? y : x, odd ? b : a);
    xa = uniform_f64(r);
    yb = uniform_f64(dpp_f64<0xb1>(r));       // lane 0 reads lane 1
}

// A swing vertex multiplies by 1.0 / M: the quotient is formed once per solve (the same bits),
// kept in a register and passed in M's place
template <int VM>
constexpr bool kInverse0 = VM == ND_VM_SWING;
template <int VM>
__device__ __forceinline__ void vertex_f_inv(double* dx, const double* x, double acc, const double* pv) {
    if constexpr (kInverse0<VM>) {
        const double w = x[1];
        dx[0] = w;
        dx[1] = pv[0] * (pv[2] - pv[1] * w + acc);
    } else {
        vertex_f<VM>(dx, x, acc, pv, VModel<VM>::dim);
    }
}

// Vertex parameters stay in registers for the whole solve up to three vertices per
// thread; at four they are read from memory (L1/L2-resident) in each vertex update, which
// frees the registers whose spill would otherwise cost more
template <int V>
constexpr bool kParamsInMemory = V >= 4;

// fslot = the outputs of every edge at the state ys in row order, the src side negated
// (AntiSymmetric), N consecutive edges per thread at a time.  Two block barriers: after the vertex
// outputs and after the edges.  The first batch's table records and parameters do not depend on
// the state and are read before the first barrier.
template <int VM, int EM, int V, bool FRESH, int N>
__device__ __forceinline__ void edge_flows_n(const InstDesc& I, const Lds& L, const double (&ys)[V][VModel<VM>::dim]) {
    constexpr int NP = EModel<EM>::np;
    const int T = static_cast<int>(blockDim.x);
    const int t = fresh<FRESH>(static_cast<int>(threadIdx.x));
    uint2 rec[N];
    double pe[N][NP];
    auto load = [&](int e) {
        edge_recs<N>(L, e, rec);
        const double2* ep = reinterpret_cast<const double2*>(L.epar + e * NP);
#pragma unroll
        for (int i = 0; i < N * NP; i += 2) {
            const double2 x = ep[i / 2];
            pe[i / NP][i % NP] = x.x;
            pe[(i + 1) / NP][(i + 1) % NP] = x.y;
        }
    };
    const int ne = pad_edges(I.ne);
    int e = N * t;
    if (e < ne) load(e);
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        if (v < I.n) L.theta[v] = ys[k][0];
    }
    __syncthreads();
    while (e < ne) {
        double vs[N], vd[N], y[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            vs[i] = theta_at(L.theta, rec[i].x & 0xffff);
            vd[i] = theta_at(L.theta, rec[i].x >> 16);
        }
        g_dst_n<EM, N>(vs, vd, pe, y);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            L.fslot[rec[i].y & 0xffff] = -y[i];
            L.fslot[rec[i].y >> 16] = y[i];
        }
        e += N * T;
        if (e < ne) load(e);
    }
    __syncthreads();
}

// SMALL: two at a time where there are no more than two per thread, so that fewer threads idle while
// others have four.  1024 networks of 64 / 100 vertices, Tsit5 (128 threads): 673 / 731 us with four,
// 605 / 687 with two.  In kernels of their own, for launches a quarter of whose instances are so small: the
// second path costs the others up to 5 %.
template <int VM, int EM, int V, bool FRESH, bool SMALL>
__device__ __forceinline__ void edge_flows(const InstDesc& I, const Lds& L, const double (&ys)[V][VModel<VM>::dim]) {
    const int T = static_cast<int>(blockDim.x);
    if (SMALL && I.ne <= 2 * T) edge_flows_n<VM, EM, V, FRESH, 2>(I, L, ys);
    else edge_flows_n<VM, EM, V, FRESH, kEdgeBatch>(I, L, ys);
}

// the entries of pairs first .. first + N - 1 of a row; pairs past its end are the zeros (an
// address select in place of a bound on every entry)
template <int N>
__device__ __forceinline__ void row_read(const Lds& L, uint32_t start, int np, int first, double2 (&f)[N]) {
    const double2* fs = reinterpret_cast<const double2*>(L.fslot);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double2* base = fs + (first + i < np ? start : L.zero_pair);
        f[i] = base[first + i];
    }
}
template <int N>
__device__ __forceinline__ void row_add(const double2 (&f)[N], double& part) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        part += f[i].x;
        part += f[i].y;
    }
}

// out = f(ys) for the thread's vertices: each edge is evaluated once, then every vertex sums
// its own row in list order, kChunk entries at a time.  Rows longer than kRowMax (hubs) are
// summed by chunks spread over the block first, which takes a third barrier.  row: the
// thread's row words; pv: the vertex parameters in registers, or pg: the instance's vertex
// parameters in memory (kParamsInMemory)
template <int VM, int EM, int V, bool FRESH, bool SMALL>
__device__ __forceinline__ void rhs(const InstDesc& I, const Lds& L, const double (&ys)[V][VModel<VM>::dim],
                                    const double (&pv)[V][VPar<VM>::np > 0 ? VPar<VM>::np : 1],
                                    const double* __restrict__ pg, const uint32_t (&row_)[V],
                                    double (&out)[V][VModel<VM>::dim]) {
    const int T = static_cast<int>(blockDim.x);
    edge_flows<VM, EM, V, FRESH, SMALL>(I, L, ys);
    const int t = fresh<FRESH>(static_cast<int>(threadIdx.x));
    uint32_t row[V];
#pragma unroll
    for (int k = 0; k < V; ++k) row[k] = fresh<FRESH>(row_[k]);
    // parameters in memory: on their way while the rows are summed (read where they are used,
    // one vertex after the other, they cost four memory latencies per evaluation)
    constexpr int NPV = VPar<VM>::np > 0 ? VPar<VM>::np : 1;
    double pm[kParamsInMemory<V> ? V : 1][NPV];
    if constexpr (kParamsInMemory<V>) {
#pragma unroll
        for (int k = 0; k < V; ++k)
#pragma unroll
            for (int j = 0; j < VPar<VM>::np; ++j)
                pm[k][j] = kInverse0<VM> && j == 0 ? pv[k][0]
                                                   : pg[static_cast<int64_t>(min(t + k * T, I.n - 1)) * VPar<VM>::np + j];
    }
    constexpr int CP = kChunk / 2;
    for (int c = t; c < I.nhc; c += T) {
        const uint32_t h = table_load<uint32_t>(L.tab_lds, L.hc, L.hc_g, c);
        double2 f[CP];
        double part = 0.0;
        row_read<CP>(L, h & 0xffff, static_cast<int>(h >> 16), 0, f);
        row_add<CP>(f, part);
        L.partial[c] = part;
    }
    double acc[V];
    {
        double2 f[V][2];
#pragma unroll
        for (int k = 0; k < V; ++k)
            row_read<2>(L, row[k] & 0xffff, (row[k] & kRowHub) ? 0 : static_cast<int>(row[k] >> 16), 0, f[k]);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int np = (row[k] & kRowHub) ? 0 : static_cast<int>(row[k] >> 16);
            double part = 0.0;
            acc[k] = 0.0;
            row_add<2>(f[k], part);
            if (__any(np > 2)) {
                double2 g[2];
                row_read<2>(L, row[k] & 0xffff, np, 2, g);
                row_add<2>(g, part);
                if (__any(np > CP)) {
                    acc[k] += part;
                    part = 0.0;
                    double2 h[CP];
                    row_read<CP>(L, row[k] & 0xffff, np, CP, h);
                    row_add<CP>(h, part);
                }
            }
            acc[k] += part;
        }
    }
    if (I.nhc > 0) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < V; ++k)
            if (row[k] & kRowHub) {
                const int c0 = row[k] & 0xffff, nc = static_cast<int>((row[k] & ~kRowHub) >> 16);
                double a = 0.0;
                for (int c = 0; c < nc; c += 4) {
                    double f[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) f[j] = L.partial[c0 + min(c + j, nc - 1)];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (c + j < nc) a += f[j];
                }
                acc[k] = a;
            }
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        if (v < I.n) {
            if constexpr (kParamsInMemory<V>)
                vertex_f_inv<VM>(out[k], ys[k], acc[k], pm[k]);
            else
                vertex_f_inv<VM>(out[k], ys[k], acc[k], pv[k]);
        }
    }
}

// Line tripping (the component callback of the reference's cascading-failure example,
// docs/examples/cascading_failure.jl: condition |P_line| - limit, affect K = 0), checked
// at the end of every accepted step on the flows in fslot: a line whose |flow| exceeds
// its limit gets its first parameter set to 0, in LDS and in p.  Returns the number of
// lines tripped in this check (block-uniform).
template <int VM, int EM>
__device__ __forceinline__ int trip_lines(const SolveArgs& a, const InstDesc& I, Lds& L) {
    constexpr int NPE = EModel<EM>::np > 0 ? EModel<EM>::np : 1;
    const int T = static_cast<int>(blockDim.x), t = static_cast<int>(threadIdx.x);
    const double* lim = a.limit + I.eoff;
    double* pe_g = a.p + I.poff + static_cast<int64_t>(I.n) * VPar<VM>::np;
    double cnt = 0.0;
    for (int e = t; e < I.ne; e += T) {
        if (L.epar[e * NPE] != 0.0 && fabs(L.fslot[edge_rec(L, e).y >> 16]) > lim[e]) {
            L.epar[e * NPE] = 0.0;
            pe_g[static_cast<int64_t>(e) * NPE] = 0.0;
            cnt += 1.0;
        }
    }
    return static_cast<int>(L.red.sum(cnt));
}

// The preset-time trip of one edge (PresetTimeComponentCallback with the same affect):
// its first parameter goes to 0 in LDS and in p.  Returns 1 if it was not 0 before
// (block-uniform).
template <int VM, int EM>
__device__ __forceinline__ int trip_edge(const SolveArgs& a, const InstDesc& I, const Lds& L, int e) {
    constexpr int NPE = EModel<EM>::np > 0 ? EModel<EM>::np : 1;
    const bool was = L.epar[e * NPE] != 0.0;
    __syncthreads();
    if (threadIdx.x == 0) {
        L.epar[e * NPE] = 0.0;
        a.p[I.poff + static_cast<int64_t>(I.n) * VPar<VM>::np + static_cast<int64_t>(e) * NPE] = 0.0;
    }
    __syncthreads();
    return was ? 1 : 0;
}

// Steady-state test after an accepted step (the allDerivPass test of DiffEqCallbacks'
// TerminateSteadyState): every |du_i| <= ss_abstol or <= ss_reltol*|u_i|.  Block-uniform.
template <int V, int D>
__device__ __forceinline__ bool at_steady_state(const SolveArgs& a, const InstDesc& I, Lds& L,
                                                const double (&y)[V][D], const double (&du)[V][D]) {
    const int T = static_cast<int>(blockDim.x), t = static_cast<int>(threadIdx.x);
    double fail = 0.0;
#pragma unroll
    for (int q = 0; q < V; ++q)
        if (t + q * T < I.n)
#pragma unroll
            for (int j = 0; j < D; ++j) {
                const double d = fabs(du[q][j]);
                if (!(d <= a.ss_abstol || d <= a.ss_reltol * fabs(y[q][j]))) fail = 1.0;
            }
    return L.red.sum(fail) == 0.0;
}

// Line crossings (ND_LINES_CROSSING).  sign8 codes the sign of a condition value (2 for
// NaN, which never crosses); crossed(p, n) is the event test of DiffEqBase's
// VectorContinuousCallback when both directions have an affect: the sign p at the step
// start is nonzero and p*n <= 0.
__device__ __forceinline__ int8_t sign8(double g) {
    return static_cast<int8_t>(g > 0.0 ? 1 : g < 0.0 ? -1 : g == 0.0 ? 0 : 2);
}
__device__ __forceinline__ bool crossed(int8_t p, int8_t n) {
    return (p == -1 && (n == 1 || n == 0)) || (p == 1 && (n == -1 || n == 0));
}

// the condition |P_line| - limit of edge e (docs/examples/cascading_failure.jl:104-106)
// at the phases th
template <int EM>
__device__ __forceinline__ double line_cond(const Lds& L, const double* th, const double* lim, int e) {
    constexpr int NPE = EModel<EM>::np > 0 ? EModel<EM>::np : 1;
    const uint32_t ends = edge_rec(L, e).x;
    return fabs(g_dst<EM>(theta_at(th, ends & 0xffff), theta_at(th, ends >> 16), L.epar + e * NPE)) - lim[e];
}

// sg[e] = sign8 of every edge's condition at the state y (two block barriers)
template <int VM, int EM, int V, bool FRESH>
__device__ __forceinline__ void line_signs(const InstDesc& I, const Lds& L, const double* lim,
                                           const double (&y)[V][VModel<VM>::dim], int8_t* sg) {
    const int T = static_cast<int>(blockDim.x), t = fresh<FRESH>(static_cast<int>(threadIdx.x));
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        if (v < I.n) L.theta[v] = y[k][0];
    }
    __syncthreads();
    for (int e = t; e < I.ne; e += T) sg[e] = sign8(line_cond<EM>(L, L.theta, lim, e));
    __syncthreads();
}

// Tsitouras (2011) 5(4) coefficients: stage matrix a (row s = stage s+1), error weights
// btilde = b - bhat (b = the last row, first same as last) and nodes c = a * 1.  The
// kernel reads these names and nd_tsit5_tableau exports the same table, so the order
// conditions checked on the exported copy hold for the kernel's.
struct Tsit5Tableau {
    double a[7][6];
    double bt[7];
    double c[7];
};
constexpr Tsit5Tableau kTsit5 = {
    {{0, 0, 0, 0, 0, 0},
     {0.161, 0, 0, 0, 0, 0},
     {-0.008480655492356989, 0.335480655492357, 0, 0, 0, 0},
     {2.897153057105493, -6.359448489975075, 4.3622954328695815, 0, 0, 0},
     {5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525, 0, 0},
     {5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401, -0.028269050394068383, 0},
     {0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081, 2.324710524099774}},
    {-0.00178001105222577714, -0.0008164344596567469, 0.007880878010261995, -0.1447110071732629,
     0.5823571654525552, -0.45808210592918697, 0.015151515151515152},
    {0.0, 0.161, 0.327, 0.9, 0.9800255409045097, 1.0, 1.0}};
constexpr double c_a21 = kTsit5.a[1][0];
constexpr double c_a31 = kTsit5.a[2][0], c_a32 = kTsit5.a[2][1];
constexpr double c_a41 = kTsit5.a[3][0], c_a42 = kTsit5.a[3][1], c_a43 = kTsit5.a[3][2];
constexpr double c_a51 = kTsit5.a[4][0], c_a52 = kTsit5.a[4][1], c_a53 = kTsit5.a[4][2], c_a54 = kTsit5.a[4][3];
constexpr double c_a61 = kTsit5.a[5][0], c_a62 = kTsit5.a[5][1], c_a63 = kTsit5.a[5][2], c_a64 = kTsit5.a[5][3],
                 c_a65 = kTsit5.a[5][4];
constexpr double c_a71 = kTsit5.a[6][0], c_a72 = kTsit5.a[6][1], c_a73 = kTsit5.a[6][2], c_a74 = kTsit5.a[6][3],
                 c_a75 = kTsit5.a[6][4], c_a76 = kTsit5.a[6][5];
constexpr double c_bt1 = kTsit5.bt[0], c_bt2 = kTsit5.bt[1], c_bt3 = kTsit5.bt[2], c_bt4 = kTsit5.bt[3],
                 c_bt5 = kTsit5.bt[4], c_bt6 = kTsit5.bt[5], c_bt7 = kTsit5.bt[6];

// Tsitouras' continuous extension of the pair, the dense output OrdinaryDiffEqTsit5
// interpolates solutions and locates callback events on: u(t + s h) = u + h sum_i b_i(s) k_i,
// b_i(s) = sum_j r[i][j-1] s^j (only stage 1 has a linear term; b_i(1) is the last row of
// a).  nd_tsit5_dense exports this table, so its order conditions are checked on the
// kernel's copy.
struct Tsit5Dense {
    double r[7][4];
};
constexpr Tsit5Dense kTsit5Dense = {{{1.0, -2.763706197274826, 2.9132554618219126, -1.0530884977290216},
                                     {0.0, 0.13169999999999998, -0.2234, 0.1017},
                                     {0.0, 3.9302962368947516, -5.941033872131505, 2.490627285651253},
                                     {0.0, -12.411077166933676, 30.33818863028232, -16.548102889244902},
                                     {0.0, 37.50931341651104, -88.1789048947664, 47.37952196281928},
                                     {0.0, -27.896526289197286, 65.09189467479366, -34.8706578614966},
                                     {0.0, 1.5, -4.0, 2.5}}};
#define ND_R(i, j) kTsit5Dense.r[i - 1][j - 1]

// the dense output at s from the step's start value y0, first derivative k1 and the
// coefficients d_j = sum_i r_ij k_i of s^2, s^3, s^4
__device__ __forceinline__ double dense_at(double y0, double k1, double d2, double d3, double d4, double h, double s) {
    return y0 + h * (s * (k1 + s * (d2 + s * (d3 + s * d4))));
}

template <int VM, int EM, int METHOD, int V, int LB, bool FRESH>
__device__ __forceinline__ void ensemble_body(const SolveArgs& a, int inst, const InstDesc& I, double2* smem) {
    constexpr int D = VModel<VM>::dim;
    constexpr int NPV = VPar<VM>::np > 0 ? VPar<VM>::np : 1;
    constexpr int NPE = EModel<EM>::np;
    constexpr bool kSmall = LB <= 256 && V <= 2;
    const int T = static_cast<int>(blockDim.x), t = static_cast<int>(threadIdx.x);
    const int ne4 = pad_edges(I.ne);
    Lds L;
    L.theta = reinterpret_cast<double*>(smem);
    L.fslot = L.theta + pad2(I.n);
    L.zero_pair = static_cast<uint32_t>(I.npair);
    L.epar = L.fslot + 2 * (I.npair + kZeroPairs + kDumpPairs);
    L.red = BlockRed{L.epar + ne4 * NPE};
    double* locate = L.red.red + 32;             // METHOD 2: the crossing location's arrays
    constexpr bool kLocate = METHOD == 2;
    const int32_t extra = kLocate ? locate_bytes(I.n, I.ne) : 0;
    L.tab_lds = I.lds_bytes + extra + I.tab_bytes <= a.lds_max;
    uint2* tab = reinterpret_cast<uint2*>(reinterpret_cast<char*>(locate) + extra);
    L.partial = reinterpret_cast<double*>(tab + (L.tab_lds ? ne4 : 0));
    uint32_t* hc = reinterpret_cast<uint32_t*>(L.partial + I.nhc);
    L.tab = tab;
    L.tab_g = a.tab + I.toff;
    L.hc = hc;
    L.hc_g = a.hc + I.hoff;
    if (L.tab_lds) {
        for (int i = t; i < ne4; i += T) tab[i] = L.tab_g[i];
        for (int i = t; i < I.nhc; i += T) hc[i] = L.hc_g[i];
    }
    for (int i = t; i < 2 * (I.npair + kZeroPairs + kDumpPairs); i += T) L.fslot[i] = 0.0;
    const double* pe_g = a.p + I.poff + static_cast<int64_t>(I.n) * VPar<VM>::np;
    for (int i = t; i < ne4 * NPE; i += T) L.epar[i] = i < I.ne * NPE ? pe_g[i] : 0.0;

    double y[V][D], pv[V][NPV];
    uint32_t row[V];
    const double* pg = a.p + I.poff;                 // the instance's vertex parameters
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        row[k] = v < I.n ? a.row[I.voff + v] : 0;
#pragma unroll
        for (int j = 0; j < D; ++j) y[k][j] = v < I.n ? a.u[I.uoff + static_cast<int64_t>(v) * D + j] : 0.0;
#pragma unroll
        for (int j = 0; j < NPV; ++j)
            pv[k][j] = ((!kParamsInMemory<V> || (kInverse0<VM> && j == 0)) && v < I.n && VPar<VM>::np > 0)
                           ? a.p[I.poff + static_cast<int64_t>(v) * VPar<VM>::np + j] : 0.0;
        if constexpr (kInverse0<VM>) pv[k][0] = 1.0 / pv[k][0];
    }
    __syncthreads();

    double tcur = a.t0;
    int64_t naccept = 0, nreject = 0, nf = 0;
    int retcode = 0, ntrip = 0;
    // preset trip: fires once at te (t0 < te <= t1), else never
    double te = __builtin_inf();
    int32_t ee = -1;
    if (a.event_t) {
        te = a.event_t[inst];
        ee = a.event_e[inst];
        if (!(te > a.t0 && te <= a.t1) || ee < 0 || ee >= I.ne) {
            te = __builtin_inf();
            ee = -1;
        }
    }
    double dt = a.dt0;
    const double inv_len = 1.0 / (static_cast<double>(I.n) * D);

    // The right-hand side appears once in each method below, inside one loop over the
    // evaluations: with a copy per stage the Tsit5 loop's code, about 100 KB of nine copies,
    // exceeded the instruction cache.  (It saves no scalar registers: the Tsit5 kernels spill 147
    // to 199 of them, 67 to 104 with the copies.)
#define ND_EACH                                        \
    _Pragma("unroll") for (int q = 0; q < V; ++q)      \
        _Pragma("unroll") for (int j = 0; j < D; ++j)
    double ys[V][D], k[V][D];
    if constexpr (METHOD == 1) {
        // fixed-step classic RK4: u + dt/6*(((k1 + 2k2) + 2k3) + k4)
        double acc[V][D];
        const int64_t nsteps = static_cast<int64_t>(llround((a.t1 - a.t0) / dt));
        const double half = 0.5 * dt, sixth = dt / 6.0;
        int64_t done = nsteps;
        ND_EACH { ys[q][j] = y[q][j]; acc[q][j] = 0.0; }
        int stage = 0;                              // 0..3, 4: the steady-state check's evaluation
        for (int64_t step = 0; step < nsteps;) {
            rhs<VM, EM, V, FRESH, kSmall>(I, L, ys, pv, pg, row, k);
            ++nf;
            if (stage < 3) {
                const double hs = stage == 2 ? dt : half;
                if (stage == 0) ND_EACH acc[q][j] = k[q][j];
                else ND_EACH acc[q][j] = acc[q][j] + 2.0 * k[q][j];
                ND_EACH ys[q][j] = y[q][j] + hs * k[q][j];
                ++stage;
                continue;
            }
            if (stage == 3) {
                ND_EACH { y[q][j] = y[q][j] + sixth * (acc[q][j] + k[q][j]); ys[q][j] = y[q][j]; }
                ++naccept;
                if (a.limit) {
                    edge_flows<VM, EM, V, FRESH, kSmall>(I, L, y);
                    ntrip += trip_lines<VM, EM>(a, I, L);
                }
                if (ee >= 0 && step + 1 == static_cast<int64_t>(llround((te - a.t0) / dt))) ntrip += trip_edge<VM, EM>(a, I, L, ee);
                if (a.ss) {
                    stage = 4;
                    continue;
                }
            } else if (at_steady_state<V, D>(a, I, L, y, k)) {
                done = step + 1;
                retcode = 4;
                break;
            }
            stage = 0;
            ++step;
        }
        tcur = a.t0 + static_cast<double>(done) * dt;
    } else {
        // k3..k5 hold the dense-output coefficients d2..d4 over the first six stages once the last
        // evaluation has begun (crossing location), k2 the error estimate's sum over the first six stages
        double k1[V][D], k2[V][D], k3[V][D], k4[V][D], k5[V][D], k6[V][D];
        auto &d2 = k3, &d3 = k4, &d4 = k5;
        ND_EACH { ys[q][j] = y[q][j]; k1[q][j] = k2[q][j] = k3[q][j] = k4[q][j] = k5[q][j] = k6[q][j] = 0.0; }
        auto wnorm2 = [&](const double (&x)[V][D], const double (&ref)[V][D]) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < V; ++q)
                if (t + q * T < I.n)
#pragma unroll
                    for (int j = 0; j < D; ++j) {
                        const double sc = a.abstol + fabs(ref[q][j]) * a.reltol;
                        const double r = x[q][j] / sc;
                        s += r * r;
                    }
            return L.red.sum(s);
        };
        double qold = 1e-4, d1 = 0.0, h = 0.0;
        int64_t iters = 0;
        double tstop = ee >= 0 ? te : a.t1;       // the next time a step must end on
        bool last = false;
        // crossing location: a second phase buffer and, per edge, the condition's sign at
        // the step start (gsign) and end (gnext) and the first point of the step where it
        // crossed (gev), in LDS after the reduction buffers
        const double* lim = a.limit ? a.limit + I.eoff : nullptr;
        double* theta2 = nullptr;
        int8_t *gsign = nullptr, *gnext = nullptr, *gev = nullptr;
        if constexpr (kLocate) {
            theta2 = locate;
            gsign = reinterpret_cast<int8_t*>(theta2 + I.n);
            gnext = gsign + I.ne;
            gev = gnext + I.ne;
        }
        // what the evaluation at ys is: 0 the first derivative, 1..6 the step's stages 2..7,
        // 7 the initial step's probe, 8 the first derivative again after a trip
        int phase = 0;
        for (;;) {
            rhs<VM, EM, V, FRESH, kSmall>(I, L, ys, pv, pg, row, k);
            ++nf;
            bool accepted = false, begun = true;
            if (phase >= 1 && phase <= 5) {
                // stage derivative k_{phase+1}, then the next stage's state
#define ND_STAGE(kn, expr)                                                   \
    ND_EACH {                                                                \
        kn[q][j] = k[q][j];                                                  \
        ys[q][j] = y[q][j] + h * (expr);                                     \
    }
                if (phase == 1) {
                    ND_STAGE(k2, c_a31 * k1[q][j] + c_a32 * k2[q][j])
                } else if (phase == 2) {
                    ND_STAGE(k3, c_a41 * k1[q][j] + c_a42 * k2[q][j] + c_a43 * k3[q][j])
                } else if (phase == 3) {
                    ND_STAGE(k4, c_a51 * k1[q][j] + c_a52 * k2[q][j] + c_a53 * k3[q][j] + c_a54 * k4[q][j])
                } else if (phase == 4) {
                    ND_STAGE(k5, c_a61 * k1[q][j] + c_a62 * k2[q][j] + c_a63 * k3[q][j] + c_a64 * k4[q][j] +
                                     c_a65 * k5[q][j])
                } else {
                    ND_STAGE(k6, c_a71 * k1[q][j] + c_a72 * k2[q][j] + c_a73 * k3[q][j] + c_a74 * k4[q][j] +
                                     c_a75 * k5[q][j] + c_a76 * k6[q][j])
                    // before the last evaluation: the error estimate's sum and the dense
                    // output's coefficients over k1..k6 take the place of k2..k5
                    ND_EACH {
                        const double e = c_bt1 * k1[q][j] + c_bt2 * k2[q][j] + c_bt3 * k3[q][j] + c_bt4 * k4[q][j] +
                                         c_bt5 * k5[q][j] + c_bt6 * k6[q][j];
                        if constexpr (kLocate) {
                            const double e2 = ND_R(1, 2) * k1[q][j] + ND_R(2, 2) * k2[q][j] +
                                              ND_R(3, 2) * k3[q][j] + ND_R(4, 2) * k4[q][j] +
                                              ND_R(5, 2) * k5[q][j] + ND_R(6, 2) * k6[q][j];
                            const double e3 = ND_R(1, 3) * k1[q][j] + ND_R(2, 3) * k2[q][j] +
                                              ND_R(3, 3) * k3[q][j] + ND_R(4, 3) * k4[q][j] +
                                              ND_R(5, 3) * k5[q][j] + ND_R(6, 3) * k6[q][j];
                            const double e4 = ND_R(1, 4) * k1[q][j] + ND_R(2, 4) * k2[q][j] +
                                              ND_R(3, 4) * k3[q][j] + ND_R(4, 4) * k4[q][j] +
                                              ND_R(5, 4) * k5[q][j] + ND_R(6, 4) * k6[q][j];
                            d2[q][j] = e2;
                            d3[q][j] = e3;
                            d4[q][j] = e4;
                        }
                        k2[q][j] = e;
                    }
                }
#undef ND_STAGE
                ++phase;
                continue;
            }
            if (phase == 6) {
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < V; ++q)
                    if (t + q * T < I.n)
#pragma unroll
                        for (int j = 0; j < D; ++j) {
                            const double e = h * (k2[q][j] + c_bt7 * k[q][j]);
                            const double sc = a.abstol + fmax(fabs(y[q][j]), fabs(ys[q][j])) * a.reltol;
                            const double r = e / sc;
                            s += r * r;
                        }
                const double eest = sqrt(L.red.sum(s) * inv_len);
                double q11, qold8;
                step_pow2(eest, 0.14, qold, 0.08, q11, qold8);
                if (eest <= 1.0) {
                    double qq = eest == 0.0 ? 0.1 : fmax(0.1, fmin(5.0, q11 / qold8 / 0.9));
                    // a step that ends within 100 ulp of the stop time ends on it (as
                    // OrdinaryDiffEq's fixed_t_for_floatingpoint_error! does)
                    const double tn = tcur + h;
                    const bool at_stop = last || fabs(tn - tstop) < 100.0 * 2.220446049250313e-16 * fmax(fabs(tcur), fabs(tstop));
                    qold = fmax(eest, 1e-4);
                    dt = fmin(h / qq, a.dtmax);
                    ++naccept;
                    int changed = 0;
                    bool located = false;
                    if constexpr (kLocate) {
                        if (lim) {
                            const int t = fresh<FRESH>(static_cast<int>(threadIdx.x));
                            // the dense output's coefficients with the last derivative, in arrays of their
                            // own: updated in place, both values would be live around the loop over the
                            // phases (210 spilled registers at four vertices per thread instead of 63, 67
                            // instead of 6 at three; 512 networks of 1700 / 1900 vertices 32 / 39 ms instead
                            // of 22 / 25)
                            double e2[V][D], e3[V][D], e4[V][D];
                            ND_EACH {
                                e2[q][j] = d2[q][j] + ND_R(7, 2) * k[q][j];
                                e3[q][j] = d3[q][j] + ND_R(7, 3) * k[q][j];
                                e4[q][j] = d4[q][j] + ND_R(7, 4) * k[q][j];
                            }
                            // the condition at the points s = m/9 of the step (m = 9: the accepted
                            // state), against its sign at the step start
                            double first = 10.0;
#pragma unroll 1
                            for (int m = 1; m <= 9; ++m) {
                                double* th = (m & 1) ? theta2 : L.theta;   // alternate: one barrier a point
                                const double s = static_cast<double>(m) / 9.0;
#pragma unroll
                                for (int q = 0; q < V; ++q) {
                                    const int v = t + q * T;
                                    if (v < I.n)
                                        th[v] = m == 9 ? ys[q][0]
                                                       : dense_at(y[q][0], k1[q][0], e2[q][0], e3[q][0], e4[q][0], h, s);
                                }
                                __syncthreads();
                                for (int e = t; e < I.ne; e += T) {
                                    const int8_t ns = sign8(line_cond<EM>(L, th, lim, e));
                                    if (m == 1) gev[e] = 0;
                                    if (gev[e] == 0 && crossed(gsign[e], ns)) {
                                        gev[e] = static_cast<int8_t>(m);
                                        first = fmin(first, static_cast<double>(m));
                                    }
                                    if (m == 9) gnext[e] = ns;
                                }
                            }
                            first = L.red.min(first);
                            if (first < 10.0) {
                                // bisect [point mf-1, point mf] on the dense output, over the edges
                                // that crossed at point mf, down to adjacent doubles
                                const int mf = static_cast<int>(first);
                                double lo = tcur + h * (static_cast<double>(mf - 1) / 9.0);
                                double hi = tcur + h * (static_cast<double>(mf) / 9.0);
                                bool hi_end = mf == 9;                  // hi: still the accepted state
                                for (int it = 0; it < 256; ++it) {
                                    const double mid = lo + 0.5 * (hi - lo);
                                    if (!(mid > lo && mid < hi)) break;
                                    const double s = (mid - tcur) / h;
#pragma unroll
                                    for (int q = 0; q < V; ++q) {
                                        const int v = t + q * T;
                                        if (v < I.n) L.theta[v] = dense_at(y[q][0], k1[q][0], e2[q][0], e3[q][0], e4[q][0], h, s);
                                    }
                                    __syncthreads();
                                    double hit = 0.0;
                                    for (int e = t; e < I.ne; e += T)
                                        if (gev[e] == mf && crossed(gsign[e], sign8(line_cond<EM>(L, L.theta, lim, e)))) hit = 1.0;
                                    if (L.red.sum(hit) > 0.0) {
                                        hi = mid;
                                        hi_end = false;
                                    } else {
                                        lo = mid;
                                    }
                                }
                                // the edges that crossed by hi trip; the solution moves to lo, the
                                // left end of the bracket (DiffEqBase's LeftRootFind)
                                const double shi = (hi - tcur) / h;
#pragma unroll
                                for (int q = 0; q < V; ++q) {
                                    const int v = t + q * T;
                                    if (v < I.n)
                                        L.theta[v] = hi_end ? ys[q][0]
                                                            : dense_at(y[q][0], k1[q][0], e2[q][0], e3[q][0], e4[q][0], h, shi);
                                }
                                __syncthreads();
                                constexpr int NPE1 = NPE > 0 ? NPE : 1;
                                double* pw = a.p + I.poff + static_cast<int64_t>(I.n) * VPar<VM>::np;
                                double cnt = 0.0;
                                for (int e = t; e < I.ne; e += T)
                                    if (gev[e] == mf && crossed(gsign[e], sign8(line_cond<EM>(L, L.theta, lim, e)))) {
                                        L.epar[e * NPE1] = 0.0;
                                        pw[static_cast<int64_t>(e) * NPE1] = 0.0;
                                        cnt += 1.0;
                                    }
                                ntrip += static_cast<int>(L.red.sum(cnt));
                                const double slo = (lo - tcur) / h;
#pragma unroll
                                for (int q = 0; q < V; ++q)
#pragma unroll
                                    for (int j = 0; j < D; ++j)
                                        y[q][j] = dense_at(y[q][j], k1[q][j], e2[q][j], e3[q][j], e4[q][j], h, slo);
                                tcur = lo;
                                located = true;
                                changed = 1;                            // the state moved: new derivative
                            }
                        }
                    }
                    if (!located) {
                        tcur = at_stop ? tstop : tn;
#pragma unroll
                        for (int q = 0; q < V; ++q)
#pragma unroll
                            for (int j = 0; j < D; ++j) { y[q][j] = ys[q][j]; k1[q][j] = k[q][j]; }
                        if constexpr (kLocate) {
                            int8_t* sw = gsign;                         // the end signs start the next step
                            gsign = gnext;
                            gnext = sw;
                        } else if (a.limit) {
                            // fslot holds the flows at the accepted state (the last evaluation was at ys)
                            const int tr = trip_lines<VM, EM>(a, I, L);
                            ntrip += tr;
                            changed += tr;
                        }
                        if (at_stop && ee >= 0 && tstop == te) {   // the preset trip's time is reached
                            const int tr = trip_edge<VM, EM>(a, I, L, ee);
                            ntrip += tr;
                            changed += tr;
                            ee = -1;
                            tstop = a.t1;
                        }
                    }
                    // after a trip or a move to a crossing the first-same-as-last derivative
                    // (and the condition signs) are stale: evaluate them again
                    if (changed > 0) {
                        ND_EACH ys[q][j] = y[q][j];
                        phase = 8;
                        continue;
                    }
                    accepted = true;
                } else {
                    dt = h / fmin(5.0, q11 / 0.9);
                    ++nreject;
                }
            } else if (phase == 8) {
                ND_EACH k1[q][j] = k[q][j];
                if constexpr (kLocate)
                    if (lim) line_signs<VM, EM, V, FRESH>(I, L, lim, y, gsign);
                accepted = true;
            } else {
                // the start: k1, then for an automatic initial step its probe (Hairer, Norsett &
                // Wanner, Solving ODEs I, II.4)
                if (phase == 0) {
                    ND_EACH k1[q][j] = k[q][j];
                    if (!(dt > 0.0)) {
                        const double d0 = sqrt(wnorm2(y, y) * inv_len);
                        d1 = sqrt(wnorm2(k1, y) * inv_len);
                        h = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
                        h = fmin(h, a.t1 - a.t0);
                        ND_EACH ys[q][j] = y[q][j] + h * k1[q][j];
                        phase = 7;
                        continue;
                    }
                } else {
                    ND_EACH k[q][j] = k[q][j] - k1[q][j];
                    const double dd2 = sqrt(wnorm2(k, y) * inv_len) / h;
                    const double m = fmax(d1, dd2);
                    const double h1 = m <= 1e-15 ? fmax(1e-6, h * 1e-3) : uniform_f64(step_pow(0.01 / m, 1.0 / 6.0));
                    dt = fmin(100.0 * h, h1);
                }
                dt = fmin(dt, a.dtmax);
                begun = false;
                if constexpr (kLocate)
                    if (lim) line_signs<VM, EM, V, FRESH>(I, L, lim, y, gsign);
            }
            if (accepted && a.ss && at_steady_state<V, D>(a, I, L, y, k1)) {
                retcode = 4;
                break;
            }
            if (begun && !(dt == dt)) { retcode = 3; break; }
            if (!(tcur < a.t1)) break;
            if (iters++ >= a.maxiters) { retcode = 1; break; }
            if (dt < a.dtmin) { retcode = 2; break; }
            last = tcur + dt >= tstop;
            h = last ? tstop - tcur : dt;
            ND_EACH ys[q][j] = y[q][j] + h * (c_a21 * k1[q][j]);
            phase = 1;
        }
    }
#undef ND_EACH
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int v = t + k * T;
        if (v < I.n)
#pragma unroll
            for (int j = 0; j < D; ++j) a.u[I.uoff + static_cast<int64_t>(v) * D + j] = y[k][j];
    }
    if (t == 0) {
        nd_ensemble_stat st;
        st.t = tcur;
        st.dt = dt;
        st.naccept = naccept;
        st.nreject = nreject;
        st.nf = nf;
        st.retcode = retcode;
        st.ntrip = ntrip;
        a.stats[inst] = st;
    }
}

// Waves per SIMD that a kernel leaves registers for.  Three where a small workgroup's kernel comes
// close to their 168 registers by itself (RK4, one state per vertex).  DENSE: four
template <int VM, int METHOD, int V, int LB, bool DENSE>
constexpr int kMinWaves = DENSE || LB > 512 ? 4 : LB <= 256 && V <= 2 && (METHOD == 1 || (METHOD == 0 && VModel<VM>::dim == 1)) ? 3 : 2;

template <int VM, int EM, int METHOD, int V, int LB, bool DENSE = false>
__global__ void __launch_bounds__(LB, (kMinWaves<VM, METHOD, V, LB, DENSE>)) k_ensemble(SolveArgs a) {
    extern __shared__ double2 smem[];
    const int inst = a.order[a.first + static_cast<int>(blockIdx.x)];
    const InstDesc I = a.inst[inst];
    ensemble_body<VM, EM, METHOD, V, LB, kFresh<V, LB> || DENSE>(a, inst, I, smem);
}

// Several size classes of one thread count in one launch: each instance runs with its
// class's vertices per thread.
template <int VM, int EM, int METHOD, int LB>
__global__ void __launch_bounds__(LB, 2) k_ensemble_mixed(SolveArgs a) {
    extern __shared__ double2 smem[];
    const int inst = a.order[a.first + static_cast<int>(blockIdx.x)];
    const InstDesc I = a.inst[inst];
    switch (__builtin_amdgcn_readfirstlane(I.vper)) {
    case 1: ensemble_body<VM, EM, METHOD, 1, LB, kFresh<1, LB>>(a, inst, I, smem); break;
    case 2: ensemble_body<VM, EM, METHOD, 2, LB, kFresh<2, LB>>(a, inst, I, smem); break;
    case 3: ensemble_body<VM, EM, METHOD, 3, LB, kFresh<3, LB>>(a, inst, I, smem); break;
    default: ensemble_body<VM, EM, METHOD, 4, LB, kFresh<4, LB>>(a, inst, I, smem); break;
    }
}

using EnsKernel = void (*)(SolveArgs);

// vper 0: by instance
template <int VM, int EM, int METHOD, int LB>
EnsKernel pick_vper(int vper, bool dense) {
    if constexpr (METHOD == 1) {
        if (dense && vper == 1) return k_ensemble<VM, EM, METHOD, 1, LB, true>;
        if (dense && vper == 2) return k_ensemble<VM, EM, METHOD, 2, LB, true>;
    }
    switch (vper) {
    case 0: return k_ensemble_mixed<VM, EM, METHOD, LB>;
    case 1: return k_ensemble<VM, EM, METHOD, 1, LB>;
    case 3: return k_ensemble<VM, EM, METHOD, 3, LB>;
    case 4: return k_ensemble<VM, EM, METHOD, 4, LB>;
    default: return k_ensemble<VM, EM, METHOD, 2, LB>;
    }
}
// Workgroups of up to 512 threads take any vper; 1024-thread workgroups (16 waves, at most 128
// VGPRs each) take one or two vertices per thread.  small: at most 256 threads, and few edges per
// thread in a quarter of the instances or more
template <int VM, int EM, int METHOD>
EnsKernel pick_v(int vper, int threads, bool small, bool dense) {
    if (threads > 512) return vper == 1 ? k_ensemble<VM, EM, METHOD, 1, 1024> : k_ensemble<VM, EM, METHOD, 2, 1024>;
    return small ? pick_vper<VM, EM, METHOD, 256>(vper, dense) : pick_vper<VM, EM, METHOD, 512>(vper, dense);
}

// kernel method: 0 Tsit5, 1 RK4, 2 Tsit5 with line crossings located on the dense output
template <int VM, int EM>
EnsKernel pick_m(int kmethod, int vper, int threads, bool small, bool dense) {
    switch (kmethod) {
    case 1: return pick_v<VM, EM, 1>(vper, threads, small, dense);
    case 2: return pick_v<VM, EM, 2>(vper, threads, small, dense);
    default: return pick_v<VM, EM, 0>(vper, threads, small, dense);
    }
}

EnsKernel pick_ensemble(int vm, int em, int kmethod, int vper, int threads, bool small, bool dense) {
    if (vm == ND_VM_SWING && em == ND_EM_KURAMOTO) return pick_m<ND_VM_SWING, ND_EM_KURAMOTO>(kmethod, vper, threads, small, dense);
    if (vm == ND_VM_SWING && em == ND_EM_STATIC_LINE) return pick_m<ND_VM_SWING, ND_EM_STATIC_LINE>(kmethod, vper, threads, small, dense);
    if (vm == ND_VM_KURAMOTO && em == ND_EM_KURAMOTO) return pick_m<ND_VM_KURAMOTO, ND_EM_KURAMOTO>(kmethod, vper, threads, small, dense);
    if (vm == ND_VM_KURAMOTO && em == ND_EM_STATIC_LINE)
        return pick_m<ND_VM_KURAMOTO, ND_EM_STATIC_LINE>(kmethod, vper, threads, small, dense);
    return nullptr;
}

// the kernel method of a solve: crossings are located for Tsit5 with line limits unless
// step-end checks were asked for
int kernel_method(const nd_ensemble_opts* o) {
    if (o->method == ND_METHOD_RK4) return 1;
    return (o->line_limit && o->line_events != ND_LINES_STEP_END) ? 2 : 0;
}

int vpar(int vm) {
    switch (vm) {
    case ND_VM_KURAMOTO: return 1;
    case ND_VM_SWING: return 3;
    default: return -1;
    }
}
int epar(int em) { return em == ND_EM_KURAMOTO ? 1 : em == ND_EM_STATIC_LINE ? 2 : -1; }

int hip_err(hipError_t e, const char* what) {
    if (e == hipSuccess) return ND_OK;
    return nd::set_error(ND_ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
}

}  // namespace

struct nd_ensemble {
    int device = 0;
    int lds_max = 0;                                // dynamic LDS a workgroup may take
    int cus = 0;                                    // of the device
    int32_t ninst = 0;
    nd_kind vk{}, ek{};
    int32_t dim = 0;
    int64_t total_states = 0, total_params = 0;
    std::vector<InstDesc> inst;
    int32_t cls_threads[ND_ENSEMBLE_CLASSES] = {128, 256, 512, 512, 512, 512};
    int32_t cls_vper[ND_ENSEMBLE_CLASSES] = {2, 2, 2, 3, 4, 4};
    std::vector<void*> allocs;
    InstDesc* d_inst = nullptr;
    int32_t* d_order = nullptr;
    uint2* d_tab = nullptr;
    uint32_t *d_row = nullptr, *d_hc = nullptr;
    std::vector<int32_t> order;                     // instances grouped by class, largest first
    int32_t cls_first[ND_ENSEMBLE_CLASSES + 1] = {};   // class c: order[cls_first[c + 1] .. cls_first[c]), the last first
    int64_t generation = 0;                         // bumped whenever the class layout changes
    // side streams so the class launches overlap; forked from and joined back to the
    // caller's stream with events (default priority, non-blocking)
    hipStream_t side_stream[kSideStreams] = {};
    hipEvent_t ev_fork = nullptr;
    hipEvent_t ev_join[kSideStreams] = {};
    hipStream_t cap_stream = nullptr;               // origin stream of graph captures
    ~nd_ensemble() {
        for (void* p : allocs) (void)hipFree(p);
        for (auto& x : side_stream) if (x) (void)hipStreamDestroy(x);
        for (auto& x : ev_join) if (x) (void)hipEventDestroy(x);
        if (ev_fork) (void)hipEventDestroy(ev_fork);
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
    }
};

struct nd_ensemble_graph {
    nd_ensemble* en = nullptr;
    int64_t generation = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    ~nd_ensemble_graph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

namespace {

template <typename T>
int up(nd_ensemble* en, const std::vector<T>& h, T** d) {
    *d = nullptr;
    if (h.empty()) return ND_OK;
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, h.size() * sizeof(T));
    if (e != hipSuccess) return nd::set_error(ND_ERR_ALLOC, "hipMalloc: %s", hipGetErrorString(e));
    en->allocs.push_back(p);
    e = hipMemcpy(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_err(e, "hipMemcpy");
    *d = static_cast<T*>(p);
    return ND_OK;
}

int class_of(const nd_ensemble* en, int32_t n) {
    for (int c = 0; c < ND_ENSEMBLE_CLASSES; ++c)
        if (n <= en->cls_threads[c] * en->cls_vper[c]) return c;
    return -1;
}

int regroup(nd_ensemble* en) {
    ++en->generation;
    std::vector<std::vector<std::pair<int32_t, int32_t>>> byc(ND_ENSEMBLE_CLASSES);
    for (int32_t i = 0; i < en->ninst; ++i) {
        const int c = class_of(en, en->inst[i].n);
        if (c < 0) return nd::set_error(ND_ERR_UNSUPPORTED, "instance %d: %d vertices exceed the largest class", i, en->inst[i].n);
        en->inst[i].cls = c;
        en->inst[i].vper = en->cls_vper[c];
        byc[c].emplace_back(-en->inst[i].n, i);
    }
    en->order.clear();
    en->cls_first[ND_ENSEMBLE_CLASSES] = 0;
    for (int c = ND_ENSEMBLE_CLASSES - 1; c >= 0; --c) {
        std::sort(byc[c].begin(), byc[c].end());
        for (auto& x : byc[c]) en->order.push_back(x.second);
        en->cls_first[c] = static_cast<int32_t>(en->order.size());
    }
    if (en->d_order) {
        auto it = std::find(en->allocs.begin(), en->allocs.end(), static_cast<void*>(en->d_order));
        if (it != en->allocs.end()) { (void)hipFree(*it); en->allocs.erase(it); }
        en->d_order = nullptr;
    }
    int rc = up(en, en->order, &en->d_order);
    if (rc) return rc;
    if (en->d_inst) {
        return hip_err(hipMemcpy(en->d_inst, en->inst.data(), en->inst.size() * sizeof(InstDesc), hipMemcpyHostToDevice),
                       "hipMemcpy");
    }
    return ND_OK;
}

int make_args(nd_ensemble* en, double* u, double* p, double t0, double t1, const nd_ensemble_opts* o,
              nd_ensemble_stat* stats, SolveArgs* a) {
    if (!en || !u || !p || !o || !stats) return nd::set_error(ND_ERR_ARGUMENT, "NULL argument");
    if (!(t1 >= t0)) return nd::set_error(ND_ERR_ARGUMENT, "t1 < t0");
    if (o->method != ND_METHOD_TSIT5 && o->method != ND_METHOD_RK4) return nd::set_error(ND_ERR_ARGUMENT, "unknown method");
    if (o->method == ND_METHOD_RK4 && !(o->dt0 > 0.0)) return nd::set_error(ND_ERR_ARGUMENT, "RK4 needs dt0 > 0");
    if (o->line_events != ND_LINES_DEFAULT && o->line_events != ND_LINES_STEP_END && o->line_events != ND_LINES_CROSSING)
        return nd::set_error(ND_ERR_ARGUMENT, "line_events must be ND_LINES_DEFAULT, ND_LINES_STEP_END or ND_LINES_CROSSING");
    if (o->method == ND_METHOD_RK4 && o->line_events == ND_LINES_CROSSING)
        return nd::set_error(ND_ERR_UNSUPPORTED, "line crossings are located on Tsit5's dense output; RK4 checks limits "
                             "at step ends (ND_LINES_STEP_END)");
    int dev = -1;
    (void)hipGetDevice(&dev);
    if (dev != en->device) return nd::set_error(ND_ERR_ARGUMENT, "ensemble lives on device %d", en->device);
    *a = SolveArgs{};
    a->inst = en->d_inst;
    a->order = en->d_order;
    a->tab = en->d_tab;
    a->row = en->d_row;
    a->hc = en->d_hc;
    a->lds_max = en->lds_max;
    a->u = u;
    a->p = p;
    a->limit = o->line_limit;
    if ((o->event_t == nullptr) != (o->event_e == nullptr))
        return nd::set_error(ND_ERR_ARGUMENT, "event_t and event_e go together");
    a->event_t = o->event_t;
    a->event_e = o->event_e;
    a->stats = stats;
    a->t0 = t0;
    a->t1 = t1;
    a->dt0 = o->dt0;
    a->reltol = o->reltol > 0 ? o->reltol : 1e-3;
    a->abstol = o->abstol > 0 ? o->abstol : 1e-6;
    a->dtmax = o->dtmax > 0 ? o->dtmax : (t1 - t0);
    a->dtmin = o->dtmin > 0 ? o->dtmin : 1e-14 * std::max(1.0, std::fabs(t1));
    a->maxiters = o->maxiters > 0 ? o->maxiters : 1000000;
    if (!(o->ss_abstol >= 0.0) || !(o->ss_reltol >= 0.0))
        return nd::set_error(ND_ERR_ARGUMENT, "steady-state tolerances must be >= 0");
    a->ss_abstol = o->ss_abstol;
    a->ss_reltol = o->ss_reltol;
    a->ss = (o->ss_abstol > 0.0 || o->ss_reltol > 0.0) ? 1 : 0;
    return ND_OK;
}

// dynamic LDS of class c: the largest need of its instances, each with its tables where they
// fit as well (the kernel decides by the same sum)
int32_t class_lds(const nd_ensemble* en, int c, int kmethod) {
    int32_t lds = 0;
    for (int32_t q = en->cls_first[c + 1]; q < en->cls_first[c]; ++q) {
        const InstDesc& I = en->inst[en->order[q]];
        const int32_t need = I.lds_bytes + (kmethod == 2 ? locate_bytes(I.n, I.ne) : 0);
        lds = std::max(lds, need + I.tab_bytes <= en->lds_max ? need + I.tab_bytes : need);
    }
    return lds;
}

// the figure the instances of class c are limited by: with line crossings located, a second
// phase buffer and three bytes per edge more.  Never below what the kernel takes without the
// edge table.
int32_t class_limit(const nd_ensemble* en, int c, int kmethod) {
    int32_t lim = 0;
    for (int32_t q = en->cls_first[c + 1]; q < en->cls_first[c]; ++q) {
        const InstDesc& I = en->inst[en->order[q]];
        lim = std::max(lim, I.limit_bytes + (kmethod == 2 ? 8 + 8 * I.n + 3 * I.ne : 0));
    }
    return lim;
}

// RK4 at one and two vertices per thread comes within 128 registers with its addresses recomputed,
// which costs 5 % where the instances are on the chip at once (168 registers, twelve waves a CU)
// and gains where they are not.  us for 1024 swing networks, 168 / 128 registers: 128 vertices (128
// threads) 704 / 741, 300 (256 threads) 1493 / 1219, 700 (512 threads) 3447 / 2490; 4096 of 20 to 250
// vertices 2134 / 2014; one of 1000 792 / 850.
constexpr int kSparseWaves = 12;

// The launches of a solve, largest instances first.  Neighbouring classes of one thread
// count share a launch: at 512 threads a CU holds one workgroup of most kernels whatever its
// vertices per thread, and one list of instances by decreasing size ends more evenly than several
// launches side by side.  (1024 networks of 100 to 2000 vertices, default classes, three
// ensembles solved in turn, swing Tsit5: 46.9 ms each with a launch and a stream per class, since
// streams beyond the four hardware queues of a process share one and their classes run one after
// the other; 40.2 ms so.  Where the separate kernels would leave room for a second workgroup, RK4,
// the two are even: 4.56 ms and 4.49 for swing, 4.27 and 4.36 for first-order vertices.)
struct Launch {
    EnsKernel kernel;
    int32_t first, count, threads, lds;
};
int launches(const nd_ensemble* en, int kmethod, Launch* out) {
    int n = 0;
    for (int c = ND_ENSEMBLE_CLASSES - 1; c >= 0;) {
        if (en->cls_first[c] == en->cls_first[c + 1]) { --c; continue; }
        const int32_t threads = en->cls_threads[c];
        int32_t vper = en->cls_vper[c], lds = 0;
        Launch l{nullptr, en->cls_first[c + 1], 0, threads, 0};
        for (; c >= 0; --c) {
            if (en->cls_first[c] == en->cls_first[c + 1]) continue;
            if (en->cls_threads[c] != threads || (threads > 512 && en->cls_vper[c] != vper)) break;
            if (en->cls_vper[c] != vper) vper = 0;
            lds = std::max(lds, class_lds(en, c, kmethod));
            l.count = en->cls_first[c] - l.first;
        }
        l.lds = lds;
        int32_t few = 0;
        for (int32_t q = l.first; q < l.first + l.count; ++q) few += en->inst[en->order[q]].ne <= 2 * threads;
        const bool small = threads <= 256 && 4 * few > l.count;
        l.kernel = pick_ensemble(en->vk.model, en->ek.model, kmethod, vper, threads, small,
                                 l.count > en->cus * std::max(1, kSparseWaves * kWave / threads));
        out[n++] = l;
    }
    return n;
}

// Streams, events and the dynamic-LDS limit of every class kernel; host-side only,
// so a capture that follows records nothing but the launches and the event edges.
int prepare(nd_ensemble* en, int kmethod) {
    int rc = ND_OK;
    if (!en->ev_fork) rc = hip_err(hipEventCreateWithFlags(&en->ev_fork, hipEventDisableTiming), "hipEventCreate");
    for (int c = 0; c < kSideStreams && !rc; ++c) {
        if (!en->side_stream[c])
            rc = hip_err(hipStreamCreateWithFlags(&en->side_stream[c], hipStreamNonBlocking), "hipStreamCreateWithFlags");
        if (!rc && !en->ev_join[c])
            rc = hip_err(hipEventCreateWithFlags(&en->ev_join[c], hipEventDisableTiming), "hipEventCreate");
    }
    if (rc) return rc;
    Launch ls[ND_ENSEMBLE_CLASSES];
    const int n = launches(en, kmethod, ls);
    for (int c = 0; c < ND_ENSEMBLE_CLASSES; ++c)
        if (en->cls_first[c] > en->cls_first[c + 1] && class_limit(en, c, kmethod) > en->lds_max)
            return nd::set_error(ND_ERR_UNSUPPORTED, "class %d needs %d bytes of LDS with line crossings located "
                                 "(device limit %d)", c, class_limit(en, c, kmethod), en->lds_max);
    // one template instance may serve several launches: give it the largest need
    for (int i = 0; i < n; ++i) {
        if (!ls[i].kernel) return nd::set_error(ND_ERR_UNSUPPORTED, "no ensemble kernel for these models");
        int32_t need = 0;
        for (int j = 0; j < n; ++j)
            if (ls[j].kernel == ls[i].kernel) need = std::max(need, ls[j].lds);
        rc = hip_err(hipFuncSetAttribute(reinterpret_cast<const void*>(ls[i].kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, need),
                     "hipFuncSetAttribute(LDS)");
        if (rc) return rc;
    }
    return ND_OK;
}

// The first launch (the largest instances) runs on the caller's stream, up to three more on
// side streams forked from it and joined back with events, any others behind the first.  All
// launches come before the first wait, which is a barrier in the caller's hardware queue.
int launch_classes(nd_ensemble* en, SolveArgs a, int kmethod, hipStream_t s) {
    Launch ls[ND_ENSEMBLE_CLASSES];
    const int n = launches(en, kmethod, ls);
    const int nside = std::min<int>(kSideStreams, n - 1);
    int rc = nside > 0 ? hip_err(hipEventRecord(en->ev_fork, s), "hipEventRecord") : ND_OK;
    for (int i = 0; i < n && !rc; ++i) {
        const int side = i >= 1 && i <= nside ? i - 1 : -1;
        hipStream_t cs = side >= 0 ? en->side_stream[side] : s;
        if (side >= 0) rc = hip_err(hipStreamWaitEvent(cs, en->ev_fork, 0), "hipStreamWaitEvent");
        if (rc) break;
        a.first = ls[i].first;
        a.count = ls[i].count;
        hipLaunchKernelGGL(ls[i].kernel, dim3(static_cast<unsigned>(a.count)), dim3(static_cast<unsigned>(ls[i].threads)),
                           static_cast<unsigned>(ls[i].lds), cs, a);
        rc = hip_err(hipGetLastError(), "ensemble launch");
        if (!rc && side >= 0) rc = hip_err(hipEventRecord(en->ev_join[side], cs), "hipEventRecord");
    }
    for (int i = 0; i < nside && !rc; ++i)
        rc = hip_err(hipStreamWaitEvent(s, en->ev_join[i], 0), "hipStreamWaitEvent");
    return rc;
}

}  // namespace

extern "C" {

int nd_ensemble_create(int32_t ninst, const int64_t* nv, const int64_t* ne, const int64_t* src, const int64_t* dst,
                       const nd_kind* vkind, const nd_kind* ekind, nd_ensemble** out) {
    nd::clear_error();
    if (!out || ninst < 1 || !nv || !ne || !vkind || !ekind) return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    *out = nullptr;
    if (vkind->is_edge || !ekind->is_edge) return nd::set_error(ND_ERR_ARGUMENT, "kinds: need a vertex and an edge kind");
    if (vpar(vkind->model) < 0 || vkind->pdim != vpar(vkind->model) || vkind->ff != ND_FF_PURESTATEMAP ||
        vkind->outdim_dst != 1 || vkind->mask_dst[0] != 1)
        return nd::set_error(ND_ERR_UNSUPPORTED, "ensemble vertex model %d (needs Kuramoto or swing with output x[1])",
                             vkind->model);
    if (epar(ekind->model) < 0 || ekind->pdim != epar(ekind->model) || ekind->wrapper != ND_WRAP_ANTISYMMETRIC ||
        ekind->outdim_dst != 1 || ekind->dim != 0)
        return nd::set_error(ND_ERR_UNSUPPORTED, "ensemble edge model %d (needs an AntiSymmetric Kuramoto or static line)",
                             ekind->model);
    nd_ensemble* en = new (std::nothrow) nd_ensemble;
    if (!en) return nd::set_error(ND_ERR_ALLOC, "allocation failed");
    (void)hipGetDevice(&en->device);
    int lds_max = 0;
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, en->device) != hipSuccess || lds_max <= 0)
        lds_max = 64 * 1024;
    en->lds_max = lds_max;
    if (hipDeviceGetAttribute(&en->cus, hipDeviceAttributeMultiprocessorCount, en->device) != hipSuccess || en->cus <= 0)
        en->cus = 256;
    en->ninst = ninst;
    en->vk = *vkind;
    en->ek = *ekind;
    en->dim = vkind->dim;
    std::vector<uint2> tab;
    std::vector<uint32_t> rows, hc;
    int64_t eoff = 0, uoff = 0, poff = 0;
    for (int32_t i = 0; i < ninst; ++i) {
        const int64_t n = nv[i], m = ne[i];
        if (n < 1 || n > 32767 || m < 0 || 2 * m > 65535) {
            delete en;
            return nd::set_error(ND_ERR_UNSUPPORTED, "instance %d: sizes outside the ensemble kernel limits", i);
        }
        // destination lists in the reference aggregation order: increasing edge index,
        // src output before dst output (aggregators.jl:54-86, 140-151)
        std::vector<int32_t> deg(static_cast<size_t>(n) + 1, 0);
        for (int64_t e = 0; e < m; ++e) {
            const int64_t s = src[eoff + e] - 1, d = dst[eoff + e] - 1;
            if (s < 0 || s >= n || d < 0 || d >= n) {
                delete en;
                return nd::set_error(ND_ERR_ARGUMENT, "instance %d: edge endpoint out of range", i);
            }
            deg[s + 1]++;
            deg[d + 1]++;
        }
        for (int64_t v = 0; v < n; ++v) deg[v + 1] += deg[v];
        InstDesc I{};
        I.n = static_cast<int32_t>(n);
        I.ne = static_cast<int32_t>(m);
        I.uoff = uoff;
        I.poff = poff;
        I.eoff = eoff;
        I.toff = static_cast<int64_t>(tab.size());
        I.voff = static_cast<int64_t>(rows.size());
        I.hoff = static_cast<int64_t>(hc.size());
        // rows of whole pairs; a row longer than kRowMax is cut into chunks of kChunk entries
        std::vector<uint32_t> fill(static_cast<size_t>(n));
        int64_t nch = 0, nhc = 0, npair = 0;
        for (int64_t v = 0; v < n; ++v) {
            const uint32_t len = static_cast<uint32_t>(deg[v + 1] - deg[v]), pairs = (len + 1) / 2;
            const uint32_t chunks = (len + kChunk - 1) / kChunk, first = static_cast<uint32_t>(npair);
            nch += chunks;
            fill[static_cast<size_t>(v)] = 2 * first;
            if (len <= kRowMax) {
                rows.push_back(first | pairs << 16);
            } else {
                rows.push_back(kRowHub | static_cast<uint32_t>(nhc) | chunks << 16);
                for (uint32_t b = 0; b < pairs; b += kChunk / 2)
                    hc.push_back((first + b) | std::min<uint32_t>(kChunk / 2, pairs - b) << 16);
                nhc += chunks;
            }
            npair += pairs;
        }
        const uint32_t dump = static_cast<uint32_t>(2 * (npair + kZeroPairs));
        I.npair = static_cast<int32_t>(npair);
        for (int64_t e = 0; e < pad_edges(static_cast<int>(m)); ++e) {
            if (e >= m) {
                tab.push_back(make_uint2(0, dump | dump << 16));
                continue;
            }
            const uint32_t s = static_cast<uint32_t>(src[eoff + e] - 1), d = static_cast<uint32_t>(dst[eoff + e] - 1);
            const uint32_t ps = fill[s]++, pd = fill[d]++;
            tab.push_back(make_uint2(8 * s | (8 * d) << 16, ps | pd << 16));
        }
        I.nhc = static_cast<int32_t>(nhc);
        const int npe = epar(ekind->model);
        I.lds_bytes = static_cast<int32_t>(8 * (pad2(static_cast<int>(n)) + 2 * (npair + kZeroPairs + kDumpPairs) +
                                                pad_edges(static_cast<int>(m)) * npe + 32 + nhc));
        I.tab_bytes = static_cast<int32_t>(8 * pad_edges(static_cast<int>(m)) + 4 * nhc);
        // The limit on an instance's size: 8 bytes per vertex, edge parameter, edge and 8-entry
        // chunk of the destination lists and 2 per entry of 16-bit index tables.  An instance
        // within it takes less without its tables: a row of odd length costs 8 bytes more than
        // its entries and its chunks at least 4 (12 from 17 entries on) less than there
        I.limit_bytes = static_cast<int32_t>(8 * (n + m * npe + m + nch + 32) + 2 * (2 * 2 * m + 2 * nch + 1 + n + 1));
        if (I.limit_bytes > lds_max) {
            delete en;
            return nd::set_error(ND_ERR_UNSUPPORTED, "instance %d needs %d bytes of LDS (device limit %d)", i, I.limit_bytes,
                                 lds_max);
        }
        en->inst.push_back(I);
        eoff += m;
        uoff += n * vkind->dim;
        poff += n * vkind->pdim + m * ekind->pdim;
    }
    en->total_states = uoff;
    en->total_params = poff;
    int rc = regroup(en);
    rc = rc ? rc : up(en, en->inst, &en->d_inst);
    rc = rc ? rc : up(en, tab, &en->d_tab);
    rc = rc ? rc : up(en, rows, &en->d_row);
    rc = rc ? rc : up(en, hc, &en->d_hc);
    if (rc) { delete en; return rc; }
    *out = en;
    return ND_OK;
}

void nd_ensemble_destroy(nd_ensemble* en) { delete en; }

int nd_ensemble_sizes(const nd_ensemble* en, int64_t* total_states, int64_t* total_params, int64_t* state_offsets,
                      int64_t* param_offsets) {
    if (!en) return nd::set_error(ND_ERR_ARGUMENT, "NULL ensemble");
    if (total_states) *total_states = en->total_states;
    if (total_params) *total_params = en->total_params;
    for (int32_t i = 0; i < en->ninst; ++i) {
        if (state_offsets) state_offsets[i] = en->inst[i].uoff;
        if (param_offsets) param_offsets[i] = en->inst[i].poff;
    }
    return ND_OK;
}

int nd_ensemble_set_class(nd_ensemble* en, int32_t cls, int32_t threads, int32_t vper) {
    if (!en || cls < 0 || cls >= ND_ENSEMBLE_CLASSES) return nd::set_error(ND_ERR_ARGUMENT, "bad class");
    if (threads < kWave || threads > 1024 || threads % kWave || vper < 1 || vper > 4 || (threads > 512 && vper > 2))
        return nd::set_error(ND_ERR_ARGUMENT, "threads must be a multiple of 64 in [64,1024], vper in {1,2,3,4} "
                             "(in {1,2} above 512 threads)");
    // regrouping replaces the instance-order array: queued solves finish with the old one
    int rc = hip_err(hipDeviceSynchronize(), "hipDeviceSynchronize");
    if (rc) return rc;
    en->cls_threads[cls] = threads;
    en->cls_vper[cls] = vper;
    return regroup(en);
}

int nd_tsit5_dense(double* r) {
    if (!r) return nd::set_error(ND_ERR_ARGUMENT, "NULL argument");
    for (int i = 0; i < 7; ++i)
        for (int j = 0; j < 4; ++j) r[i * 4 + j] = kTsit5Dense.r[i][j];
    return ND_OK;
}

int nd_tsit5_tableau(double* a, double* btilde, double* c) {
    if (!a || !btilde || !c) return nd::set_error(ND_ERR_ARGUMENT, "NULL argument");
    for (int i = 0; i < 7; ++i) {
        for (int j = 0; j < 6; ++j) a[i * 6 + j] = kTsit5.a[i][j];
        btilde[i] = kTsit5.bt[i];
        c[i] = kTsit5.c[i];
    }
    return ND_OK;
}

int nd_ensemble_solve(nd_ensemble* en, double* u, double* p, double t0, double t1, const nd_ensemble_opts* o,
                      nd_ensemble_stat* stats, void* stream) {
    SolveArgs a{};
    int rc = make_args(en, u, p, t0, t1, o, stats, &a);
    rc = rc ? rc : prepare(en, kernel_method(o));
    return rc ? rc : launch_classes(en, a, kernel_method(o), static_cast<hipStream_t>(stream));
}

int nd_ensemble_graph_create(nd_ensemble* en, double* u, double* p, double t0, double t1,
                             const nd_ensemble_opts* o, nd_ensemble_stat* stats, nd_ensemble_graph** out) {
    if (!out) return nd::set_error(ND_ERR_ARGUMENT, "NULL argument");
    *out = nullptr;
    SolveArgs a{};
    int rc = make_args(en, u, p, t0, t1, o, stats, &a);
    rc = rc ? rc : prepare(en, kernel_method(o));
    if (rc) return rc;
    if (!en->cap_stream) {
        rc = hip_err(hipStreamCreateWithFlags(&en->cap_stream, hipStreamNonBlocking), "hipStreamCreateWithFlags");
        if (rc) return rc;
    }
    nd_ensemble_graph* gr = new (std::nothrow) nd_ensemble_graph;
    if (!gr) return nd::set_error(ND_ERR_ALLOC, "allocation failed");
    gr->en = en;
    gr->generation = en->generation;
    rc = hip_err(hipStreamBeginCapture(en->cap_stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    if (rc) { delete gr; return rc; }
    const int lrc = launch_classes(en, a, kernel_method(o), en->cap_stream);
    hipGraph_t g = nullptr;
    rc = hip_err(hipStreamEndCapture(en->cap_stream, &g), "hipStreamEndCapture");
    gr->graph = g;
    if (lrc || rc) { delete gr; return lrc ? lrc : rc; }
    rc = hip_err(hipGraphInstantiate(&gr->exec, gr->graph, nullptr, nullptr, 0), "hipGraphInstantiate");
    if (rc) { delete gr; return rc; }
    *out = gr;
    return ND_OK;
}

int nd_ensemble_graph_launch(nd_ensemble_graph* gr, void* stream) {
    if (!gr || !gr->exec) return nd::set_error(ND_ERR_ARGUMENT, "NULL graph");
    if (gr->generation != gr->en->generation)
        return nd::set_error(ND_ERR_ARGUMENT, "the ensemble's size classes changed after this graph was captured");
    int dev = -1;
    (void)hipGetDevice(&dev);
    if (dev != gr->en->device) return nd::set_error(ND_ERR_ARGUMENT, "graph lives on device %d", gr->en->device);
    return hip_err(hipGraphLaunch(gr->exec, static_cast<hipStream_t>(stream)), "hipGraphLaunch");
}

void nd_ensemble_graph_destroy(nd_ensemble_graph* gr) { delete gr; }

}  // extern "C"
