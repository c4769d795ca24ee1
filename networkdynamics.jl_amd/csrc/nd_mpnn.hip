// Message-passing network for fixpoint warm starts: FP32 forward, backward and Adam,
// all in hand-written kernels.
//
// Nodes of a batch of grids are stacked (n rows); the graph is a row-normalised
// weighted adjacency (a_fwd[s] = K_s / sum of the row's K) in CSR form, plus its
// transpose weights a_bwd for the backward pass.  Layers (hidden width 64):
//   H0  = relu(X W_in + b_in)                              X: n x F features
//   H_l = relu((A H_{l-1}) W_l + H_{l-1} U_l + b_l)        l = 1..4
//   out = H_4 w_out + b_out                                (n)
// Loss: mean squared error against the target.  Weight gradients are reduced in
// two stages (per-block partials, then a fixed-order sum), so training is
// deterministic.
//
// A layer is one kernel in either direction.  Aggregating the 64 columns of H before the product
// instead of half of a 128-column product after it leaves one n x 64 read (plus the neighbours'
// rows, from L2) and one n x 64 write per layer; a product kernel and an aggregation kernel
// passed memory five times that.  For 773 293 nodes of power grids (4 layers, head and input) a
// forward pass went from 1902 to 771 us, forward and backward over 130 804 nodes from 1334 to
// 496 us.
//
// Parameter vector: W_in[F*64], b_in[64], {W_l|U_l [64*128], b_l[64]} x 4, w_out[64], b_out[1].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "nd_internal.h"

namespace {

constexpr int kH = 64;          // hidden width
constexpr int kLayers = 4;
constexpr int kWave = 64;

// ---- MFMA (v_mfma_f32_16x16x4f32) dense products ---------------------------------------
// Operand layout of one 16x16x4 step in a 64-lane wave: lane l holds A[i][k] and B[k][j]
// with i = j = l % 16, k = l / 16; the 4 accumulators of lane l are D[4*(l/16) + r][l % 16].
typedef float floatx4 __attribute__((ext_vector_type(4)));

// The input layer for feature counts other than 8: C[M x 64] = relu(A[M x K] * B[K x 64] + bias),
// K <= 128.  256 threads: a workgroup owns 128 rows, each wave 32 rows (2 row tiles) x 64
// columns; A's rows and all of B are staged in LDS with strides padded so the fragment reads
// are free of bank conflicts.
// dynamic LDS floats: A rows (stride Kp + 2) and B (stride N + 16)
inline size_t gemm_mfma_lds_floats(int K, int N) {
    const int Kp = (K + 3) & ~3;
    return static_cast<size_t>(128) * (Kp + 2) + static_cast<size_t>(Kp) * (N + 16);
}

template <int N>
__global__ void __launch_bounds__(256) k_gemm_mfma(int64_t M, int K, const float* __restrict__ A, int lda,
                                                   const float* __restrict__ B, int ldb, float* __restrict__ C, int ldc,
                                                   const float* __restrict__ bias, int relu) {
    constexpr int SB = N + 16, CT = N / 16;
    extern __shared__ float smem_f[];
    const int t = threadIdx.x, lane = t % kWave, w = t / kWave;
    const int Kp = (K + 3) & ~3;
    const int SA = Kp + 2;
    float* As = smem_f;
    float* Bs = smem_f + 128 * SA;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * 128;
    for (int i = t; i < 128 * Kp; i += 256) {
        const int r = i / Kp, k = i % Kp;
        As[r * SA + k] = (row0 + r < M && k < K) ? A[(row0 + r) * lda + k] : 0.0f;
    }
    for (int i = t; i < Kp * N; i += 256) {
        const int k = i / N, j = i % N;
        float v = 0.0f;
        if (k < K) v = B[static_cast<int64_t>(k) * ldb + j];
        Bs[k * SB + j] = v;
    }
    __syncthreads();
    floatx4 acc[2][CT];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int li = lane % 16, lk = lane / 16;
    for (int k0 = 0; k0 < Kp; k0 += 4) {
        float a[2], b[CT];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) a[rt] = As[(w * 32 + rt * 16 + li) * SA + k0 + lk];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) b[ct] = Bs[(k0 + lk) * SB + ct * 16 + li];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt], b[ct], acc[rt][ct], 0, 0, 0);
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = row0 + w * 32 + rt * 16 + 4 * lk + r;
                const int col = ct * 16 + li;
                if (row < M) {
                    float v = acc[rt][ct][r] + (bias ? bias[col] : 0.0f);
                    if (relu) v = fmaxf(v, 0.0f);
                    C[row * ldc + col] = v;
                }
            }
}

// partial[b] = A[rows_b]^T * B[rows_b] on MFMA: KA <= 64 output rows (one 16-row tile per
// wave), NB <= 128 output columns, part_rows(M) rows of the product's inner dimension
// per workgroup, staged through LDS 64 rows at a time.
constexpr int kTnChunk = 64;      // rows staged per LDS round
template <int NBT>
__global__ void __launch_bounds__(256) k_gemm_tn_mfma(int64_t M, int KA, int NB, const float* __restrict__ A, int lda,
                                                      const float* __restrict__ B, int ldb, float* __restrict__ part,
                                                      int rows_per_block) {
    constexpr int SA = 64 + 16, SB = NBT * 16 + 16;
    __shared__ float As[kTnChunk * SA];
    __shared__ float Bs[kTnChunk * SB];
    const int t = threadIdx.x, lane = t % kWave, w = t / kWave;
    const int li = lane % 16, lk = lane / 16;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < M ? r0 + rows_per_block : M;
    floatx4 acc[NBT];
#pragma unroll
    for (int ct = 0; ct < NBT; ++ct) acc[ct] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t rb = r0; rb < r1; rb += kTnChunk) {
        for (int i = t; i < kTnChunk * 64; i += 256) {
            const int rr = i / 64, c = i % 64;
            As[rr * SA + c] = (rb + rr < r1 && c < KA) ? A[(rb + rr) * lda + c] : 0.0f;
        }
        for (int i = t; i < kTnChunk * NBT * 16; i += 256) {
            const int rr = i / (NBT * 16), c = i % (NBT * 16);
            Bs[rr * SB + c] = (rb + rr < r1 && c < NB) ? B[(rb + rr) * ldb + c] : 0.0f;
        }
        __syncthreads();
        // output rows w*16 .. w*16+15 of A^T B: A^T[i][k] = As[k][i]
        for (int k0 = 0; k0 < kTnChunk; k0 += 4) {
            const float a = As[(k0 + lk) * SA + w * 16 + li];
#pragma unroll
            for (int ct = 0; ct < NBT; ++ct)
                acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bs[(k0 + lk) * SB + ct * 16 + li], acc[ct], 0, 0, 0);
        }
        __syncthreads();
    }
    const int nout = KA * NB;
#pragma unroll
    for (int ct = 0; ct < NBT; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = w * 16 + 4 * lk + r, j = ct * 16 + li;
            if (i < KA && j < NB) part[static_cast<int64_t>(blockIdx.x) * nout + i * NB + j] = acc[ct][r];
        }
}

// ---- dense: partial[b] = A[rows_b]^T * B[rows_b]  (KA x NB, KA*NB <= 8192) ---------------
// Rows of the inner dimension per workgroup of these two-stage sums (A^T B, column and
// vector sums): enough workgroups to fill the chip, at most kMaxPartBlocks of them, at
// least 64 rows each.  The partials are then added in a fixed order (k_reduce_partials),
// so every sum is deterministic for a given M.
constexpr int kMaxPartBlocks = 1024;
constexpr int64_t kWgradBlocks = 256;    // one workgroup per CU
inline int part_rows(int64_t M) {
    const int64_t r = (M + kMaxPartBlocks - 1) / kMaxPartBlocks;
    return static_cast<int>(std::max<int64_t>(64, (r + 63) / 64 * 64));
}
__global__ void __launch_bounds__(256) k_sgemm_tn_partial(int64_t M, int KA, int NB, const float* __restrict__ A, int lda,
                                                          const float* __restrict__ B, int ldb, float* __restrict__ part,
                                                          int rows_per_block) {
    __shared__ float As[16][128];
    __shared__ float Bs[16][128];
    const int nout = KA * NB;
    float acc[32];
#pragma unroll
    for (int q = 0; q < 32; ++q) acc[q] = 0.0f;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_block;
    const int64_t r1 = std::min<int64_t>(r0 + rows_per_block, M);
    for (int64_t rb = r0; rb < r1; rb += 16) {
        for (int i = threadIdx.x; i < 16 * 128; i += 256) {
            const int rr = i / 128, c = i % 128;
            const int64_t r = rb + rr;
            As[rr][c] = (r < r1 && c < KA) ? A[r * lda + c] : 0.0f;
            Bs[rr][c] = (r < r1 && c < NB) ? B[r * ldb + c] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 32; ++q) {
            const int o = threadIdx.x + q * 256;
            if (o < nout) {
                const int i = o / NB, j = o % NB;
                float s = 0.0f;
#pragma unroll
                for (int rr = 0; rr < 16; ++rr) s += As[rr][i] * Bs[rr][j];
                acc[q] += s;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < 32; ++q) {
        const int o = threadIdx.x + q * 256;
        if (o < nout) part[static_cast<int64_t>(blockIdx.x) * nout + o] = acc[q];
    }
}

// out[i] = sum_b part[b * ld + i] for i < nout, in block order
// (64 outputs per workgroup of kRedWaves waves: wave w adds the partials of blocks
// [nb*w/kRedWaves, nb*(w+1)/kRedWaves) in order, then the wave sums are added in wave order).
// The workgroups after those take a second array (nout2 columns, dense) to out2.
constexpr int kRedWaves = 16;
__global__ void __launch_bounds__(kRedWaves * 64) k_reduce_partials(int nb, int nout, int ld, const float* __restrict__ part,
                                                                    float* __restrict__ out, int nb2, int nout2,
                                                                    const float* __restrict__ part2,
                                                                    float* __restrict__ out2) {
    __shared__ float sh[kRedWaves][kWave];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    int blk = blockIdx.x;
    const int first2 = (nout + kWave - 1) / kWave;
    if (blk >= first2) {
        blk -= first2;
        nb = nb2;
        nout = ld = nout2;
        part = part2;
        out = out2;
    }
    const int i = blk * kWave + lane;
    const int b0 = nb * w / kRedWaves, b1 = nb * (w + 1) / kRedWaves;
    float s = 0.0f;
    if (i < nout) {
#pragma unroll 4
        for (int b = b0; b < b1; ++b) s += part[static_cast<int64_t>(b) * ld + i];
    }
    sh[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < nout) {
        float t = sh[0][lane];
        for (int q = 1; q < kRedWaves; ++q) t += sh[q][lane];
        out[i] = t;
    }
}

// column sums of G[M x 64] into per-block partials (bias gradients)
__global__ void __launch_bounds__(256) k_colsum_partial(int64_t M, const float* __restrict__ G, int ldg, float* __restrict__ part,
                                                        int rows_per_block) {
    __shared__ float sh[4][kH];
    const int c = threadIdx.x % kH, w = threadIdx.x / kH;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_block;
    const int64_t r1 = std::min<int64_t>(r0 + rows_per_block, M);
    float s = 0.0f;
    for (int64_t r = r0 + w; r < r1; r += 4) s += G[r * ldg + c];
    sh[w][c] = s;
    __syncthreads();
    if (w == 0) part[static_cast<int64_t>(blockIdx.x) * kH + c] = sh[0][c] + sh[1][c] + sh[2][c] + sh[3][c];
}

// Workgroups are dispatched to the chip's 8 XCDs round robin (workgroup b to XCD b % 8).  Each
// XCD works through one contiguous eighth of the tiles, so that rows of one grid, which read
// each other's rows, share one L2.  Neighbouring tiles go to different workgroups of the XCD:
// their row pointers and entries share cache lines, and a CU's L1 stands still when a load
// meets a line that is still on its way.
struct TileRange {
    int64_t first, end, step;
};
__device__ __forceinline__ TileRange wave_tiles(int64_t ntiles, int waves, int w) {
    const int64_t b = blockIdx.x, nb = gridDim.x;
    if (nb < 8) return {b + nb * w, ntiles, nb * waves};
    const int64_t x = b % 8, c = (ntiles + 7) / 8, per = nb / 8 + (x < nb % 8 ? 1 : 0);
    return {x * c + b / 8 + per * w, (x + 1) * c < ntiles ? (x + 1) * c : ntiles, per * waves};
}

// ---- a layer, forward and backward -----------------------------------------------------------
// A wave takes tiles of 16 nodes.  Global memory is read and written with 16 lanes per node,
// four nodes at a time: lane (li, lk) = (lane % 16, lane / 16) holds features 4 li .. 4 li + 3
// of node 4 p + lk (p = 0..3), so a row is one access of 256 bytes.  The products want lane
// (li, lk) to hold features 16 q + 4 lk + e (q, e = 0..3) of node li; a tile goes from one
// layout to the other through the wave's own 16 rows of LDS.  One v_mfma_f32_16x16x4f32 step
// takes the weights as its first operand (lane (li, lk): output column li of the column tile,
// input feature 16 q + 4 lk + e) and the nodes as its second, and lane (li, lk) receives node
// li's columns 16 q + 4 lk + e.
constexpr int kWS = 68;             // LDS stride of a weight or node row: 16-byte columns free of bank conflicts
constexpr int kTile = 16;           // nodes per wave and step
constexpr int kAhead = 2;           // entries of each of four nodes whose rows are in flight at once
// Entries of a row that are summed beside those of the tile's other nodes; the others of a longer row
// the wave takes 32 at a time (gather_long).  Forward passes with every row beside its tile's others /
// so: a star of 20 000 lines 14.8 / 1.46 ms, one preferential attachment graph of 1e5 nodes 666 / 508
// us, 100 of 2000 nodes 329 / 290 (cap 64: 274), 20 dense graphs of 30 to 90 lines a node 283 / 284
// (cap 64: 293).  The check costs a small batch (5 grids of 1000 nodes, 74 us) 2 %.
constexpr int kRowCap = 96;

// lane J of each 16 lanes to all of them; the 16 lanes moved down by kAhead
template <int J>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + J, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t row_down(uint32_t v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x120 + 16 - kAhead, 0xf, 0xf, true);
}
// order between a wave's own writes and reads of LDS
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// n rows of 64 floats.  Below 2 GB a row is reached through a buffer descriptor, whose bounds
// check turns an offset past the end into zeros without a memory access; beyond (WIDE) by
// index.  offset: the row's byte offset or index.
template <bool WIDE>
struct Rows {
    const float* X;
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Rows(const float* x, int64_t n) : X(x) {
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0,
                                              static_cast<int>(static_cast<uint32_t>(n * kH * sizeof(float))), 0x00020000);
    }
    static constexpr uint32_t kNone = 0x80000000u;
    static __device__ __forceinline__ uint32_t at(int32_t row) {
        return static_cast<uint32_t>(row) * (WIDE ? 1 : kH * sizeof(float));
    }
    __device__ __forceinline__ float4 part(uint32_t offset, int li) const {
        if constexpr (WIDE) {
            if (offset == kNone) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            return *reinterpret_cast<const float4*>(X + static_cast<int64_t>(offset) * kH + 4 * li);
        } else {
            return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(offset + 16 * li), 0, 0));
        }
    }
};

// The entries of a tile: its row pointers (lanes 0..16) and its first 64 neighbours and weights
struct TileEntries {
    int32_t rows, nbr;
    float a;
};
// lanes 0..16: the row pointers of nodes 16 tile .. 16 tile + 16 (those past the end repeat the last)
__device__ __forceinline__ int32_t tile_rows(const int32_t* __restrict__ rp, int64_t tile, int64_t n, int lane) {
    const int64_t r = tile * kTile + (lane < kTile ? lane : kTile);
    return rp[r < n ? r : n];
}
__device__ __forceinline__ void tile_entries(const int32_t* __restrict__ nbr, const float* __restrict__ a, int lane,
                                             TileEntries& t) {
    const int32_t first = __builtin_amdgcn_readfirstlane(t.rows), count = __builtin_amdgcn_readlane(t.rows, kTile) - first;
    if (count == 0) return;
    const int64_t s = first + static_cast<int64_t>(lane < count ? lane : count - 1);
    t.nbr = nbr[s];
    t.a = a[s];
}
// The entries of one row from position first on, added to the row's z: the wave takes 32 at a time,
// eight on each of its four node lanes, and adds the four sums at the end.
template <bool WIDE>
__device__ __forceinline__ float4 gather_long(const int32_t* __restrict__ nbr, const float* __restrict__ a,
                                              const Rows<WIDE>& X, int32_t first, int32_t end, int lane, int li, int lk) {
    float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto entries = [&](int64_t base, uint32_t& at, float& w) {
        const int64_t s = base + lane;
        at = s < end ? X.at(nbr[s]) : X.kNone;
        w = s < end ? a[s] : 0.0f;
    };
    uint32_t at;
    float w;
    entries(first, at, w);
    for (int64_t base = first; base < end; base += kWave) {
        const uint32_t at0 = at;
        const float w0 = w;
        entries(base + kWave, at, w);                     // the next 64 are on their way meanwhile
#pragma unroll 1
        for (int h = 0; h < kWave && base + h < end; h += 32) {
            float4 x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                x[i] = X.part(static_cast<uint32_t>(__shfl(static_cast<int>(at0), h + 4 * i + lk, kWave)), li);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float c = __shfl(w0, h + 4 * i + lk, kWave);
                z.x = __builtin_fmaf(c, x[i].x, z.x);
                z.y = __builtin_fmaf(c, x[i].y, z.y);
                z.z = __builtin_fmaf(c, x[i].z, z.z);
                z.w = __builtin_fmaf(c, x[i].w, z.w);
            }
        }
    }
#pragma unroll
    for (int off = 16; off < kWave; off *= 2) {
        z.x += __shfl_xor(z.x, off, kWave);
        z.y += __shfl_xor(z.y, off, kWave);
        z.z += __shfl_xor(z.z, off, kWave);
        z.w += __shfl_xor(z.w, off, kWave);
    }
    return z;
}
// z[p] = sum_s a[s] X[nbr[s], 4 li ..] over the entries of node 4 p + lk: the first kRowCap in order
// and side by side for all nodes, the others of a longer row by gather_long.  (The order depends on
// the row alone, so a node's sum does not depend on its place in the batch.)
template <bool WIDE>
__device__ __forceinline__ void gather_tile(const int32_t* __restrict__ nbr, const float* __restrict__ a, const Rows<WIDE>& X,
                                            const TileEntries& t, int li, int lk, float4 (&z)[4]) {
    const int32_t first = __builtin_amdgcn_readfirstlane(t.rows), count = __builtin_amdgcn_readlane(t.rows, kTile) - first;
    // the longest row of the tile (lanes 0..15)
    int32_t most = __shfl(t.rows, 16 * lk + li + 1, kWave) - t.rows;
    most = max(most, __builtin_amdgcn_update_dpp(0, most, 0x128, 0xf, 0xf, true));    // row_ror:8, 4, 2, 1
    most = max(most, __builtin_amdgcn_update_dpp(0, most, 0x124, 0xf, 0xf, true));
    most = max(most, __builtin_amdgcn_update_dpp(0, most, 0x122, 0xf, 0xf, true));
    most = max(most, __builtin_amdgcn_update_dpp(0, most, 0x121, 0xf, 0xf, true));
    most = __builtin_amdgcn_readfirstlane(most);
    const int32_t side = most < kRowCap ? most : kRowCap;
#pragma unroll
    for (int p = 0; p < 4; ++p) z[p] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t nb[4], av[4];                                // the next 16 entries of each node, one per lane
    for (int32_t k = 0; k < side; k += kAhead) {
        if (k % 16 == 0) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int32_t start = __shfl(t.rows, 4 * p + lk, kWave), end = __shfl(t.rows, 4 * p + lk + 1, kWave);
                const int64_t s = start + static_cast<int64_t>(k + li);
                const int32_t pos = static_cast<int32_t>(s - first);
                nb[p] = static_cast<uint32_t>(__shfl(t.nbr, pos & 63, kWave));
                av[p] = __float_as_uint(__shfl(t.a, pos & 63, kWave));
                if (count > kWave) {                      // a tile of more than 64 entries
                    if (s < end && pos >= kWave) {
                        nb[p] = static_cast<uint32_t>(nbr[s]);
                        av[p] = __float_as_uint(a[s]);
                    }
                    asm volatile("" : "+v"(nb[p]), "+v"(av[p]));     // waited for here, not on every path
                }
                nb[p] = s < end ? X.at(static_cast<int32_t>(nb[p])) : X.kNone;
                av[p] = s < end ? av[p] : 0u;
            }
        }
        float4 x[4][kAhead];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            x[p][0] = X.part(row_bcast<0>(nb[p]), li);
            x[p][1] = X.part(row_bcast<1>(nb[p]), li);
            if (kAhead > 2) {
                x[p][kAhead - 2] = X.part(row_bcast<kAhead - 2>(nb[p]), li);
                x[p][kAhead - 1] = X.part(row_bcast<kAhead - 1>(nb[p]), li);
            }
            nb[p] = row_down(nb[p]);
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float c[4] = {__uint_as_float(row_bcast<0>(av[p])), __uint_as_float(row_bcast<1>(av[p])),
                                __uint_as_float(row_bcast<2>(av[p])), __uint_as_float(row_bcast<3>(av[p]))};
            av[p] = row_down(av[p]);
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                z[p].x = __builtin_fmaf(c[i], x[p][i].x, z[p].x);
                z[p].y = __builtin_fmaf(c[i], x[p][i].y, z[p].y);
                z[p].z = __builtin_fmaf(c[i], x[p][i].z, z[p].z);
                z[p].w = __builtin_fmaf(c[i], x[p][i].w, z[p].w);
            }
        }
    }
    if (most > kRowCap) {
        const int lane = 16 * lk + li;
#pragma unroll 1
        for (int j = 0; j < kTile; ++j) {
            const int32_t start = __builtin_amdgcn_readlane(t.rows, j), end = __builtin_amdgcn_readlane(t.rows, j + 1);
            if (end - start <= kRowCap) continue;
            const float4 y = gather_long<WIDE>(nbr, a, X, start + kRowCap, end, lane, li, lk);
#pragma unroll
            for (int p = 0; p < 4; ++p)
                if (j == 4 * p + lk) z[p] = make_float4(z[p].x + y.x, z[p].y + y.y, z[p].z + y.z, z[p].w + y.w);
        }
    }
}
// the rows of the tile itself
template <bool WIDE>
__device__ __forceinline__ void own_rows(const Rows<WIDE>& X, int64_t tile, int64_t n, int li, int lk, float4 (&x)[4]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int64_t row = tile * kTile + 4 * p + lk;
        x[p] = X.part(row < n ? X.at(static_cast<int32_t>(row)) : X.kNone, li);
    }
}
// between the layouts, through the wave's 16 rows of LDS
__device__ __forceinline__ void tile_put(float* T, int li, int lk, const float4 (&z)[4]) {
    wave_fence();
#pragma unroll
    for (int p = 0; p < 4; ++p) *reinterpret_cast<float4*>(T + (4 * p + lk) * kWS + 4 * li) = z[p];
    wave_fence();
}
__device__ __forceinline__ void tile_get(float* T, int li, int lk, const floatx4 (&acc)[4], float4 (&y)[4]) {
    wave_fence();
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<floatx4*>(T + li * kWS + 16 * q + 4 * lk) = acc[q];
    wave_fence();
#pragma unroll
    for (int p = 0; p < 4; ++p) y[p] = *reinterpret_cast<const float4*>(T + (4 * p + lk) * kWS + 4 * li);
}

// sum += x w: the tile's rows x in T times 64 rows of weights (stride kWS), sums of 32 products
// each
__device__ __forceinline__ void product64(const float* Ws, const float* T, int li, int lk, floatx4 (&sum)[4]) {
    const float* w = Ws + 4 * lk * kWS + li;
#pragma unroll
    for (int q2 = 0; q2 < 2; ++q2) {
        floatx4 acc[4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) acc[ct] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 2 * q2; q < 2 * q2 + 2; ++q) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(T + li * kWS + 16 * q + 4 * lk);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int ct = 0; ct < 4; ++ct)
                    acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[(16 * q + e) * kWS + 16 * ct], x[e], acc[ct], 0, 0, 0);
            // the fence keeps the compiler from hoisting every weight read into registers at once
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) sum[ct] = sum[ct] + acc[ct];
    }
}

// Hout = relu((A H) W + H U + bias), W and U the halves of WU (64 x 128); with `out` also the
// head out = Hout w_out + b_out.
// At 773 293 nodes of 3.2 entries: 180 us, of which the matrix cores are busy for 81 (128 x 64
// products at 153 TFLOP/s); reading and writing H alone takes 106.  Both overlap only in part:
// the registers allow 16 waves a CU, and the neighbours' rows come from L2 with some 460 cycles
// each.  What mattered, from 268 us: whole rows per access in the gather (64-byte pieces of 16
// rows meet lines still on their way to L1; 247), the same for all other loads, and
// neighbouring tiles on different CUs (239 -> 195), stores past L2, which leave it to the rows
// that are gathered, and one workgroup of 16 waves (195 -> 180).  Four entries of each node in
// flight instead of two, wave priorities and skipping padded entries measured the same; 20
// waves of 96 registers 948 us a forward pass against 777.
template <int NT, bool WIDE>
__global__ void __launch_bounds__(NT, NT / 256) k_layer(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ nbr,
                                                 const float* __restrict__ a, const float* __restrict__ H,
                                                 const float* __restrict__ WU, const float* __restrict__ bias,
                                                 float* __restrict__ Hout, const float* __restrict__ wout,
                                                 const float* __restrict__ bout, float* __restrict__ out) {
    __shared__ float Ws[2 * kH * kWS];
    __shared__ float Ts[NT / kWave][kTile * kWS];
    __shared__ float bs[2 * kH];                          // bias, w_out
    const int t = threadIdx.x, lane = t % kWave, w = __builtin_amdgcn_readfirstlane(t / kWave), li = lane % 16, lk = lane / 16;
    for (int i = t; i < 2 * kH * kH; i += NT) {
        const int k = i / kH, j = i % kH;
        Ws[k * kWS + j] = WU[(k % kH) * 2 * kH + (k / kH) * kH + j];
    }
    if (t < kH) {
        bs[t] = bias[t];
        bs[kH + t] = wout[t];
    }
    __syncthreads();
    const Rows<WIDE> X(H, n);
    const TileRange tr = wave_tiles((n + kTile - 1) / kTile, NT / kWave, w);
    TileEntries te{tile_rows(rp, tr.first, n, lane), 0, 0.0f};
    tile_entries(nbr, a, lane, te);
    for (int64_t tile = tr.first; tile < tr.end; tile += tr.step) {
        // the next tile's entries are read while this one is multiplied
        const int32_t next = tile_rows(rp, tile + tr.step, n, lane);
        __builtin_amdgcn_sched_barrier(0);
        float4 z[4], h[4], y[4];
        gather_tile<WIDE>(nbr, a, X, te, li, lk, z);
        own_rows<WIDE>(X, tile, n, li, lk, h);
        te.rows = next;
        tile_entries(nbr, a, lane, te);
        floatx4 acc[4] = {};
        tile_put(Ts[w], li, lk, z);
        product64(Ws, Ts[w], li, lk, acc);
        tile_put(Ts[w], li, lk, h);
        product64(Ws + kH * kWS, Ts[w], li, lk, acc);
        tile_get(Ts[w], li, lk, acc, y);
        const float4 b4 = *reinterpret_cast<const float4*>(bs + 4 * li);
        const float4 w4 = *reinterpret_cast<const float4*>(bs + kH + 4 * li);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int64_t row = tile * kTile + 4 * p + lk;
            y[p] = make_float4(fmaxf(y[p].x + b4.x, 0.0f), fmaxf(y[p].y + b4.y, 0.0f), fmaxf(y[p].z + b4.z, 0.0f),
                               fmaxf(y[p].w + b4.w, 0.0f));
            if (row < n)
                __builtin_nontemporal_store(__builtin_bit_cast(floatx4, y[p]),
                                            reinterpret_cast<floatx4*>(Hout + row * kH + 4 * li));
            if (out) {
                float d = __builtin_fmaf(y[p].w, w4.w, __builtin_fmaf(y[p].z, w4.z, __builtin_fmaf(y[p].y, w4.y, y[p].x * w4.x)));
#pragma unroll
                for (int off = 8; off > 0; off >>= 1) d += __shfl_xor(d, off, kWave);
                if (row < n && li == 0) out[row] = d + bout[0];
            }
        }
    }
}

// From g = dL/d(layer's sum): Z = A^T g (for the weight gradients) and Gin = ([Z | g] [W | U]^T)
// masked by H > 0, the gradient at the sum of the layer below (H: this layer's input).  The
// layer kernel's shape and bounds: 42 us at 130 804 nodes; the four kernels that it replaces
// (mask, aggregation, product, column sums) took 107.
template <int NT, bool WIDE>
__global__ void __launch_bounds__(NT, NT / 256) k_layer_bwd(int64_t n, const int32_t* __restrict__ rp,
                                                     const int32_t* __restrict__ nbr, const float* __restrict__ a,
                                                     const float* __restrict__ G, const float* __restrict__ WU,
                                                     const float* __restrict__ H, float* __restrict__ Z,
                                                     float* __restrict__ Gin) {
    __shared__ float Ws[2 * kH * kWS];
    __shared__ float Ts[NT / kWave][kTile * kWS];
    const int t = threadIdx.x, lane = t % kWave, w = __builtin_amdgcn_readfirstlane(t / kWave), li = lane % 16, lk = lane / 16;
    for (int i = t; i < 2 * kH * kH; i += NT) {
        const int j = i / (2 * kH), k = i % (2 * kH);
        Ws[k * kWS + j] = WU[j * 2 * kH + k];
    }
    __syncthreads();
    const Rows<WIDE> X(G, n), Y(H, n);
    const TileRange tr = wave_tiles((n + kTile - 1) / kTile, NT / kWave, w);
    TileEntries te{tile_rows(rp, tr.first, n, lane), 0, 0.0f};
    tile_entries(nbr, a, lane, te);
    for (int64_t tile = tr.first; tile < tr.end; tile += tr.step) {
        const int32_t next = tile_rows(rp, tile + tr.step, n, lane);
        __builtin_amdgcn_sched_barrier(0);
        float4 z[4], own[4], h[4], y[4];
        gather_tile<WIDE>(nbr, a, X, te, li, lk, z);
        own_rows<WIDE>(X, tile, n, li, lk, own);
        te.rows = next;
        tile_entries(nbr, a, lane, te);
        floatx4 acc[4] = {};
        tile_put(Ts[w], li, lk, z);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int64_t row = tile * kTile + 4 * p + lk;
            if (row < n) *reinterpret_cast<float4*>(Z + row * kH + 4 * li) = z[p];
        }
        product64(Ws, Ts[w], li, lk, acc);
        tile_put(Ts[w], li, lk, own);
        own_rows<WIDE>(Y, tile, n, li, lk, h);
        product64(Ws + kH * kWS, Ts[w], li, lk, acc);
        tile_get(Ts[w], li, lk, acc, y);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int64_t row = tile * kTile + 4 * p + lk;
            if (row < n)
                *reinterpret_cast<float4*>(Gin + row * kH + 4 * li) =
                    make_float4(h[p].x > 0.0f ? y[p].x : 0.0f, h[p].y > 0.0f ? y[p].y : 0.0f, h[p].z > 0.0f ? y[p].z : 0.0f,
                                h[p].w > 0.0f ? y[p].w : 0.0f);
        }
    }
}

// Per block the partial sums of d[W | U] = H^T [Z | g] (64 x 128) and of the columns of g, over
// rows_per_block rows.  A wave takes four nodes a step: lane (li, lk) loads 16 bytes, columns
// 4 li .. 4 li + 3, of node lk's row of H, Z and g, and register e of the three is the operand
// of a product whose tile holds the features 4 li + e -- so three contiguous loads feed 32
// matrix instructions and nothing passes through LDS until the waves' sums are added, two and
// two.  31 us at 130 804 nodes against 91 for tiles staged in LDS; 14 at the matrix cores'
// rate, 20 for the three arrays' bytes.  A sum through one LDS array in wave order took 12 more.
constexpr int kWgradWaves = 8;      // two per SIMD, as many as the registers allow
__global__ void __launch_bounds__(64 * kWgradWaves, 2) k_wgrad(int64_t n, const float* __restrict__ H, const float* __restrict__ Z,
                                               const float* __restrict__ G, float* __restrict__ part,
                                               float* __restrict__ bpart, int rows_per_block) {
    __shared__ float sum[kWgradWaves / 2][kH * 2 * kH];
    __shared__ float bsum[kWgradWaves][kH];
    const int t = threadIdx.x, lane = t % kWave, w = t / kWave, li = lane % 16, lk = lane / 16;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < n ? r0 + rows_per_block : n;
    floatx4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float4 bs = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto load = [&](const float* X, int64_t r) {
        return r + lk < r1 ? *reinterpret_cast<const float4*>(X + (r + lk) * kH + 4 * li) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    };
    // the waves take the block's steps of four rows in turn; the next step's rows are loaded
    // while the current ones are multiplied
    int64_t r = r0 + 4 * w;
    float4 h = load(H, r), z = load(Z, r), g = load(G, r);
    for (; r < r1; r += 4 * kWgradWaves) {
        const int64_t rn = r + 4 * kWgradWaves;
        const float4 hn = load(H, rn), zn = load(Z, rn), gn = load(G, rn);
        const float ha[4] = {h.x, h.y, h.z, h.w};
        const float zg[8] = {z.x, z.y, z.z, z.w, g.x, g.y, g.z, g.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ha[i], zg[j], acc[i][j], 0, 0, 0);
        bs.x += g.x;
        bs.y += g.y;
        bs.z += g.z;
        bs.w += g.w;
        h = hn;
        z = zn;
        g = gn;
    }
    // column sums: the four node lanes, then the waves
    float b4[4] = {bs.x, bs.y, bs.z, bs.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        b4[e] += __shfl_xor(b4[e], 16, kWave);
        b4[e] += __shfl_xor(b4[e], 32, kWave);
        if (lk == 0) bsum[w][4 * li + e] = b4[e];
    }
    // acc[i][j][r] of lane (li, lk): row 4 (4 lk + r) + i, column 4 li + j % 4 of half j / 4
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) f((4 * (4 * lk + r4) + i) * 2 * kH + hf * kH + 4 * li, i, 4 * hf, r4);
    };
    auto put = [&](float* dst) {
        each([&](int o, int i, int j, int r4) {
            *reinterpret_cast<float4*>(dst + o) = make_float4(acc[i][j][r4], acc[i][j + 1][r4], acc[i][j + 2][r4], acc[i][j + 3][r4]);
        });
    };
    auto add = [&](const float* src) {
        each([&](int o, int i, int j, int r4) {
            const float4 v = *reinterpret_cast<const float4*>(src + o);
            acc[i][j][r4] += v.x;
            acc[i][j + 1][r4] += v.y;
            acc[i][j + 2][r4] += v.z;
            acc[i][j + 3][r4] += v.w;
        });
    };
#pragma unroll
    for (int s = 1; s < kWgradWaves; s *= 2) {
        if (w % (2 * s) == s) put(sum[w / (2 * s)]);
        __syncthreads();
        if (w % (2 * s) == 0) add(sum[w / (2 * s)]);
        __syncthreads();
    }
    if (w == 0) {
        float* dst = part + static_cast<int64_t>(blockIdx.x) * kH * 2 * kH;
        each([&](int o, int i, int j, int r4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[o + e] = acc[i][j + e][r4];
        });
    }
    if (t < kH) {
        float s = bsum[0][t];
#pragma unroll
        for (int i = 1; i < kWgradWaves; ++i) s += bsum[i][t];
        bpart[static_cast<int64_t>(blockIdx.x) * kH + t] = s;
    }
}

// H0 = relu(X W_in + b_in) for 8 features: 16 lanes per node, four columns each.  Bound by the
// write of H0: 51 us at 773 293 nodes (4.3 TB/s); the matrix kernel above takes 71, padded to
// a tile's rows in LDS.
__global__ void __launch_bounds__(256) k_input8(int64_t n, const float* __restrict__ X, const float* __restrict__ Win,
                                                const float* __restrict__ bin, float* __restrict__ H) {
    const int c = static_cast<int>(threadIdx.x % 16) * 4;
    float4 w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = *reinterpret_cast<const float4*>(Win + k * kH + c);
    const float4 b = *reinterpret_cast<const float4*>(bin + c);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 16 + threadIdx.x / 16; i < n; i += static_cast<int64_t>(gridDim.x) * 16) {
        const float4 x0 = *reinterpret_cast<const float4*>(X + i * 8), x1 = *reinterpret_cast<const float4*>(X + i * 8 + 4);
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            s.x = __builtin_fmaf(x[k], w[k].x, s.x);
            s.y = __builtin_fmaf(x[k], w[k].y, s.y);
            s.z = __builtin_fmaf(x[k], w[k].z, s.z);
            s.w = __builtin_fmaf(x[k], w[k].w, s.w);
        }
        *reinterpret_cast<float4*>(H + i * kH + c) = make_float4(fmaxf(s.x + b.x, 0.0f), fmaxf(s.y + b.y, 0.0f),
                                                                 fmaxf(s.z + b.z, 0.0f), fmaxf(s.w + b.w, 0.0f));
    }
}

// Sums over the 16 node groups of a 256-thread block (16 lanes x 4 columns each): the four
// groups of a wave by lane exchange, then the waves in order.  K vectors of 64 columns; row k
// goes to dst + 64 k.  sh: K x 4 x 64 floats.
template <int K>
__device__ __forceinline__ void block_columns(float (&v)[K][4], float* sh, float* __restrict__ dst) {
    const int t = threadIdx.x, lane = t % kWave, w = t / kWave, c = (t % 16) * 4;
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[k][e] += __shfl_xor(v[k][e], 16, kWave);
            v[k][e] += __shfl_xor(v[k][e], 32, kWave);
            if (lane < 16) sh[(k * 4 + w) * kH + c + e] = v[k][e];
        }
    __syncthreads();
    for (int i = t; i < K * kH; i += 256) {
        const float* s = sh + (i / kH) * 4 * kH + i % kH;
        dst[i] = ((s[0] + s[kH]) + s[2 * kH]) + s[3 * kH];
    }
}

// per-block partials of d W_in = X^T g (8 x 64) and d b_in (64), consecutive as in the
// parameters: 13 us at 130 804 nodes against 46 for a product and a column sum
__global__ void __launch_bounds__(256) k_input_grad8(int64_t n, const float* __restrict__ X, const float* __restrict__ G,
                                                     float* __restrict__ part) {
    __shared__ float sh[9 * 4 * kH];
    const int c = static_cast<int>(threadIdx.x % 16) * 4;
    float v[9][4] = {};
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 16 + threadIdx.x / 16; i < n; i += static_cast<int64_t>(gridDim.x) * 16) {
        const float4 x0 = *reinterpret_cast<const float4*>(X + i * 8), x1 = *reinterpret_cast<const float4*>(X + i * 8 + 4);
        const float4 g4 = *reinterpret_cast<const float4*>(G + i * kH + c);
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, g[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[k][e] = __builtin_fmaf(x[k], g[e], v[k][e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[8][e] += g[e];
    }
    block_columns<9>(v, sh, part + static_cast<int64_t>(blockIdx.x) * 9 * kH);
}

// The head backward: e = H4 w + b - target, g_i = 2 e_i / n; G = g w masked by H4 > 0 (the
// gradient at the last layer's sum), the losses of nodes 4 j .. 4 j + 3 summed in loss_part[j],
// and per-block partials of d w_out = H4^T g (64) and d b_out (the first of the next 64): one
// pass over H4, 17 us at 130 804 nodes, where the head, the sums and the mask took 86 in five.
__global__ void __launch_bounds__(256) k_head_bwd(int64_t n, const float* __restrict__ H, const float* __restrict__ w,
                                                  const float* __restrict__ b, const float* __restrict__ target,
                                                  float* __restrict__ G, float* __restrict__ loss_part,
                                                  float* __restrict__ part) {
    __shared__ float sh[2 * 4 * kH];
    const int t = threadIdx.x, lane = t % kWave, c = (t % 16) * 4;
    const float4 wc = *reinterpret_cast<const float4*>(w + c);
    const float b0 = b[0];
    float v[2][4] = {};
    for (int64_t i0 = static_cast<int64_t>(blockIdx.x) * 16; i0 < n; i0 += static_cast<int64_t>(gridDim.x) * 16) {
        const int64_t i = i0 + t / 16;
        const bool valid = i < n;
        const float4 h = valid ? *reinterpret_cast<const float4*>(H + i * kH + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float d = __builtin_fmaf(h.w, wc.w, __builtin_fmaf(h.z, wc.z, __builtin_fmaf(h.y, wc.y, h.x * wc.x)));
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) d += __shfl_xor(d, off, kWave);
        const float e = valid ? d + b0 - target[i] : 0.0f;
        const float g = 2.0f * e / static_cast<float>(n);
        if (valid)
            *reinterpret_cast<float4*>(G + i * kH + c) = make_float4(h.x > 0.0f ? g * wc.x : 0.0f, h.y > 0.0f ? g * wc.y : 0.0f,
                                                                     h.z > 0.0f ? g * wc.z : 0.0f, h.w > 0.0f ? g * wc.w : 0.0f);
        v[0][0] = __builtin_fmaf(h.x, g, v[0][0]);
        v[0][1] = __builtin_fmaf(h.y, g, v[0][1]);
        v[0][2] = __builtin_fmaf(h.z, g, v[0][2]);
        v[0][3] = __builtin_fmaf(h.w, g, v[0][3]);
        if (c == 0) v[1][0] += g;
        const float l = e * e;
        const float l1 = __shfl(l, 16, kWave), l2 = __shfl(l, 32, kWave), l3 = __shfl(l, 48, kWave);
        if (lane == 0 && i < n) loss_part[i / 4] = l + l1 + l2 + l3;
    }
    block_columns<2>(v, sh, part + static_cast<int64_t>(blockIdx.x) * 2 * kH);
}

__global__ void k_adam(int64_t n, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

unsigned nblk(int64_t n, int b) { return static_cast<unsigned>((n + b - 1) / b); }

// ---- per-node inputs of the network (nd_ws_features) ------------------------------------
// One thread per node, entries in CSR order: D = theta[j] - theta[i]; s0 = sum w (sin D - D),
// sum w D^2, max |D|, kdeg = sum w; the columns of X that need only the node's own entries.
constexpr int kFeat = 8;
__global__ void __launch_bounds__(256) k_ws_features(int64_t n, const int32_t* __restrict__ rp,
                                                     const int32_t* __restrict__ nbr, const double* __restrict__ w,
                                                     const double* __restrict__ th, const double* __restrict__ P,
                                                     const double* __restrict__ gen, double* __restrict__ s0,
                                                     double* __restrict__ X) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double ti = th[i];
    double s = 0.0, sq = 0.0, mx = 0.0, kd = 0.0;
    const int32_t k1 = rp[i + 1];
    for (int32_t k = rp[i]; k < k1; ++k) {
        const double D = th[nbr[k]] - ti, wk = w[k];
        s += wk * (sin(D) - D);
        sq += wk * D * D;
        mx = fmax(mx, fabs(D));
        kd += wk;
    }
    s0[i] = s;
    double* x = X + i * kFeat;
    x[0] = P[i];
    x[1] = gen[i];
    x[2] = kd > 0.0 ? log(kd) : 0.0;        // a node without entries: 0
    x[3] = static_cast<double>(k1 - rp[i]) / 6.0;
    x[4] = s;
    x[6] = sq;
    x[7] = mx;
}

// |F_i| / scale_i of the fixpoint residual F_i = P_i + sum_s w_s sin(theta[nbr_s] - theta_i),
// the quantity the batched Newton solver drives to its tolerance (entries in CSR order)
__global__ void __launch_bounds__(256) k_ws_residual(int64_t n, const int32_t* __restrict__ rp,
                                                     const int32_t* __restrict__ nbr, const double* __restrict__ w,
                                                     const double* __restrict__ th, const double* __restrict__ P,
                                                     const double* __restrict__ scale, double* __restrict__ r) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double ti = th[i];
    double F = P[i];
    const int32_t k1 = rp[i + 1];
    for (int32_t k = rp[i]; k < k1; ++k) F += w[k] * sin(th[nbr[k]] - ti);
    r[i] = fabs(F) / scale[i];
}

// the K-weighted neighbour mean of s0 (X column 5), after k_ws_features
__global__ void __launch_bounds__(256) k_ws_features_nbr(int64_t n, const int32_t* __restrict__ rp,
                                                         const int32_t* __restrict__ nbr, const double* __restrict__ w,
                                                         const double* __restrict__ s0, double* __restrict__ X) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    double ns = 0.0, kd = 0.0;
    const int32_t k1 = rp[i + 1];
    for (int32_t k = rp[i]; k < k1; ++k) {
        const double wk = w[k];
        ns += wk * s0[nbr[k]];
        kd += wk;
    }
    X[i * kFeat + 5] = kd > 0.0 ? ns / kd : 0.0;
}

struct Offsets {
    int64_t win, bin, wl[kLayers], bl[kLayers], wout, bout, total;
};
Offsets offsets(int F) {
    Offsets o{};
    int64_t k = 0;
    o.win = k; k += static_cast<int64_t>(F) * kH;
    o.bin = k; k += kH;
    for (int l = 0; l < kLayers; ++l) { o.wl[l] = k; k += kH * 2 * kH; o.bl[l] = k; k += kH; }
    o.wout = k; k += kH;
    o.bout = k; k += 1;
    o.total = k;
    return o;
}

int herr(hipError_t e, const char* w) {
    return e == hipSuccess ? ND_OK : nd::set_error(ND_ERR_DEVICE, "%s: %s", w, hipGetErrorString(e));
}

// the input layer for any feature count up to 128
void input_gemm(hipStream_t s, int64_t M, int K, const float* A, const float* B, float* C, const float* bias) {
    const size_t lds = gemm_mfma_lds_floats(K, kH) * sizeof(float);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_gemm_mfma<kH>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(lds));
    hipLaunchKernelGGL(k_gemm_mfma<kH>, dim3(nblk(M, 128)), dim3(256), lds, s, M, K, A, K, B, kH, C, kH, bias, 1);
}

// persistent workgroups over `groups` pieces of work, at most `most` of them
unsigned persistent(int64_t groups, int64_t most) { return static_cast<unsigned>(std::max<int64_t>(1, std::min(groups, most))); }

// The layer kernels run one workgroup per CU, of as many waves (16 nodes each) as that takes, up
// to 16: the weights are staged once per workgroup, and 16 waves are what the registers allow a
// CU anyway.  A forward pass over 485 / 15 327 / 30 850 / 77 268 / 773 293 nodes took 51 / 58 /
// 107 / 187 / 1099 us with 4 waves a workgroup (and up to four workgroups a CU), 52 / 59 / 92 /
// 129 / 805 with 8 (up to two) and 69 / 83 / 91 / 106 / 772 with 16.
struct LayerShape {
    unsigned blocks;
    int threads;
    bool wide;      // 2 GB of rows and more
};
LayerShape layer_shape(int64_t n) {
    constexpr int64_t kCus = 256;
    const int threads = n <= kCus * 64 ? 256 : n <= kCus * 128 ? 512 : 1024;
    return {persistent((n + threads / 4 - 1) / (threads / 4), kCus), threads, n >= int64_t(1) << 23};
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// out = A^T B over all M rows (KA <= 128, NB = 64): per-block partials, then a fixed-order sum
// (deterministic).  MFMA for KA <= 64, the FP32 VALU kernel above.
void gemm_tn(hipStream_t s, int64_t M, int KA, int NB, const float* A, int lda, const float* B, int ldb, float* part,
             float* out) {
    const int rows = part_rows(M);
    const unsigned nb = std::max(1u, nblk(M, rows));
    if (KA <= 64)
        hipLaunchKernelGGL(k_gemm_tn_mfma<4>, dim3(nb), dim3(256), 0, s, M, KA, NB, A, lda, B, ldb, part, rows);
    else
        hipLaunchKernelGGL(k_sgemm_tn_partial, dim3(nb), dim3(256), 0, s, M, KA, NB, A, lda, B, ldb, part, rows);
    hipLaunchKernelGGL(k_reduce_partials, dim3(nblk(KA * NB, kWave)), dim3(kRedWaves * 64), 0, s, static_cast<int>(nb),
                       KA * NB, KA * NB, part, out, 0, 0, nullptr, nullptr);
}

void colsum(hipStream_t s, int64_t M, const float* G, int ldg, float* part, float* out) {
    const int rows = part_rows(M);
    const unsigned nb = std::max(1u, nblk(M, rows));
    hipLaunchKernelGGL(k_colsum_partial, dim3(nb), dim3(256), 0, s, M, G, ldg, part, rows);
    hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(kRedWaves * 64), 0, s, static_cast<int>(nb), kH, kH, part, out, 0, 0,
                       nullptr, nullptr);
}

}  // namespace

extern "C" {

int64_t nd_mp_param_count(int32_t nfeat) { return offsets(nfeat).total; }

int64_t nd_mp_workspace_floats(int64_t nnodes) {
    // per node: activations H0..H4 (5*64), two gradients in turn and A^T g (3*64); then the
    // column sums' partials (64 per workgroup) and the other partial sums (at most 128 * 64 for
    // every 64 nodes).  Every array starts at a multiple of 64 floats.
    const int64_t nb = std::min<int64_t>(kMaxPartBlocks, (nnodes + 63) / 64);
    return nnodes * (8 * kH) + kWgradBlocks * kH + (nb + 2) * (kH * 2 * kH);
}

int nd_mp_forward(int64_t n, const int32_t* rowptr, const int32_t* nbr, const float* a_fwd, const float* X, int32_t nfeat,
                  const float* params, float* work, float* out, void* stream) {
    if (n < 1 || n > INT32_MAX - 8 || !rowptr || !X || !params || !work || !out || nfeat < 1 || nfeat > 128)
        return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    if ((reinterpret_cast<uintptr_t>(params) | reinterpret_cast<uintptr_t>(work)) & 15)
        return nd::set_error(ND_ERR_ARGUMENT, "params and work must be 16-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Offsets o = offsets(nfeat);
    float* H = work;                        // H_l at H + l*n*64
    const LayerShape sh = layer_shape(n);
    const auto layer = sh.wide ? k_layer<1024, true> : sh.threads == 1024 ? k_layer<1024, false>
                                                   : sh.threads == 512    ? k_layer<512, false> : k_layer<256, false>;
    if (nfeat == 8 && aligned16(X))
        hipLaunchKernelGGL(k_input8, dim3(persistent((n + 15) / 16, 2048)), dim3(256), 0, s, n, X, params + o.win,
                           params + o.bin, H);
    else
        input_gemm(s, n, nfeat, X, params + o.win, H, params + o.bin);
    for (int l = 0; l < kLayers; ++l) {
        const bool last = l == kLayers - 1;
        hipLaunchKernelGGL(layer, dim3(sh.blocks), dim3(sh.threads), 0, s, n, rowptr, nbr, a_fwd,
                           H + l * n * kH, params + o.wl[l], params + o.bl[l], H + (l + 1) * n * kH, params + o.wout,
                           params + o.bout, last ? out : nullptr);
    }
    return herr(hipGetLastError(), "nd_mp_forward");
}

// Gradient of the mean squared error; the forward pass must have filled `work`
// with the same inputs.  loss_part: n/4 + 1 floats of per-block loss sums.
int nd_mp_backward(int64_t n, const int32_t* rowptr, const int32_t* nbr, const float* a_bwd, const float* X,
                   int32_t nfeat, const float* params, const float* target, float* work, float* grads,
                   float* loss_part, void* stream) {
    if (n < 1 || n > INT32_MAX - 8 || !rowptr || !X || !params || !work || !grads || !target || !loss_part || nfeat < 1 ||
        nfeat > 128)
        return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    if ((reinterpret_cast<uintptr_t>(params) | reinterpret_cast<uintptr_t>(work)) & 15)
        return nd::set_error(ND_ERR_ARGUMENT, "params and work must be 16-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Offsets o = offsets(nfeat);
    float* H = work;
    float* G = work + 5 * n * kH;                 // gradients at the layers' sums, in turn: n x 64 each
    float* G2 = G + n * kH;
    float* Z = G2 + n * kH;                       // A^T g: n x 64
    float* bpart = Z + n * kH;                    // column-sum partials
    float* part = bpart + kWgradBlocks * kH;      // partials
    const LayerShape sh = layer_shape(n);
    const auto layer_bwd = sh.wide ? k_layer_bwd<1024, true> : sh.threads == 1024 ? k_layer_bwd<1024, false>
                                                           : sh.threads == 512    ? k_layer_bwd<512, false> : k_layer_bwd<256, false>;
    const unsigned hb = persistent((n + 15) / 16, kMaxPartBlocks);
    hipLaunchKernelGGL(k_head_bwd, dim3(hb), dim3(256), 0, s, n, H + 4 * n * kH, params + o.wout, params + o.bout, target, G,
                       loss_part, part);
    // w_out's 64 gradients and b_out's follow each other in the parameters and in a partial
    hipLaunchKernelGGL(k_reduce_partials, dim3(2), dim3(kRedWaves * 64), 0, s, static_cast<int>(hb), kH + 1, 2 * kH, part,
                       grads + o.wout, 0, 0, nullptr, nullptr);
    const int64_t wblocks = persistent((n + 63) / 64, kWgradBlocks);
    const int64_t wstep = 4 * kWgradWaves * wblocks;
    const int rows = static_cast<int>((n + wstep - 1) / wstep) * 4 * kWgradWaves;
    const unsigned wb = nblk(n, rows);
    for (int l = kLayers - 1; l >= 0; --l) {
        hipLaunchKernelGGL(layer_bwd, dim3(sh.blocks), dim3(sh.threads), 0, s, n, rowptr, nbr, a_bwd,
                           G, params + o.wl[l], H + l * n * kH, Z, G2);
        hipLaunchKernelGGL(k_wgrad, dim3(wb), dim3(64 * kWgradWaves), 0, s, n, H + l * n * kH, Z, G, part, bpart, rows);
        hipLaunchKernelGGL(k_reduce_partials, dim3(nblk(kH * 2 * kH, kWave) + 1), dim3(kRedWaves * 64), 0, s,
                           static_cast<int>(wb), kH * 2 * kH, kH * 2 * kH, part, grads + o.wl[l], static_cast<int>(wb), kH,
                           bpart, grads + o.bl[l]);
        std::swap(G, G2);
    }
    if (nfeat == 8 && aligned16(X)) {
        const unsigned ib = persistent((n + 15) / 16, kMaxPartBlocks);
        hipLaunchKernelGGL(k_input_grad8, dim3(ib), dim3(256), 0, s, n, X, G, part);
        hipLaunchKernelGGL(k_reduce_partials, dim3(nblk(9 * kH, kWave)), dim3(kRedWaves * 64), 0, s, static_cast<int>(ib),
                           9 * kH, 9 * kH, part, grads + o.win, 0, 0, nullptr, nullptr);
    } else {
        colsum(s, n, G, kH, part, grads + o.bin);
        gemm_tn(s, n, nfeat, kH, X, nfeat, G, kH, part, grads + o.win);
    }
    return herr(hipGetLastError(), "nd_mp_backward");
}

int nd_ws_features(int64_t n, const int32_t* rowptr, const int32_t* nbr, const double* w, const double* theta,
                   const double* P, const double* is_gen, double* s0, double* X, void* stream) {
    if (n < 1 || !rowptr || !nbr || !w || !theta || !P || !is_gen || !s0 || !X)
        return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_ws_features, dim3(nblk(n, 256)), dim3(256), 0, s, n, rowptr, nbr, w, theta, P, is_gen, s0, X);
    hipLaunchKernelGGL(k_ws_features_nbr, dim3(nblk(n, 256)), dim3(256), 0, s, n, rowptr, nbr, w, s0, X);
    return herr(hipGetLastError(), "nd_ws_features");
}

int nd_ws_residual(int64_t n, const int32_t* rowptr, const int32_t* nbr, const double* w, const double* theta,
                   const double* P, const double* scale, double* r, void* stream) {
    if (n < 1 || !rowptr || !nbr || !w || !theta || !P || !scale || !r) return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    hipLaunchKernelGGL(k_ws_residual, dim3(nblk(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), n, rowptr, nbr, w,
                       theta, P, scale, r);
    return herr(hipGetLastError(), "nd_ws_residual");
}

int nd_mp_adam(int64_t np, float* params, const float* grads, float* m, float* v, float lr, float b1, float b2,
               float eps, int64_t step, void* stream) {
    if (np < 1 || !params || !grads || !m || !v || step < 1) return nd::set_error(ND_ERR_ARGUMENT, "bad arguments");
    const float c1 = 1.0f - std::pow(b1, static_cast<float>(step));
    const float c2 = 1.0f - std::pow(b2, static_cast<float>(step));
    hipLaunchKernelGGL(k_adam, dim3(nblk(np, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), np, params, grads,
                       m, v, lr, b1, b2, eps, c1, c2);
    return herr(hipGetLastError(), "nd_mp_adam");
}

}  // extern "C"
