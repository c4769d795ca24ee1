// Wave and block reductions shared by the kernels.
//
// A wave's xor butterfly (offsets 32, 16, 8, 4, 2, 1) runs on lane permutes of the vector
// unit instead of the LDS permutes that __shfl_xor compiles to (a round trip of more than a
// hundred cycles each, twelve of them for one double):
//   32, 16  v_permlane32_swap / v_permlane16_swap: with both operands x the two results
//           hold, on every lane, x of the lower and of the upper partner;
//   8       row_ror:8, which is xor 8 within a row of 16;
//   4       row_ror:4: the values repeat every 8 lanes by then, so lane i + 4 holds what
//           lane i ^ 4 holds;
//   2, 1    quad_perm.
// Every step combines the same two values as the butterfly, so sums have the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace nd {

#if defined(__HIP_DEVICE_COMPILE__)
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ __forceinline__ double join_f64(unsigned lo, unsigned hi) {
    return __longlong_as_double((static_cast<long long>(hi) << 32) | lo);
}
// x of the lower (a) and the upper (b) partner at lane distance 32 or 16
template <int OFF>
__device__ __forceinline__ void partners(double v, double& a, double& b) {
    const long long x = __double_as_longlong(v);
    const unsigned lo = static_cast<unsigned>(x), hi = static_cast<unsigned>(x >> 32);
    if constexpr (OFF == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        a = join_f64(l[0], h[0]);
        b = join_f64(l[1], h[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        a = join_f64(l[0], h[0]);
        b = join_f64(l[1], h[1]);
    }
}
#else
template <int CTRL> __device__ __forceinline__ double dpp_f64(double v) { return v; }
template <int OFF> __device__ __forceinline__ void partners(double v, double& a, double& b) { a = b = v; }
#endif

// a value known to be the same on every lane, in scalar registers
__device__ __forceinline__ double uniform_f64(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(b)));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(b >> 32)));
    return __longlong_as_double((static_cast<long long>(hi) << 32) | lo);
}

struct SumOp {
    __device__ __forceinline__ double operator()(double a, double b) const { return a + b; }
};
struct MinOp {
    __device__ __forceinline__ double operator()(double a, double b) const { return fmin(a, b); }
};
// max that propagates NaN (fmax drops it): a residual with a NaN entry must read as NaN
struct MaxNanOp {
    __device__ __forceinline__ double operator()(double a, double b) const { return (b > a || b != b) ? b : a; }
};

// op over the 64 lanes of a full wave, on every lane
template <typename Op>
__device__ __forceinline__ double wave_reduce(double v, Op op) {
    double a, b;
    partners<32>(v, a, b);
    v = op(a, b);
    partners<16>(v, a, b);
    v = op(a, b);
    v = op(v, dpp_f64<0x128>(v));
    v = op(v, dpp_f64<0x124>(v));
    v = op(v, dpp_f64<0x4e>(v));
    return op(v, dpp_f64<0xb1>(v));
}

// Block reductions of at most 16 waves with one barrier each: the wave results go to one of
// two buffers of 16 doubles in turn, and every thread combines them in wave order.  A
// buffer is written again two reductions later, behind the barrier of the reduction in
// between, which every thread reaches only after it has read this one.
// NW: the waves that contribute (the first ones), 0 for all of the launch's.
template <int NW = 0>
struct BlockRedN {
    double* red;        // LDS: 32 doubles, 64 with sum2
    int turn = 0;
    int stride = 16;    // doubles per buffer: 32 with sum2

    template <typename Op>
    __device__ __forceinline__ double combine(const double* buf, int nw, Op op) {
        // all reads go out together; in-order combination, the same on every thread.  The
        // result is handed over through scalar registers, so branches on it are scalar ones
        constexpr int M = NW > 0 ? NW : 16;
        double x[M];
#pragma unroll
        for (int w = 0; w < M; ++w) x[w] = buf[NW > 0 || w < nw ? w : 0];
        double s = x[0];
#pragma unroll
        for (int w = 1; w < M; ++w)
            if (NW > 0 || w < nw) s = op(s, x[w]);
        return uniform_f64(s);
    }
    template <typename Op>
    __device__ __forceinline__ double reduce(double v, Op op) {
        v = wave_reduce(v, op);
        double* buf = red + stride * turn;
        turn ^= 1;
        const int t = static_cast<int>(threadIdx.x), nw = static_cast<int>(blockDim.x) / 64;
        if ((t & 63) == 0 && (NW == 0 || t < NW * 64)) buf[t / 64] = v;
        __syncthreads();
        return combine(buf, nw, op);
    }
    __device__ __forceinline__ double sum(double v) { return reduce(v, SumOp{}); }
    __device__ __forceinline__ double min(double v) { return reduce(v, MinOp{}); }
    __device__ __forceinline__ double max_nan(double v) { return reduce(v, MaxNanOp{}); }
    // two sums behind one barrier (stride 32)
    __device__ __forceinline__ void sum2(double& v, double& w) {
        v = wave_reduce(v, SumOp{});
        w = wave_reduce(w, SumOp{});
        double* buf = red + stride * turn;
        turn ^= 1;
        const int t = static_cast<int>(threadIdx.x), nw = static_cast<int>(blockDim.x) / 64;
        if ((t & 63) == 0 && (NW == 0 || t < NW * 64)) {
            buf[t / 64] = v;
            buf[16 + t / 64] = w;
        }
        __syncthreads();
        v = combine(buf, nw, SumOp{});
        w = combine(buf + 16, nw, SumOp{});
    }
};

using BlockRed = BlockRedN<0>;

}  // namespace nd
