// Device-side reduction helpers shared by the vector and PCG kernels.
// Wave64 shuffle tree, then an LDS tree across the workgroup's wavefronts;
// per-workgroup partials are stored with plain stores and combined, in a
// fixed order, by a later kernel (no atomics, no device-scope fences).
#pragma once

#include <hip/hip_runtime.h>

#include "gip_internal.h"

namespace gip {

enum { RED_SUM = 0, RED_MAXABS = 1, RED_MIN = 2 };

template <int OP>
struct RedOp;

template <>
struct RedOp<RED_SUM> {
    __device__ static double identity() { return 0.0; }
    __device__ static double combine(double a, double b) { return a + b; }
    __device__ static double term(const double *x, const double *y, int i) { return x[i] * y[i]; }
};

template <>
struct RedOp<RED_MAXABS> {
    __device__ static double identity() { return 0.0; }
    // NaN terms never replace the running value, as in GIP_VectorMulticore.cpp:151-153
    __device__ static double combine(double a, double b) { return b > a ? b : a; }
    __device__ static double term(const double *x, const double *, int i) { return fabs(x[i]); }
};

template <>
struct RedOp<RED_MIN> {
    __device__ static double identity() { return 1e20; }
    __device__ static double combine(double a, double b) { return b < a ? b : a; }
    __device__ static double term(const double *x, const double *, int i) { return x[i]; }
};

constexpr int kWaves = kBlock / 64;  // wavefronts per workgroup

// v of lane i - (CTRL - 0x110) within the lane's row of 16 (0 past the
// row's start): a DPP row shift, moved as two 32-bit halves
template <int CTRL>
__device__ inline double dpp_row_shr(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Wavefront sums by DPP: an inclusive scan of each row of 16 lanes, then row
// 0's total onto row 1's and row 2's onto row 3's (row broadcast), then lane
// 31's onto the last row: a fixed order, no LDS, no lane reads.  The total
// is in lane 63 (18 vector instructions).
template <int CTRL, int ROWS>
__device__ inline double dpp_row_bcast(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ inline double half_sum_dpp(double v) {  // lanes 31 and 63: the totals of their halves
    v = v + dpp_row_shr<0x111>(v);
    v = v + dpp_row_shr<0x112>(v);
    v = v + dpp_row_shr<0x114>(v);
    v = v + dpp_row_shr<0x118>(v);
    return v + dpp_row_bcast<0x142, 0xa>(v);
}
__device__ inline double wave_sum_63(double v) {
    v = half_sum_dpp(v);
    return v + dpp_row_bcast<0x143, 0xc>(v);
}
// Two sums for little more than one: the lower half of the wavefront takes
// a, the upper half b (each lane's value and the one 32 lanes on), and the
// halves are summed together.  a's total is in lane 31, b's in lane 63.
__device__ inline double wave_sum_two(double a, double b) {
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    const double p = __longlong_as_double(((long long)hi[0] << 32) | (long long)lo[0]);
    const double q = __longlong_as_double(((long long)hi[1] << 32) | (long long)lo[1]);
    return half_sum_dpp(p + q);
}
// Reduce v over the workgroup; the result is valid in thread 0.
template <int OP>
__device__ inline double block_reduce(double v) {
    __shared__ double sh[kBlock / 64];
    __syncthreads();  // protect sh against a previous call
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = RedOp<OP>::combine(v, __shfl_down(v, off, 64));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        v = sh[0];
#pragma unroll
        for (int k = 1; k < kBlock / 64; ++k) v = RedOp<OP>::combine(v, sh[k]);
    }
    return v;
}

// M sums over the workgroup at once, valid in thread 0: each value takes
// block_reduce's shuffle tree and final order (so each total is bitwise
// block_reduce<RED_SUM>'s), and all M share one LDS exchange and its pair
// of barriers.
template <int M>
__device__ inline void block_reduce_n(double (&v)[M]) {
    __shared__ double sh[M][kBlock / 64];
    __syncthreads();  // protect sh against a previous call
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[m] = v[m] + __shfl_down(v[m], off, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int m = 0; m < M; ++m) sh[m][wid] = v[m];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            v[m] = sh[m][0];
#pragma unroll
            for (int k = 1; k < kBlock / 64; ++k) v[m] = v[m] + sh[m][k];
        }
}

// M sums of partials at once, for partial arrays of kMaxRedBlocks doubles
// whose entries past their producer's grid hold zeros.  Every load is
// issued unconditionally (a load under a bounds test would be turned into a
// branch with a wait at its join): a slot past n[m] is read from the array's
// last entry, a zero whenever n[m] < kMaxRedBlocks, so those reads are one
// broadcast cache line.  All loads are issued before the first is used
// (load(), early in a kernel) and reduce() sums them: the M sums cost one
// memory round trip.  The zero slots make each total bitwise the one
// sum_partials<RED_SUM> gives over the first n[m] entries.
template <int M>
struct PaddedSums {
    static constexpr int K = kMaxRedBlocks / kBlock;
    double v[M][K];
    __device__ inline void load(const double *const (&part)[M], const int (&n)[M]) {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int i = threadIdx.x + k * kBlock;
                v[m][k] = part[m][i < n[m] ? i : kMaxRedBlocks - 1];
            }
    }
    __device__ inline void reduce(double (&out)[M]) {
        __shared__ double s_all[M];
        double acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            acc[m] = 0.0;
#pragma unroll
            for (int k = 0; k < K; ++k) acc[m] = acc[m] + v[m][k];
        }
        block_reduce_n<M>(acc);
        if (threadIdx.x == 0)
#pragma unroll
            for (int m = 0; m < M; ++m) s_all[m] = acc[m];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m) out[m] = s_all[m];
    }
};

template <int M>
__device__ inline void sum_padded(const double *const (&part)[M], const int (&n)[M], double (&out)[M]) {
    PaddedSums<M> ps;
    ps.load(part, n);
    ps.reduce(out);
}

// Combine n partials in index order (thread t takes t, t+256, ..., then the
// fixed tree): the same value in every workgroup that calls it.  Used in
// kernel prologues to read the previous kernel's per-workgroup partials
// without atomics or cross-XCD fences (the kernel boundary orders them).
template <int OP>
__device__ inline double sum_partials(const double *__restrict__ part, int n) {
    __shared__ double s_all;
    // n <= kMaxRedBlocks: all of a thread's loads are issued before the first
    // is used (one memory round trip), then combined in index order
    constexpr int K = kMaxRedBlocks / kBlock;
    double v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = threadIdx.x + k * kBlock;
        v[k] = i < n ? part[i] : RedOp<OP>::identity();
    }
    double acc = RedOp<OP>::identity();
#pragma unroll
    for (int k = 0; k < K; ++k) acc = RedOp<OP>::combine(acc, v[k]);
    acc = block_reduce<OP>(acc);
    if (threadIdx.x == 0) s_all = acc;
    __syncthreads();
    return s_all;
}

// M arrays of n partials summed together (n <= kMaxRedBlocks): only the
// slots below n are read, in a workgroup-uniform loop of ceil(n / 256)
// rounds, the M arrays' loads of a round issued together; the same total in
// every workgroup (thread t takes t, t+256, ..., then the fixed tree).
template <int M>
__device__ inline void sum_partials_n(const double *const (&part)[M], int n, double (&out)[M]) {
    __shared__ double s_all[M];
    double acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.0;
    const int rounds = (n + kBlock - 1) / kBlock;
    for (int k = 0; k < rounds; ++k) {
        const int i = threadIdx.x + k * kBlock;
        double v[M];
#pragma unroll
        for (int m = 0; m < M; ++m) v[m] = i < n ? part[m][i] : 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = acc[m] + v[m];
    }
    block_reduce_n<M>(acc);
    if (threadIdx.x == 0)
#pragma unroll
        for (int m = 0; m < M; ++m) s_all[m] = acc[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) out[m] = s_all[m];
}

int launch_reduce(gip_ctx *c, int op, int n, const double *x, const double *y, double *dres);

}  // namespace gip
