// Device helpers shared by the matrix-free operator applications: the CG
// direction formed on the fly, the partial sums of a finished iteration and
// the per-block partial sums of ⟨in, out⟩.
#pragma once

#include <hipcub/hipcub.hpp>

#include "operators.hpp"

namespace sil {

constexpr int kApplyBlock = 256;

template <typename T>
__device__ __forceinline__ T p_value(const PUpdate<T>* pu, const T* x, int64_t idx)
{
    // value of the direction at row idx: either x[idx] or z + β p_old
    if (pu == nullptr) return x[idx];
    const double beta = *pu->beta;
    const double z = pu->inv_diag ? (double)pu->r[idx] * (double)pu->inv_diag[idx] : (double)pu->r[idx];
    return (T)(z + beta * (double)pu->p_old[idx]);
}

template <typename T>
__device__ __forceinline__ T p_value_of(const PUpdate<T>& pu, double beta, int64_t idx)
{
    const double z = pu.inv_diag ? (double)pu.r[idx] * (double)pu.inv_diag[idx] : (double)pu.r[idx];
    return (T)(z + beta * (double)pu.p_old[idx]);
}

// Sums of K partial-sum arrays in every thread of a workgroup of THREADS, in a
// fixed order (the same bits in every workgroup).  Up to 4 · THREADS values
// are in flight per array.
template <int THREADS, int K>
__device__ __forceinline__ void reduce_all(const double* const (&p)[K], const int (&count)[K], double (&out)[K])
{
    __shared__ double sh[K][THREADS / 64];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double v = 0.0;
        for (int i = threadIdx.x; i < count[k]; i += 4 * THREADS) {
            double q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = i + u * THREADS < count[k] ? p[k][i + u * THREADS] : 0.0;
            v += (q[0] + q[1]) + (q[2] + q[3]);
        }
        out[k] = v;
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
        for (int off = 32; off > 0; off >>= 1) out[k] += __shfl_xor(out[k], off, 64);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) sh[k][threadIdx.x >> 6] = out[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        out[k] = sh[k][0];
#pragma unroll
        for (int w = 1; w < THREADS / 64; ++w) out[k] += sh[k][w];
    }
}

// The previous iteration's end (β, the iteration count, the stopping test) in
// the first kernel of the next: every workgroup sums the partials itself and
// workgroup 0 records the scalars, so no kernel of one workgroup stands
// between the two (4.5 µs each at 2048 partials).  False: the solve is over.
template <int THREADS>
__device__ __forceinline__ bool cg_begin(const CgStep& st, double& beta)
{
    CgScalars& sc = *st.sc;
    const int s = st.slot;
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (st.part_rz == nullptr) {
        beta = sc.beta;
        if (first) {
            sc.rzs[s] = sc.rz;
            sc.iters[s] = sc.iter;
            sc.stops[s] = sc.done;
        }
        return !sc.done;
    }
    if (sc.stops[s ^ 1]) {
        if (first) sc.stops[s] = 1;
        return false;
    }
    double v[2];
    reduce_all<THREADS, 2>({st.part_rz, st.part_rr}, {st.count, st.count}, v);
    const double prev = sc.rzs[s ^ 1];
    const int it = sc.iters[s ^ 1] + 1;
    const bool conv = v[1] <= sc.tol2bb, stop = conv || it >= sc.max_iter;
    beta = v[0] / prev;
    if (first) {
        sc.rzs[s] = v[0];
        sc.iters[s] = it;
        sc.stops[s] = stop ? 1 : 0;
        sc.beta = beta;
        sc.rz_prev = prev;
        sc.rz = v[0];
        sc.rr = v[1];
        sc.iter = it;
        if (stop) {
            sc.done = 1;
            if (conv) sc.converged = 1;
        }
    }
    return !stop;
}

// one partial per workgroup of kApplyBlock threads
template <typename T>
__device__ __forceinline__ void block_dot_store(double v, double* partials)
{
    using BR = hipcub::BlockReduce<double, kApplyBlock>;
    __shared__ typename BR::TempStorage tmp;
    double s = BR(tmp).Sum(v);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

}  // namespace sil
