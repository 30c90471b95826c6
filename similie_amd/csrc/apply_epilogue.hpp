// Device helpers shared by the matrix-free operator applications: the CG
// direction formed on the fly, the partial sums of a finished iteration and
// the per-block partial sums of ⟨in, out⟩.
#pragma once

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

// v of the lane N places round its row of 16
template <int N>
__device__ __forceinline__ double row_rotate(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x120 + N, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x120 + N, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32));
}

__device__ __forceinline__ double read_lane(double v, int lane)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// the wavefront's sum in every lane, all lanes active: rotations within the
// rows of 16 (DPP, no LDS round trips as a shuffle makes), then the four rows
__device__ __forceinline__ double wave_sum(double v)
{
    v += row_rotate<8>(v);
    v += row_rotate<4>(v);
    v += row_rotate<2>(v);
    v += row_rotate<1>(v);
    return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

// Sums of K partial-sum arrays in every thread of a workgroup of THREADS, in a
// fixed order (the same bits in every workgroup).  Each array goes to one
// wavefront (K ≥ 3), or to half or all of them, sixteen loads a lane in flight.
template <int THREADS, int K>
__device__ __forceinline__ void reduce_all(const double* const (&p)[K], const int (&count)[K], double (&out)[K])
{
    constexpr int W = THREADS / 64, parts = K == 1 ? W : (K == 2 ? W / 2 : 1), U = 16;
    __shared__ double sh[K][parts];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % parts;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (wave / parts != k % (W / parts)) continue;
        double v = 0.0;
        for (int i = part * 64 + lane; i < count[k]; i += U * 64 * parts) {
            double q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = i + u * 64 * parts < count[k] ? p[k][i + u * 64 * parts] : 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u) v += q[u];
        }
        v = wave_sum(v);
        if (lane == 0) sh[k][part] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        out[k] = sh[k][0];
#pragma unroll
        for (int w = 1; w < parts; ++w) out[k] += sh[k][w];
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
    // (read before the sums, tested after: one round trip)
    const int over = sc.stops[s ^ 1], it = sc.iters[s ^ 1] + 1;
    const double prev = sc.rzs[s ^ 1], tol2bb = sc.tol2bb;
    const int max_iter = sc.max_iter;
    double v[2];
    reduce_all<THREADS, 2>({st.part_rz, st.part_rr}, {st.count, st.count}, v);
    if (over) {
        if (first) sc.stops[s] = 1;
        return false;
    }
    const bool conv = v[1] <= tol2bb, stop = conv || it >= max_iter;
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
    __shared__ double sh[kApplyBlock / 64];
    const double s = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = sh[0];
#pragma unroll
        for (int w = 1; w < kApplyBlock / 64; ++w) t += sh[w];
        partials[blockIdx.x] = t;
    }
}

}  // namespace sil
