// Batched persistent Poisson solver (host side).
#pragma once

#include "common.hpp"

namespace sil {

struct BatchProblem {
    int64_t offset; // first node of the problem in the concatenated arrays
    int32_t side;   // n: the problem has n×n nodes, (n−2)² unknowns
    int32_t pad;
};

struct BatchResult {
    int32_t iterations;
    int32_t converged;
    double true_relative_residual;
};

struct BatchLaunch {
    const BatchProblem* problems;
    const int* order;
    int nprob;
    int* queue;
    const float *wx32, *wy32;
    const double *wx64, *wy64;
    const double* b;
    double* x;
    float *r, *p, *q;
    const float* dinv32;
    int jacobi;
    double tol;
    int max_it;
    int replace;
    BatchResult* results;
    int block; // workgroup size
    int grid;  // persistent workgroups
};

// Wide path: large problems, each spread over many workgroups.  A step of
// every problem is two kernels (batched.hip); kernel boundaries are the only
// synchronisation between workgroups.  Same arithmetic as the persistent
// kernel: FP32 recurrence, FP64 x, dot products and scalars, FP64 residual
// replacement, convergence only on the FP64 residual.
struct WideState {
    double bb, tol2bb, rz, rz_old, rr_ref, rr_true, beta;
    int32_t it, since, converged, done, mode;
    int32_t pcur; // direction buffer that holds the latest p
};

constexpr int kWideNodes = 1024;    // nodes of a workgroup per pass
constexpr int kWideMaxBlocks = 256; // most workgroups per problem (each sums the partials of all)

// a wide problem: its arrays, its workgroups and their partial sums
struct WideSlot {
    int64_t offset;
    int64_t offset2; // in the second direction buffer
    int32_t n, id;
    int32_t nb;   // workgroups
    int32_t part; // slot of the first one's partials
};

// workgroup `index` of wide problem `slot`
struct WideBlock {
    int32_t slot, index;
};

struct WideLaunch {
    const WideSlot* slots;
    int nwide;
    const WideBlock* full_map; // every workgroup of every problem
    int full_blocks;
    const WideBlock* map;      // the workgroups of the problems still running
    const int* nactive;        // their number
    const float *wx32, *wy32;
    const double *wx64, *wy64;
    const double* b;
    double* x;
    float* r;
    float* p[2]; // direction buffers: of all problems, of the wide ones
    float* q;
    const float* dinv32;
    int jacobi;
    double tol;
    int max_it;
    int replace;
    WideState* state;  // [step parity][nwide]
    double* part_pq;   // two values per workgroup
    double* part2[2];  // by step parity, two values per workgroup
    int* done;         // nwide flags (host-visible through a copy)
    BatchResult* results;
};

int wide_init(const WideLaunch& L, hipStream_t s);
// an even number of steps on `grid` workgroups
int wide_steps(const WideLaunch& L, int steps, int grid, hipStream_t s);
int wide_finish(const WideLaunch& L, hipStream_t s);

int batched_weights(const BatchProblem* problems_dev, int nprob, int max_side, const double* kappa, float* wx32,
                    float* wy32, double* wx64, double* wy64, float* dinv32, hipStream_t s);
int batched_enqueue(const BatchLaunch& L, hipStream_t s);
int batched_occupancy(int block, int* blocks_per_cu);

}  // namespace sil
