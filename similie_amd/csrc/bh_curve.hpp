// Interpolated B-H curve, device side (InterpolatedNonlinearBHCurve,
// src/similie/physics/magnetostatics/nonlinear_magnetostatics.py:14-181):
// h(b) is linear between samples, bracketed on q = b², constant h₀ below
// the first sample and extrapolated along the last segment past the end.
#pragma once

#include "operators.hpp"

namespace sil {

// The curve in LDS with its brackets laid out for a branch-free search: the
// bracket of q is the number of edges below it.  (A search that stops at the
// bracket is a chain of dependent reads, twice per node, and cost the curl-curl
// march more than its memory: 83 µs for F on 113 × 97 × 129 nodes, 34 with the
// count.)
struct BhEdges {
    alignas(16) double edge[kBhMax];
    int n;
};

struct BhTable : BhEdges {
    double b[kBhMax], h[kBhMax], dh_db[kBhMax];
};

// by every thread of the workgroup; the caller's barrier follows
__device__ __forceinline__ void load_bh_edges(BhEdges& t, const BhCurve* __restrict__ c)
{
    for (int i = threadIdx.x; i < kBhMax; i += blockDim.x) t.edge[i] = c->edge[i];
    if (threadIdx.x == 0) t.n = c->n;
}

__device__ __forceinline__ void load_bh_table(BhTable& t, const BhCurve* __restrict__ c)
{
    for (int i = threadIdx.x; i < kBhMax; i += blockDim.x) {
        // (b, h and dh_db past the last sample are never read)
        const double e = c->edge[i], b = c->b[i], h = c->h[i], dh = c->dh_db[i];
        t.edge[i] = e;
        t.b[i] = b;
        t.h[i] = h;
        t.dh_db[i] = dh;
    }
    if (threadIdx.x == 0) t.n = c->n;
}

// the bracket of q = b²
__device__ __forceinline__ int bh_bracket(const BhEdges& t, double q)
{
    typedef double D2 __attribute__((ext_vector_type(2)));
    int i = 0;
    for (int m = 0; m < t.n - 2; m += 8) {
        const D2* e = reinterpret_cast<const D2*>(&t.edge[m]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const D2 v = e[u];
            i += (q > v[0] ? 1 : 0) + (q > v[1] ? 1 : 0);
        }
    }
    return i;
}

// h(b) on bracket i of a table or the curve itself: constant below the first
// sample, along the last segment past the end
template <class Curve>
__device__ __forceinline__ double bh_h(const Curve& t, int i, double b)
{
    return b <= t.b[0] ? t.h[0] : t.h[i] + t.dh_db[i] * (b - t.b[i]);
}

// The response of a node whose induction squares to q.  With the energy
// ½ q f(q), f = h(b)/b, q = b²:
//   ∂H/∂B = a B,  ∂²H/∂B∂B = a I + c B Bᵀ,
//   a = f + q f′ = (h/b + h′)/2,   c = 2 (2 f′ + q f″) = (h′ − h/b)/(2 q)
// (f′ = (h′ b − h)/(2 b³), f″ by one more derivative: h″ = 0 on a segment).
__device__ __forceinline__ void bh_response(const BhTable& t, double q, double& a, double& c)
{
    const double b = sqrt(q);
    const int i = bh_bracket(t, b * b);
    const double dh = t.dh_db[i], h = bh_h(t, i, b);
    const bool zero = q == 0.0;
    const double f = zero ? dh : h / b;
    a = 0.5 * (f + dh);
    c = zero ? 0.0 : (dh - f) / (2.0 * q);
}

}  // namespace sil
