// Per-node kernels of d, dᵀ, ⋆, δ and Δ with the dimension and the degree
// fixed at compile time: rectilinear grids with identity or diagonal metric
// and regular spacings (no node the reference treats as degenerate), N ≤ 3,
// any strides.  dec_generic.hip serves everything else.
//
// The general kernels keep N, k and every axis set in run-time loops, so
// their index and edge arrays live in scratch memory and the star of a node
// is derived again, with its square roots and divisions, for each
// coefficient read from it: 2.76 ms for Δ of a 2-form on 107 × 75 × 93 nodes,
// where the inputs and outputs take 11 µs to stream.  Here one thread per
// node reads the star of each node it touches once, as s_a and 1/s_a per
// axis (s_a = √|g_aa|·|h_a|, 1/h_a from the grid), every coefficient is a
// product of N of them, and all axis sets are template constants.  The
// neighbours' values come through the caches: consecutive threads hold
// consecutive nodes of the last axis.  Diagonal metric, general kernel → here:
//   Δ of a 2-form, 107 × 75 × 93 nodes     2753 → 21 µs
//   Δ of a 2-form, 256³ nodes              353 µs (1.8 TB/s)
//   δ of a 2-form, 129 × 120 × 135 nodes   1633 → 54 µs (2.8 TB/s)
//   Δ of a 1-form, 2048 × 1999 nodes       3742 → 83 µs
//   ⋆ of a 1-form, 256³ nodes              1931 → 251 µs (4.8 TB/s, a copy's rate)
//   d of a 1-form, 256³ nodes              1141 → 248 µs
// δ, ⋆ and d are bound by memory, Δ on 3D grids by the steps of its march
// (k_rect_lap3_march), elsewhere by the FP64 work of a node's stars.
#include "dec_kernels.hpp"

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

namespace sil {

namespace {

constexpr int kRectBlock = 256;

template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}

template <int N, int K>
constexpr int combos()
{
    return (K < 0 || K > N) ? 0 : kCombos.count[N][K];
}

// sign of axis A within the axis set M: (−1)^(number of smaller axes in M)
template <unsigned M, int A>
constexpr double axis_sign()
{
    return (popcount4(M & ((1u << A) - 1u)) & 1) ? -1.0 : 1.0;
}

template <int N>
struct RectView {
    uint32_t ext[N];
    int64_t str[N];
    int64_t cstr;
};

template <int N>
struct RectGeom {
    const double* __restrict__ h[N]; // spacing per node
    const double* __restrict__ r[N]; // 1 / spacing
    const double* __restrict__ g;    // [node][N], null for the identity
    uint32_t ext[N];
    int64_t node[N]; // node strides of g
};

template <int N>
struct Star {
    double s[N], r[N]; // s_a and 1/s_a
};

// s = √v |h| and r = 1/s = |1/h|/√v, v = |g|: the hardware estimate of 1/√v
// refined by two Newton–Raphson steps, then √v corrected by its residual
// v − q² and 1/s by 1 − s r, each to about half an ulp (without the
// corrections the operators are twice as far from FP64's exact results).
// v = 0, the reference's singular metric, leaves both at 0; v = ∞ gives ∞
// and 0.
__device__ __forceinline__ void axis_star(double g, double h, double rh, double& s, double& r)
{
    const double v = fabs(g);
    double y = __builtin_amdgcn_rsq(v);
    const double hv = 0.5 * v;
#pragma unroll
    for (int i = 0; i < 2; ++i) y = fma(y, fma(-(hv * y), y, 0.5), y);
    double q = v * y;
    q = fma(fma(-q, q, v), 0.5 * y, q);
    const bool end = v == 0.0 || v == __builtin_inf();
    y = end ? 0.0 : y;
    q = end ? v : q;
    s = q * fabs(h);
    r = y * fabs(rh);
    const double e = fma(-s, r, 1.0);
    r = end ? r : fma(e, r, r);
}

template <int N, bool DIAG>
__device__ __forceinline__ Star<N> load_star(const RectGeom<N>& g, const uint32_t (&idx)[N])
{
    Star<N> o;
    if constexpr (DIAG) {
        int64_t lin = 0;
#pragma unroll
        for (int a = 0; a < N; ++a) lin += (int64_t)idx[a] * g.node[a];
        double m[N];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < N; ++a) {
            m[a] = g.g[lin * N + a];
            ok = ok && m[a] != 0.0;
        }
#pragma unroll
        for (int a = 0; a < N; ++a) {
            // a zero entry makes the whole metric singular
            axis_star(ok ? m[a] : 0.0, g.h[a][idx[a]], g.r[a][idx[a]], o.s[a], o.r[a]);
        }
    } else {
#pragma unroll
        for (int a = 0; a < N; ++a) {
            o.s[a] = fabs(g.h[a][idx[a]]);
            o.r[a] = fabs(g.r[a][idx[a]]);
        }
    }
    return o;
}

// ⋆ from the axes SRC onto their complement: sign · Π_tgt s / Π_src s
template <int N, unsigned SRC>
__device__ __forceinline__ double star_coef(const Star<N>& o)
{
    constexpr int sign = concat_sign(SRC, ((1u << N) - 1u) & ~SRC, N);
    double v = (SRC & 1u) ? o.r[0] : o.s[0];
    if constexpr (N > 1) v *= (SRC & 2u) ? o.r[1] : o.s[1];
    if constexpr (N > 2) v *= (SRC & 4u) ? o.r[2] : o.s[2];
    return sign < 0 ? -v : v;
}

template <int N>
__device__ __forceinline__ void rect_decode(uint32_t t, const uint32_t (&ext)[N], uint32_t (&idx)[N])
{
#pragma unroll
    for (int a = N - 1; a > 0; --a) {
        idx[a] = t % ext[a];
        t /= ext[a];
    }
    idx[0] = t;
}

template <int N>
__device__ __forceinline__ int64_t rect_offset(const RectView<N>& v, const uint32_t (&idx)[N])
{
    int64_t o = 0;
#pragma unroll
    for (int a = 0; a < N; ++a) o += (int64_t)idx[a] * v.str[a];
    return o;
}

template <int N>
struct Node {
    uint32_t i[N];
};

// the node one step along axis A: forward clamped to the last node, backward
// to the first (where `has_back` says there is none)
template <int N, int A>
__device__ __forceinline__ Node<N> next(const Node<N>& n, const uint32_t (&ext)[N])
{
    Node<N> o = n;
    o.i[A] = n.i[A] + 1 < ext[A] ? n.i[A] + 1 : n.i[A];
    return o;
}

template <int N, int A>
__device__ __forceinline__ Node<N> back(const Node<N>& n)
{
    Node<N> o = n;
    o.i[A] = n.i[A] > 0 ? n.i[A] - 1 : 0;
    return o;
}

template <int N>
struct Form {
    const double* __restrict__ p;
    RectView<N> v;

    template <unsigned MASK>
    __device__ __forceinline__ double at(const Node<N>& n) const
    {
        constexpr int c = kCombos.index[N][MASK];
        return p[rect_offset<N>(v, n.i) + c * v.cstr];
    }

    // (dω)_M at n, samples clamped into the domain
    template <unsigned M>
    __device__ __forceinline__ double d(const Node<N>& n) const
    {
        double acc = 0.0;
        static_for<N>([&](auto A) {
            constexpr int a = decltype(A)::value;
            if constexpr ((M >> a) & 1u) {
                constexpr unsigned L = M & ~(1u << a);
                acc += axis_sign<M, a>() * (at<L>(next<N, a>(n, v.ext)) - at<L>(n));
            }
        });
        return acc;
    }
};

// (δβ)_I at n of a KQ-form β, β = ω or dω:
// s · ⋆ Σ_a ± [(⋆β)(n) − (⋆β)(n − e_a)], nothing before the first node
template <int N, int KQ, unsigned I, bool OF_D, class BackStar>
__device__ __forceinline__ double codiff(const Form<N>& w, const Node<N>& n, const Star<N>& sn, BackStar&& back_star)
{
    constexpr unsigned all = (1u << N) - 1u, dual = all & ~I;
    constexpr double s = ((N * (KQ + 1) + 1) % 2 == 1) ? -1.0 : 1.0;
    double G = 0.0;
    static_for<N>([&](auto A) {
        constexpr int a = decltype(A)::value;
        if constexpr ((dual >> a) & 1u) {
            constexpr unsigned src = I | (1u << a);
            auto beta = [&](const Node<N>& m) {
                if constexpr (OF_D)
                    return w.template d<src>(m);
                else
                    return w.template at<src>(m);
            };
            const double here = star_coef<N, src>(sn) * beta(n);
            const Node<N> b = back<N, a>(n);
            const double prev = star_coef<N, src>(back_star(A, b)) * beta(b);
            G += axis_sign<dual, a>() * (here - (n.i[a] > 0 ? prev : 0.0));
        }
    });
    return s * star_coef<N, dual>(sn) * G;
}

template <int N, int K>
__global__ __launch_bounds__(kRectBlock) void k_rect_coboundary(const double* __restrict__ in, RectView<N> vin,
                                                                double* __restrict__ out, RectView<N> vout,
                                                                uint32_t total)
{
    const Form<N> w{in, vin};
    for (uint32_t t = blockIdx.x * kRectBlock + threadIdx.x; t < total; t += gridDim.x * kRectBlock) {
        Node<N> n;
        rect_decode<N>(t, vout.ext, n.i);
        const int64_t o = rect_offset<N>(vout, n.i);
#pragma unroll
        for (int a = 0; a < N; ++a) n.i[a] = min(n.i[a], vin.ext[a] - 1);
        static_for<combos<N, K + 1>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            constexpr unsigned M = kCombos.mask[N][K + 1][c];
            out[o + c * vout.cstr] = w.template d<M>(n);
        });
    }
}

template <int N, int K, bool DIAG>
__global__ __launch_bounds__(kRectBlock) void k_rect_hodge(RectGeom<N> g, const double* __restrict__ in,
                                                           RectView<N> vin, double* __restrict__ out,
                                                           RectView<N> vout, uint32_t total)
{
    const Form<N> w{in, vin};
    for (uint32_t t = blockIdx.x * kRectBlock + threadIdx.x; t < total; t += gridDim.x * kRectBlock) {
        Node<N> n;
        rect_decode<N>(t, vout.ext, n.i);
        const int64_t o = rect_offset<N>(vout, n.i);
        const Star<N> s = load_star<N, DIAG>(g, n.i);
        static_for<combos<N, N - K>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            constexpr unsigned src = ((1u << N) - 1u) & ~kCombos.mask[N][N - K][c];
            out[o + c * vout.cstr] = star_coef<N, src>(s) * w.template at<src>(n);
        });
    }
}

template <int N, int K, bool DIAG>
__global__ __launch_bounds__(kRectBlock) void k_rect_codifferential(RectGeom<N> g, const double* __restrict__ in,
                                                                    RectView<N> vin, double* __restrict__ out,
                                                                    RectView<N> vout, uint32_t total)
{
    const Form<N> w{in, vin};
    for (uint32_t t = blockIdx.x * kRectBlock + threadIdx.x; t < total; t += gridDim.x * kRectBlock) {
        Node<N> n;
        rect_decode<N>(t, vout.ext, n.i);
        const int64_t o = rect_offset<N>(vout, n.i);
        const Star<N> s = load_star<N, DIAG>(g, n.i);
        Star<N> sb[N];
        static_for<N>([&](auto A) {
            constexpr int a = decltype(A)::value;
            sb[a] = load_star<N, DIAG>(g, back<N, a>(n).i);
        });
        static_for<combos<N, K - 1>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            constexpr unsigned I = kCombos.mask[N][K - 1][c];
            out[o + c * vout.cstr] = codiff<N, K, I, false>(
                w, n, s, [&](auto A, const Node<N>&) -> const Star<N>& { return sb[decltype(A)::value]; });
        });
    }
}

// Δ = δd + dδ.  Stars of n, n ± e_a and (for dδ, where a component moves along
// one axis and δ steps back along another) n + e_a − e_b.
template <int N, int K, bool DIAG>
__global__ __launch_bounds__(kRectBlock) void k_rect_laplacian(RectGeom<N> g, const double* __restrict__ in,
                                                               RectView<N> vin, double* __restrict__ out,
                                                               RectView<N> vout, uint32_t total)
{
    const Form<N> w{in, vin};
    for (uint32_t t = blockIdx.x * kRectBlock + threadIdx.x; t < total; t += gridDim.x * kRectBlock) {
        Node<N> n;
        rect_decode<N>(t, vout.ext, n.i);
        const int64_t o = rect_offset<N>(vout, n.i);
        const Star<N> s = load_star<N, DIAG>(g, n.i);
        Star<N> sb[N];
        static_for<N>([&](auto A) {
            constexpr int a = decltype(A)::value;
            sb[a] = load_star<N, DIAG>(g, back<N, a>(n).i);
        });
        auto sb_of = [&](auto A, const Node<N>&) -> const Star<N>& { return sb[decltype(A)::value]; };
        double acc[combos<N, K>()];
        static_for<combos<N, K>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            constexpr unsigned I = kCombos.mask[N][K][c];
            acc[c] = 0.0;
            if constexpr (K < N) acc[c] += codiff<N, K + 1, I, true>(w, n, s, sb_of);
        });
        if constexpr (K > 0) {
            // (dδω)_I = Σ_a ± [(δω)_{I∖a}(n + e_a) − (δω)_{I∖a}(n)], the
            // difference 0 at the last node of the axis
            static_for<N>([&](auto A) {
                constexpr int a = decltype(A)::value;
                const Node<N> f = next<N, a>(n, g.ext);
                const bool inner = n.i[a] + 1 < g.ext[a];
                const Star<N> sf = load_star<N, DIAG>(g, f.i);
                auto sf_back = [&](auto B, const Node<N>& m) {
                    constexpr int b = decltype(B)::value;
                    if constexpr (b == a)
                        return s; // f − e_a = n (at the last node f's value is dropped)
                    else
                        return load_star<N, DIAG>(g, m.i);
                };
                static_for<combos<N, K>()>([&](auto C) {
                    constexpr int c = decltype(C)::value;
                    constexpr unsigned I = kCombos.mask[N][K][c];
                    if constexpr ((I >> a) & 1u) {
                        constexpr unsigned J = I & ~(1u << a);
                        const double here = codiff<N, K, J, false>(w, n, s, sb_of);
                        const double ahead = codiff<N, K, J, false>(w, f, sf, sf_back);
                        acc[c] += axis_sign<I, a>() * ((inner ? ahead : here) - here);
                    }
                });
            });
        }
        static_for<combos<N, K>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            out[o + c * vout.cstr] = acc[c];
        });
    }
}

// Δ on 3D grids by a march along x: a workgroup owns 62 (z) × (TY − 2) (y)
// nodes with a one-node halo and walks a chunk of x planes, so a node's star is
// formed once per tile where k_rect_laplacian forms the stars of its 13 nodes.
// Registers hold ω, the stars, ⋆ω and δω of planes p and p + 1 and ⋆dω of
// p − 1; the y and z neighbours of ω, ⋆ω, ⋆dω and δω go through LDS, two
// barriers a plane; plane p + 2 is requested a step before it is used.  Sums
// and their order are those of k_rect_laplacian.  8 rows: two workgroups of a
// 1- or 2-form a compute unit (91–106 registers, 45–53 KB of LDS), four of a 0-
// or 3-form, which hide each other's barriers.  Diagonal metric, gather → march:
//   2-form  65³ 22 → 14, 107 × 75 × 93 67 → 21, 129 × 120 × 135 177 → 43,
//           256³ 1524 → 353 µs
//   0-form  256³ 395 → 198 µs;  3-form  256³ 607 → 190 µs
//   1-form  component-first, 256³ 1517 → 316 µs (index-last: dec_fused.hip)
template <int K, int TY>
struct MarchLds {
    double w[combos<3, K>()][TY][64];                       // ω(p): +y, +z neighbours of dω
    double b[K > 0 ? combos<3, K>() : 1][TY][64];           // ⋆ω(p + 1): −y, −z neighbours of δω
    double a[K < 3 ? combos<3, K + 1>() : 1][TY][64];       // ⋆dω(p): −y, −z neighbours of δdω
    double d[2][K > 0 ? combos<3, K - 1>() : 1][TY][64];    // δω(p), δω(p + 1): +y, +z neighbours of dδω
};

template <int K, bool DIAG, int TY>
__global__ __launch_bounds__(64 * TY) void k_rect_lap3_march(RectGeom<3> g, const double* __restrict__ in,
                                                             RectView<3> vin, double* __restrict__ out,
                                                             RectView<3> vout, int ntz, int nty, int chunk)
{
    constexpr int C = combos<3, K>(), CA = combos<3, K + 1>(), CD = combos<3, K - 1>();
    constexpr unsigned all = 7u;
    __shared__ MarchLds<K, TY> sm;
    const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
    // XCD-contiguous tiles: hardware places workgroup b on XCD b % 8
    int logical;
    {
        const int nb = gridDim.x, b = blockIdx.x;
        const int per = (nb + 7) / 8, rem = nb % 8;
        const int xcd = b % 8, slot = b / 8;
        const int full = rem == 0 ? 8 : rem;
        logical = (xcd < full) ? xcd * per + slot : full * per + (xcd - full) * (per - 1) + slot;
    }
    const int tz = logical % ntz, ty = (logical / ntz) % nty, tx = logical / (ntz * nty);
    const int64_t Nx = g.ext[0], Ny = g.ext[1], Nz = g.ext[2];
    const int64_t j = (int64_t)ty * (TY - 2) - 1 + row, k = (int64_t)tz * 62 - 1 + lane;
    const int64_t xa = (int64_t)tx * chunk, xb = min(xa + (int64_t)chunk, (int64_t)vout.ext[0]);
    const bool inside = j >= 0 && k >= 0 && j < Ny && k < Nz;
    const bool writer = row >= 1 && row <= TY - 2 && lane >= 1 && lane <= 62 && j < vout.ext[1] && k < vout.ext[2];
    const bool more_y = j + 1 < Ny, more_z = k + 1 < Nz; // a next node along y, z
    const int64_t jc = min(max(j, (int64_t)0), Ny - 1), kc = min(max(k, (int64_t)0), Nz - 1);
    const int rp = row + 1 < TY ? row + 1 : row, rm = row > 0 ? row - 1 : row;
    const int lp = lane < 63 ? lane + 1 : lane, lm = lane > 0 ? lane - 1 : lane;
    const double* col = in + jc * vin.str[1] + kc * vin.str[2];
    const double* gcol = DIAG ? g.g + 3 * (jc * g.node[1] + kc) : nullptr;
    const double hy = g.h[1][jc], ry = g.r[1][jc], hz = g.h[2][kc], rz = g.r[2][kc];

    // the raw values of plane x (clamped into the grid)
    struct Raw {
        double w[C], m[3], h, r;
    };
    auto request = [&](int64_t x, Raw& o) {
        const int64_t xc = min(max(x, (int64_t)0), Nx - 1);
        const double* p = col + xc * vin.str[0];
#pragma unroll
        for (int c = 0; c < C; ++c) o.w[c] = p[c * vin.cstr];
        if constexpr (DIAG) {
            const double* q = gcol + 3 * xc * g.node[0];
#pragma unroll
            for (int a = 0; a < 3; ++a) o.m[a] = q[a];
        }
        o.h = g.h[0][xc];
        o.r = g.r[0][xc];
    };
    auto star_of = [&](const Raw& o) {
        Star<3> s;
        if constexpr (DIAG) {
            const bool ok = o.m[0] != 0.0 && o.m[1] != 0.0 && o.m[2] != 0.0;
            axis_star(ok ? o.m[0] : 0.0, o.h, o.r, s.s[0], s.r[0]);
            axis_star(ok ? o.m[1] : 0.0, hy, ry, s.s[1], s.r[1]);
            axis_star(ok ? o.m[2] : 0.0, hz, rz, s.s[2], s.r[2]);
        } else {
            s.s[0] = fabs(o.h), s.r[0] = fabs(o.r);
            s.s[1] = fabs(hy), s.r[1] = fabs(ry);
            s.s[2] = fabs(hz), s.r[2] = fabs(rz);
        }
        return s;
    };

    double W[C], B[K > 0 ? C : 1], D[K > 0 ? CD : 1], Aback[K < 3 ? CA : 1];
    Star<3> S;
    Raw next;
    {
        // plane xa − 1: before the grid it contributes nothing
        Raw first;
        request(xa - 1, first);
        request(xa, next);
        S = star_of(first);
        const bool have = xa > 0 && inside;
#pragma unroll
        for (int c = 0; c < C; ++c) W[c] = first.w[c];
        if constexpr (K > 0)
            static_for<C>([&](auto I) {
                constexpr int c = decltype(I)::value;
                B[c] = have ? star_coef<3, kCombos.mask[3][K][c]>(S) * W[c] : 0.0;
            });
    }
    if constexpr (K < 3)
        for (int c = 0; c < CA; ++c) Aback[c] = 0.0;
    if constexpr (K > 0)
        for (int c = 0; c < CD; ++c) D[c] = 0.0;

    for (int64_t p = xa - 1; p < xb; ++p) {
        const bool more_x = p + 1 < Nx;
        const int buf = (int)(p & 1);
        Raw cur = next;
        request(p + 2, next);
        const Star<3> Sn = star_of(cur);
        double Wn[C], Bn[K > 0 ? C : 1];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            Wn[c] = cur.w[c];
            sm.w[c][row][lane] = W[c];
        }
        if constexpr (K > 0)
            static_for<C>([&](auto I) {
                constexpr int c = decltype(I)::value;
                Bn[c] = inside ? star_coef<3, kCombos.mask[3][K][c]>(Sn) * Wn[c] : 0.0;
                sm.b[c][row][lane] = Bn[c];
            });
        __syncthreads();

        // ⋆dω at plane p
        double A[K < 3 ? CA : 1];
        if constexpr (K < 3)
            static_for<CA>([&](auto I) {
                constexpr int c = decltype(I)::value;
                constexpr unsigned M = kCombos.mask[3][K + 1][c];
                double acc = 0.0;
                static_for<3>([&](auto AX) {
                    constexpr int a = decltype(AX)::value;
                    if constexpr ((M >> a) & 1u) {
                        constexpr int f = kCombos.index[3][M & ~(1u << a)];
                        const double here = W[f];
                        const double ahead = a == 0 ? (more_x ? Wn[f] : here)
                                                    : (a == 1 ? (more_y ? sm.w[f][rp][lane] : here)
                                                              : (more_z ? sm.w[f][row][lp] : here));
                        acc += axis_sign<M, a>() * (ahead - here);
                    }
                });
                A[c] = (inside && p >= 0) ? star_coef<3, M>(S) * acc : 0.0;
                sm.a[c][row][lane] = A[c];
            });
        // δω at plane p + 1
        double Dn[K > 0 ? CD : 1];
        if constexpr (K > 0)
            static_for<CD>([&](auto I) {
                constexpr int c = decltype(I)::value;
                constexpr unsigned J = kCombos.mask[3][K - 1][c], dual = all & ~J;
                constexpr double s = ((3 * (K + 1) + 1) % 2 == 1) ? -1.0 : 1.0;
                double G = 0.0;
                static_for<3>([&](auto AX) {
                    constexpr int a = decltype(AX)::value;
                    if constexpr ((dual >> a) & 1u) {
                        constexpr int f = kCombos.index[3][J | (1u << a)];
                        const double prev = a == 0 ? B[f] : (a == 1 ? sm.b[f][rm][lane] : sm.b[f][row][lm]);
                        G += axis_sign<dual, a>() * (Bn[f] - prev);
                    }
                });
                Dn[c] = s * star_coef<3, dual>(Sn) * G;
                sm.d[buf ^ 1][c][row][lane] = Dn[c];
            });
        __syncthreads();

        if (p >= xa && writer) {
            double* o = out + p * vout.str[0] + j * vout.str[1] + k * vout.str[2];
            static_for<C>([&](auto I) {
                constexpr int c = decltype(I)::value;
                constexpr unsigned M = kCombos.mask[3][K][c], dual = all & ~M;
                double acc = 0.0;
                if constexpr (K < 3) {
                    constexpr double s = ((3 * (K + 2) + 1) % 2 == 1) ? -1.0 : 1.0;
                    double G = 0.0;
                    static_for<3>([&](auto AX) {
                        constexpr int a = decltype(AX)::value;
                        if constexpr ((dual >> a) & 1u) {
                            constexpr int f = kCombos.index[3][M | (1u << a)];
                            const double prev = a == 0 ? Aback[f] : (a == 1 ? sm.a[f][rm][lane] : sm.a[f][row][lm]);
                            G += axis_sign<dual, a>() * (A[f] - prev);
                        }
                    });
                    acc += s * star_coef<3, dual>(S) * G;
                }
                if constexpr (K > 0)
                    static_for<3>([&](auto AX) {
                        constexpr int a = decltype(AX)::value;
                        if constexpr ((M >> a) & 1u) {
                            constexpr int f = kCombos.index[3][M & ~(1u << a)];
                            const double here = D[f];
                            const double ahead = a == 0 ? (more_x ? Dn[f] : here)
                                                        : (a == 1 ? (more_y ? sm.d[buf][f][rp][lane] : here)
                                                                  : (more_z ? sm.d[buf][f][row][lp] : here));
                            acc += axis_sign<M, a>() * (ahead - here);
                        }
                    });
                o[c * vout.cstr] = acc;
            });
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            W[c] = Wn[c];
            if constexpr (K > 0) B[c] = Bn[c];
        }
        if constexpr (K < 3)
            for (int c = 0; c < CA; ++c) Aback[c] = A[c];
        if constexpr (K > 0)
            for (int c = 0; c < CD; ++c) D[c] = Dn[c];
        S = Sn;
    }
}

template <int N>
RectView<N> rect_view(const sil_view& v)
{
    RectView<N> r{};
    for (int a = 0; a < N; ++a) {
        r.ext[a] = static_cast<uint32_t>(v.extent[a]);
        r.str[a] = v.stride[a];
    }
    r.cstr = v.comp_stride;
    return r;
}

template <int N>
RectGeom<N> rect_geom(const DevGeom& g)
{
    RectGeom<N> r{};
    int64_t lin = 1;
    for (int a = N - 1; a >= 0; --a) {
        r.h[a] = g.spacing[a];
        r.r[a] = g.inv_spacing[a];
        r.ext[a] = static_cast<uint32_t>(g.ext[a]);
        r.node[a] = lin;
        lin *= g.ext[a];
    }
    r.g = g.metric_kind == SIL_METRIC_DIAGONAL ? g.metric : nullptr;
    return r;
}

inline dim3 rect_grid(uint32_t total)
{
    return dim3(std::min<uint32_t>((total + kRectBlock - 1) / kRectBlock, 1u << 20));
}

constexpr int kMarchRows = 8;

struct March {
    int ntz, nty, chunk;
    int64_t blocks; // 0: k_rect_laplacian
};

// The march takes a grid where enough of its lanes hold nodes to write, and a
// 0- or 3-form also needs 500 000 nodes: below, the gather of 7 stars is the
// shorter chain (65³, 0-form, diagonal metric: 8.7 against 10.7 µs; 107 × 75 ×
// 93: 19 against 16).  A gather costs a node 2 (0-form) to 5 times (2-form,
// diagonal metric) a lane's step here.  On 256 × 256 × z nodes, gather / march:
//   0-form, diagonal   z = 25: 32/40    z = 33: 42/40
//   2-form, identity   z = 17: 34/43    z = 25: 49/43
//   2-form, diagonal   z = 9:  41/56    z = 17: 76/56
//   3-form, diagonal   z = 17: 35/38    z = 25: 49/38
template <int K, bool DIAG>
March march_shape(const RectView<3>& o)
{
    March m{};
    m.ntz = (int)((o.ext[2] + 61) / 62);
    m.nty = (int)((o.ext[1] + kMarchRows - 3) / (kMarchRows - 2));
    const int64_t tiles = (int64_t)m.ntz * m.nty, column = (int64_t)o.ext[1] * o.ext[2];
    constexpr bool ends = K == 0 || K == 3;
    constexpr double used = K == 0 ? 0.375 : (!ends && DIAG ? 0.125 : 0.25);
    if ((ends && column * o.ext[0] < 500000) || (double)column < used * 64 * kMarchRows * (double)tiles) return m;
    m.chunk = march_chunk(tiles, o.ext[0], ends ? 4 : 2, &m.blocks);
    if (m.blocks > INT32_MAX) m.blocks = 0;
    return m;
}

template <int N, int K>
void rect_launch(RectOp op, const DevGeom* g, const double* in, const sil_view& vin, double* out,
                 const sil_view& vout, uint32_t total, hipStream_t stream)
{
    const dim3 grid = rect_grid(total), block(kRectBlock);
    const RectView<N> vi = rect_view<N>(vin), vo = rect_view<N>(vout);
    if (op == RectOp::Coboundary) {
        if constexpr (K < N)
            hipLaunchKernelGGL((k_rect_coboundary<N, K>), grid, block, 0, stream, in, vi, out, vo, total);
        return;
    }
    const RectGeom<N> rg = rect_geom<N>(*g);
    auto go = [&](auto D) {
        constexpr bool diag = decltype(D)::value;
        if (op == RectOp::Hodge)
            hipLaunchKernelGGL((k_rect_hodge<N, K, diag>), grid, block, 0, stream, rg, in, vi, out, vo, total);
        else if (op == RectOp::Laplacian) {
            if constexpr (N == 3) {
                const March m = march_shape<K, diag>(vo);
                if (m.blocks > 0) {
                    hipLaunchKernelGGL((k_rect_lap3_march<K, diag, kMarchRows>), dim3((unsigned)m.blocks),
                                       dim3(64 * kMarchRows), 0, stream, rg, in, vi, out, vo, m.ntz, m.nty, m.chunk);
                    return;
                }
            }
            hipLaunchKernelGGL((k_rect_laplacian<N, K, diag>), grid, block, 0, stream, rg, in, vi, out, vo, total);
        }
        else if constexpr (K > 0)
            hipLaunchKernelGGL((k_rect_codifferential<N, K, diag>), grid, block, 0, stream, rg, in, vi, out, vo,
                               total);
    };
    if (rg.g)
        go(std::true_type{});
    else
        go(std::false_type{});
}

}  // namespace

// Views the compile-time kernels take: N ≤ 3, no spectator dimensions, node
// indices in 32 bits (the grid's stride included), a non-empty input.
bool rect_views_ok(const sil_view& vin, const sil_view& vout)
{
    if (vin.ndim > 3 || vin.nbatch != 0 || vout.nbatch != 0) return false;
    for (int a = 0; a < vin.ndim; ++a)
        if (vin.extent[a] < 1 || vin.extent[a] > INT32_MAX || vout.extent[a] > INT32_MAX) return false;
    return view_nodes(vout) > 0 && view_nodes(vout) < (1LL << 31);
}

int launch_rect(RectOp op, int k, const DevGeom* g, const double* in, const sil_view& vin, double* out,
                const sil_view& vout, hipStream_t stream)
{
    const uint32_t total = static_cast<uint32_t>(view_nodes(vout));
    auto go = [&](auto NN, auto KK) {
        rect_launch<decltype(NN)::value, decltype(KK)::value>(op, g, in, vin, out, vout, total, stream);
    };
    using std::integral_constant;
    auto degrees = [&](auto NN) {
        constexpr int n = decltype(NN)::value;
        if (k == 0) go(NN, integral_constant<int, 0>{});
        if (k == 1) go(NN, integral_constant<int, 1>{});
        if constexpr (n >= 2)
            if (k == 2) go(NN, integral_constant<int, 2>{});
        if constexpr (n >= 3)
            if (k == 3) go(NN, integral_constant<int, 3>{});
    };
    if (vin.ndim == 1) degrees(integral_constant<int, 1>{});
    if (vin.ndim == 2) degrees(integral_constant<int, 2>{});
    if (vin.ndim == 3) degrees(integral_constant<int, 3>{});
    SIL_LAUNCH_CHECK();
    return SIL_OK;
}

}  // namespace sil
