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
// node forms the star of each node it touches once (star_of_edges), and
// all axis sets are template constants.  The neighbours' values come through the
// caches: consecutive threads hold consecutive nodes of the last axis.  Diagonal
// metric, general kernel → here (repeated calls, whose inputs stay in the 256 MB
// cache in front of HBM up to that size; δ below takes 51 µs without):
//   Δ of a 2-form, 107 × 75 × 93 nodes     2753 → 19 µs
//   Δ of a 2-form, 256³ nodes              327 µs (3.7 TB/s)
//   δ of a 2-form, 129 × 120 × 135 nodes   1633 → 41 µs (3.7 TB/s)
//   Δ of a 1-form, 2048 × 1999 nodes       3742 → 79 µs
//   ⋆ of a 1-form, 256³ nodes              1931 → 235 µs (5.1 TB/s, a copy's rate)
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
    const double* __restrict__ g;    // [node][N], null for the identity
    uint32_t ext[N];
    int64_t node[N]; // node strides of g
};

// The ⋆ coefficient of each source axis set, sign left out: Π_tgt s / Π_src s,
// s_a = √|g_aa|·|h_a|
template <int N>
struct Star {
    double c[1 << N];
};

// n / d, y ≈ 1/d: one rounding where a product with a rounded 1/d has two
__device__ __forceinline__ double quotient(double n, double d, double y)
{
    const double q = n * y;
    return fma(fma(-d, q, n), y, q);
}

// the hardware's estimate of 1/d (2⁻²⁴) after a Newton–Raphson step: a first
// guess for quotient
__device__ __forceinline__ double guess_reciprocal(double d)
{
    const double y = __builtin_amdgcn_rcp(d);
    return fma(y, fma(-d, y, 1.0), y);
}

// √v to half an ulp: the hardware's estimate of 1/√v (2⁻²⁴), one of Goldschmidt's
// steps and a correction by the residual v − g²
__device__ __forceinline__ double root(double v)
{
    const double y = __builtin_amdgcn_rsq(v);
    double g = v * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    return fma(fma(-g, g, v), h, g);
}

// the star of the edge measures s (in the plain range, see diag_star): the
// quotients of products that the general kernels form, with 1/V, V = Π s, as the
// first guess of every quotient's reciprocal (1/d = n/V).  Products of s and of
// rounded 1/s, which stood here before, round once more per source axis: rms of
// a coefficient, N = 3, k = 1 to 3, identity metric 8.2, 9.4, 10.5 · 1e-17, now
// 6.7, 6.7, 8.2 as in the general kernels.
template <int N>
__device__ __forceinline__ Star<N> star_of_edges(const double (&s)[N])
{
    Star<N> o;
    double V = 1.0;
#pragma unroll
    for (int a = 0; a < N; ++a) V *= s[a];
    const double y = guess_reciprocal(V);
    static_for<1 << N>([&](auto SRC) {
        constexpr unsigned src = decltype(SRC)::value;
        double num = 1.0, den = 1.0;
#pragma unroll
        for (int a = 0; a < N; ++a) ((src >> a) & 1u ? den : num) *= s[a];
        o.c[src] = src == 0 ? V : quotient(num, den, num * y);
    });
    return o;
}

// diagonal metric.  Where some √|g_aa|·|h_a| leaves 1e±45 (zero, infinite and NaN
// metrics among them; plain turns false) the node is worked out again with EXACT,
// with divisions: behind the node's other work, so that no branch keeps its loads
// from being in flight together.
template <int N, bool EXACT>
__device__ __forceinline__ Star<N> diag_star(const double (&m)[N], const double (&h)[N], bool& plain)
{
    double s[N];
    if constexpr (EXACT) {
        Star<N> o;
        bool ok = true; // a zero entry makes the whole metric singular
#pragma unroll
        for (int a = 0; a < N; ++a) {
            s[a] = sqrt(fabs(m[a])) * fabs(h[a]);
            ok = ok && m[a] != 0.0;
        }
        static_for<1 << N>([&](auto SRC) {
            constexpr unsigned src = decltype(SRC)::value;
            double num = 1.0, den = 1.0;
#pragma unroll
            for (int a = 0; a < N; ++a) ((src >> a) & 1u ? den : num) *= s[a];
            o.c[src] = ok && den != 0.0 ? num / den : 0.0;
        });
        return o;
    } else {
#pragma unroll
        for (int a = 0; a < N; ++a) {
            s[a] = root(fabs(m[a])) * fabs(h[a]);
            plain = plain && s[a] > 1e-45 && s[a] < 1e45;
        }
        return star_of_edges<N>(s);
    }
}

template <int N, bool DIAG, bool EXACT>
__device__ __forceinline__ Star<N> load_star(const RectGeom<N>& g, const uint32_t (&idx)[N], bool& plain)
{
    double h[N];
#pragma unroll
    for (int a = 0; a < N; ++a) h[a] = g.h[a][idx[a]];
    if constexpr (DIAG) {
        int64_t lin = 0;
#pragma unroll
        for (int a = 0; a < N; ++a) lin += (int64_t)idx[a] * g.node[a];
        double m[N];
#pragma unroll
        for (int a = 0; a < N; ++a) m[a] = g.g[lin * N + a];
        return diag_star<N, EXACT>(m, h, plain);
    } else {
#pragma unroll
        for (int a = 0; a < N; ++a) h[a] = fabs(h[a]);
        return star_of_edges<N>(h);
    }
}

// identity metric on the nodes of one column along x: what y and z give is
// formed once, a plane costs 10 to 17 operations (star_of_edges 20 to 40: Δ of a
// 3-form, 256³ nodes, 73 against 80 µs)
struct IdentColumn {
    double P, iP, zy, yz; // h_y h_z, its reciprocal, h_z / h_y, h_y / h_z

    __device__ __forceinline__ IdentColumn(double hy, double hz)
    {
        hy = fabs(hy);
        hz = fabs(hz);
        P = hy * hz;
        const double y = guess_reciprocal(P);
        iP = quotient(1.0, P, y);
        zy = quotient(hz, hy, hz * y);
        yz = quotient(hy, hz, hy * y);
    }

    __device__ __forceinline__ Star<3> at(double hx) const
    {
        hx = fabs(hx);
        const double rx = guess_reciprocal(hx);
        return {{hx * P, quotient(P, hx, rx), hx * zy, quotient(zy, hx, rx), hx * yz, quotient(yz, hx, rx),
                 quotient(hx, P, iP), quotient(iP, hx, rx)}};
    }
};

// ⋆ from the axes SRC onto their complement: sign · Π_tgt s / Π_src s
template <int N, unsigned SRC>
__device__ __forceinline__ double star_coef(const Star<N>& o)
{
    constexpr int sign = concat_sign(SRC, ((1u << N) - 1u) & ~SRC, N);
    return sign < 0 ? -o.c[SRC] : o.c[SRC];
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

// One node of ⋆, δ and Δ: the components at n into v; false where a metric
// asks for EXACT
template <int N, int K, bool DIAG, bool EXACT>
__device__ __forceinline__ bool hodge_node(const RectGeom<N>& g, const Form<N>& w, const Node<N>& n,
                                           double (&v)[combos<N, N - K>()])
{
    bool plain = true;
    const Star<N> s = load_star<N, DIAG, EXACT>(g, n.i, plain);
    static_for<combos<N, N - K>()>([&](auto C) {
        constexpr int c = decltype(C)::value;
        constexpr unsigned src = ((1u << N) - 1u) & ~kCombos.mask[N][N - K][c];
        v[c] = star_coef<N, src>(s) * w.template at<src>(n);
    });
    return plain;
}

template <int N, int K, bool DIAG, bool EXACT>
__device__ __forceinline__ bool codifferential_node(const RectGeom<N>& g, const Form<N>& w, const Node<N>& n,
                                                    double (&v)[combos<N, K - 1>()])
{
    bool plain = true;
    const Star<N> s = load_star<N, DIAG, EXACT>(g, n.i, plain);
    Star<N> sb[N];
    static_for<N>([&](auto A) {
        constexpr int a = decltype(A)::value;
        sb[a] = load_star<N, DIAG, EXACT>(g, back<N, a>(n).i, plain);
    });
    static_for<combos<N, K - 1>()>([&](auto C) {
        constexpr int c = decltype(C)::value;
        constexpr unsigned I = kCombos.mask[N][K - 1][c];
        v[c] = codiff<N, K, I, false>(w, n, s,
                                      [&](auto A, const Node<N>&) -> const Star<N>& { return sb[decltype(A)::value]; });
    });
    return plain;
}

// Δ = δd + dδ.  Stars of n, n ± e_a and (for dδ, where a component moves along
// one axis and δ steps back along another) n + e_a − e_b.
template <int N, int K, bool DIAG, bool EXACT>
__device__ __forceinline__ bool laplacian_node(const RectGeom<N>& g, const Form<N>& w, const Node<N>& n,
                                               double (&v)[combos<N, K>()])
{
    bool plain = true;
    const Star<N> s = load_star<N, DIAG, EXACT>(g, n.i, plain);
    Star<N> sb[N];
    static_for<N>([&](auto A) {
        constexpr int a = decltype(A)::value;
        sb[a] = load_star<N, DIAG, EXACT>(g, back<N, a>(n).i, plain);
    });
    auto sb_of = [&](auto A, const Node<N>&) -> const Star<N>& { return sb[decltype(A)::value]; };
    static_for<combos<N, K>()>([&](auto C) {
        constexpr int c = decltype(C)::value;
        constexpr unsigned I = kCombos.mask[N][K][c];
        v[c] = 0.0;
        if constexpr (K < N) v[c] += codiff<N, K + 1, I, true>(w, n, s, sb_of);
    });
    if constexpr (K > 0) {
        // (dδω)_I = Σ_a ± [(δω)_{I∖a}(n + e_a) − (δω)_{I∖a}(n)], the
        // difference 0 at the last node of the axis
        static_for<N>([&](auto A) {
            constexpr int a = decltype(A)::value;
            const Node<N> f = next<N, a>(n, g.ext);
            const bool inner = n.i[a] + 1 < g.ext[a];
            const Star<N> sf = load_star<N, DIAG, EXACT>(g, f.i, plain);
            auto sf_back = [&](auto B, const Node<N>& m) {
                constexpr int b = decltype(B)::value;
                if constexpr (b == a)
                    return s; // f − e_a = n (at the last node f's value is dropped)
                else
                    return load_star<N, DIAG, EXACT>(g, m.i, plain);
            };
            static_for<combos<N, K>()>([&](auto C) {
                constexpr int c = decltype(C)::value;
                constexpr unsigned I = kCombos.mask[N][K][c];
                if constexpr ((I >> a) & 1u) {
                    constexpr unsigned J = I & ~(1u << a);
                    const double here = codiff<N, K, J, false>(w, n, s, sb_of);
                    const double ahead = codiff<N, K, J, false>(w, f, sf, sf_back);
                    v[c] += axis_sign<I, a>() * ((inner ? ahead : here) - here);
                }
            });
        });
    }
    return plain;
}

template <RectOp OP, int N, int K, bool DIAG>
__global__ __launch_bounds__(kRectBlock) void k_rect_node(RectGeom<N> g, const double* __restrict__ in,
                                                          RectView<N> vin, double* __restrict__ out, RectView<N> vout,
                                                          uint32_t total)
{
    constexpr int KO = OP == RectOp::Hodge ? N - K : (OP == RectOp::Codifferential ? K - 1 : K);
    const Form<N> w{in, vin};
    for (uint32_t t = blockIdx.x * kRectBlock + threadIdx.x; t < total; t += gridDim.x * kRectBlock) {
        Node<N> n;
        rect_decode<N>(t, vout.ext, n.i);
        const int64_t o = rect_offset<N>(vout, n.i);
        double v[combos<N, KO>()];
        auto node = [&](auto EXACT) {
            constexpr bool exact = decltype(EXACT)::value;
            if constexpr (OP == RectOp::Hodge)
                return hodge_node<N, K, DIAG, exact>(g, w, n, v);
            else if constexpr (OP == RectOp::Codifferential)
                return codifferential_node<N, K, DIAG, exact>(g, w, n, v);
            else
                return laplacian_node<N, K, DIAG, exact>(g, w, n, v);
        };
        if (__builtin_expect(!node(std::false_type{}), 0)) {
            // read again: the registers of the plain form hold nothing for this
#pragma unroll
            for (int a = 0; a < N; ++a) asm volatile("" : "+v"(n.i[a]));
            node(std::true_type{});
        }
        static_for<combos<N, KO>()>([&](auto C) {
            constexpr int c = decltype(C)::value;
            out[o + c * vout.cstr] = v[c];
        });
    }
}

// Δ on 3D grids by a march along x: a workgroup owns 62 (z) × (TY − 2) (y)
// nodes with a one-node halo and walks a chunk of x planes, so a node's star is
// formed once per tile where k_rect_node forms the stars of its 13 nodes.
// Registers hold ω, the stars, ⋆ω and δω of planes p and p + 1 and ⋆dω of
// p − 1; the y and z neighbours of ω, ⋆ω, ⋆dω and δω go through LDS, two
// barriers a plane; plane p + 2 is requested a step before it is used.  Sums
// and their order are those of k_rect_node.  8 rows: two workgroups of a
// 1- or 2-form a compute unit (82–100 registers, 45–53 KB of LDS), three or four
// of a 0- or 3-form, which hide each other's barriers (the bound holds the
// 3-form's at 64 registers, four workgroups).  Diagonal metric, gather → march:
//   2-form  65³ 18 → 12, 107 × 75 × 93 42 → 19, 129 × 120 × 135 107 → 43,
//           256³ 981 → 330 µs
//   0-form  256³ 279 → 168 µs;  3-form  256³ 390 → 165 µs
//   1-form  component-first, 256³ 903 → 303 µs (index-last: dec_fused.hip)
template <int K, int TY>
struct MarchLds {
    double w[combos<3, K>()][TY][64];                       // ω(p): +y, +z neighbours of dω
    double b[K > 0 ? combos<3, K>() : 1][TY][64];           // ⋆ω(p + 1): −y, −z neighbours of δω
    double a[K < 3 ? combos<3, K + 1>() : 1][TY][64];       // ⋆dω(p): −y, −z neighbours of δdω
    double d[2][K > 0 ? combos<3, K - 1>() : 1][TY][64];    // δω(p), δω(p + 1): +y, +z neighbours of dδω
};

template <int K, bool DIAG, int TY>
__global__ __launch_bounds__(64 * TY, K == 3 ? 8 : 1) void
k_rect_lap3_march(RectGeom<3> g, const double* __restrict__ in, RectView<3> vin, double* __restrict__ out,
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
    const double hy = g.h[1][jc], hz = g.h[2][kc];
    const IdentColumn ident(hy, hz);

    // the raw values of plane x (clamped into the grid)
    struct Raw {
        double w[C], m[3], h;
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
    };
    auto star_of = [&](const Raw& o) {
        if constexpr (DIAG) {
            const double h[3] = {o.h, hy, hz};
            bool plain = true;
            const Star<3> s = diag_star<3, false>(o.m, h, plain);
            return __builtin_expect(plain, 1) ? s : diag_star<3, true>(o.m, h, plain);
        } else {
            return ident.at(o.h);
        }
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
    int64_t blocks; // 0: k_rect_node
};

// The march takes a grid where enough of its lanes hold nodes to write, and a
// 0- or 3-form also needs 500 000 nodes: below, the gather of 7 stars is the
// shorter chain (79³, diagonal metric: 0-form 10 against 12 µs, 3-form 14 against
// 12; 107 × 75 × 93: 14 against 14, 20 against 13).  On 256 × 256 × z nodes, of 62
// along z, gather / march in µs (1-form component-first):
//   identity  0-form  z = 29: 17/20   z = 33: 19/20   z = 41: 23/20
//             1-form  z = 17: 33/41   z = 21: 40/41   z = 25: 47/42
//             2-form  z = 17: 34/41   z = 21: 40/41   z = 25: 47/41
//             3-form  z = 25: 18/20   z = 29: 21/20
//   diagonal  0-form  z = 29: 28/34   z = 33: 31/34   z = 41: 38/34
//             1-form  z = 13: 42/53   z = 17: 54/53   z = 21: 66/53
//             2-form  z = 13: 43/52   z = 17: 54/53   z = 21: 68/53
//             3-form  z = 17: 25/31   z = 21: 30/31   z = 25: 35/31
template <int K, bool DIAG>
March march_shape(const RectView<3>& o)
{
    March m{};
    m.ntz = (int)((o.ext[2] + 61) / 62);
    m.nty = (int)((o.ext[1] + kMarchRows - 3) / (kMarchRows - 2));
    const int64_t tiles = (int64_t)m.ntz * m.nty, column = (int64_t)o.ext[1] * o.ext[2];
    constexpr bool ends = K == 0 || K == 3;
    constexpr double used = K == 0 ? 0.4 : (K == 3 ? (DIAG ? 0.26 : 0.31) : (DIAG ? 0.2 : 0.25));
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
        auto gather = [&](auto OP) {
            hipLaunchKernelGGL((k_rect_node<decltype(OP)::value, N, K, diag>), grid, block, 0, stream, rg, in, vi, out,
                               vo, total);
        };
        if (op == RectOp::Hodge) {
            gather(std::integral_constant<RectOp, RectOp::Hodge>{});
        } else if (op == RectOp::Codifferential) {
            if constexpr (K > 0) gather(std::integral_constant<RectOp, RectOp::Codifferential>{});
        } else {
            if constexpr (N == 3) {
                const March m = march_shape<K, diag>(vo);
                if (m.blocks > 0) {
                    hipLaunchKernelGGL((k_rect_lap3_march<K, diag, kMarchRows>), dim3((unsigned)m.blocks),
                                       dim3(64 * kMarchRows), 0, stream, rg, in, vi, out, vo, m.ntz, m.nty, m.chunk);
                    return;
                }
            }
            gather(std::integral_constant<RectOp, RectOp::Laplacian>{});
        }
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
