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
//   Δ of a 2-form, 107 × 75 × 93 nodes     2753 → 64 µs
//   δ of a 2-form, 129 × 120 × 135 nodes   1633 → 54 µs (2.8 TB/s)
//   Δ of a 1-form, 2048 × 1999 nodes       3742 → 83 µs
//   ⋆ of a 1-form, 256³ nodes              1931 → 251 µs (4.8 TB/s, a copy's rate)
//   d of a 1-form, 256³ nodes              1141 → 248 µs
// δ, ⋆ and d are bound by memory; Δ where it holds dδ by the FP64 work of the
// 13 stars it reads per node in 3D (164 registers, three wavefronts a SIMD).
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
        else if (op == RectOp::Laplacian)
            hipLaunchKernelGGL((k_rect_laplacian<N, K, diag>), grid, block, 0, stream, rg, in, vi, out, vo, total);
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
