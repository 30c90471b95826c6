"""The compile-time kernels of d, ⋆, δ and Δ on regular rectilinear grids
(dec_rect.hip) against the CPU oracle, at the sizes, strides and metrics where
their rule can go wrong: one- and two-node axes (the general kernels), grids
that leave a partial workgroup, component-first and permuted storage, output
domains shorter than the grid, singular and extreme metric entries."""
from itertools import combinations
from math import comb

import numpy as np
import pytest
import torch

import oracle_lib as orc

pytestmark = pytest.mark.gpu

# every coefficient is a quotient of products of N factors, within about 4 ulp
# for each, every result a sum of at most 30 products: 30 · (3·4 + 2) ulp ≈ 1e-13
TOL = 1e-13


def cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def stored(shape_last, order):
    """an empty CUDA tensor of the index-last shape, its axes stored in `order`"""
    t = torch.empty([shape_last[o] for o in order], dtype=torch.float64, device="cuda")
    return t.permute([order.index(a) for a in range(len(order))])


def orders(n):
    last = list(range(n + 1))
    return [last, [n] + list(range(n)), last[:n][::-1] + [n]]


def metric_of(rng, extents, n, kind):
    if kind == "identity":
        return None
    m = rng.uniform(0.5, 2.0, size=tuple(extents) + (n,))
    if kind == "singular":
        m.reshape(-1, n)[::3, rng.integers(0, n)] = 0.0
    if kind == "extreme":
        m.reshape(-1, n)[1::4] *= 1e90
        m.reshape(-1, n)[2::4] *= 1e-90
    return m


def close(got, ref, per_value=False):
    got = got.cpu().numpy()
    if per_value:
        den = np.where(ref == 0.0, 1.0, np.abs(ref))
    else:
        den = max(np.max(np.abs(ref)), 1e-300)
    return np.max(np.abs(got - ref) / den) <= TOL


@pytest.mark.parametrize("kind", ["identity", "diagonal", "singular"])
@pytest.mark.parametrize("extents", [[2], [300], [2, 3], [1, 5], [17, 33], [2, 2, 2], [3, 1, 4], [5, 7, 9], [4, 11, 23]])
def test_operators_match_oracle(extents, kind):
    import similie_amd.exterior as E

    n = len(extents)
    rng = np.random.default_rng(sum(extents) + 100 * n)
    axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, e - 1)])) for e in extents]
    m = metric_of(rng, extents, n, kind)
    mk = orc.METRIC_IDENTITY if m is None else orc.METRIC_DIAGONAL
    og = orc.Geometry(extents, axes=axes, metric_kind=mk, metric=None if m is None else m.reshape(-1, n))
    gg = E.Grid(extents, axis_coords=axes, metric=None if m is None else cuda(m), metric_kind=mk)
    for k in range(n + 1):
        w = rng.standard_normal(tuple(extents) + (comb(n, k),))
        for oext in (extents, [max(e - 1, 1) for e in extents]):
            for order in orders(n):
                t = stored(w.shape, order)
                t.copy_(cuda(w))
                dims = dict(grid_dims=list(range(n)), comp_dim=n)

                def out_of(kout, e=oext):
                    o = stored(tuple(e) + (comb(n, kout),), order)
                    o.fill_(float("nan"))
                    return o

                o = out_of(k)
                E.laplacian(gg, k, o, t, comp_dim=n)
                assert close(o, orc.laplacian(og, k, w, oext)), ("laplacian", k, oext, order)
                if k > 0:
                    o = out_of(k - 1)
                    E.codifferential(gg, k, o, t, comp_dim=n)
                    assert close(o, orc.codifferential(og, k, w, oext)), ("codifferential", k, oext, order)
                if k < n:
                    o = out_of(k + 1)
                    E.coboundary(o, t, k, **dims)
                    assert close(o, orc.coboundary(n, k, extents, w, oext)), ("coboundary", k, oext, order)
                o = out_of(n - k, extents)
                E.hodge_star(gg, k, o, t, comp_dim=n)
                assert close(o, orc.hodge_star(og, k, w), per_value=True), ("hodge_star", k, order)


@pytest.mark.parametrize("n", [1, 2, 3])
def test_extreme_metric_entries_keep_their_range(n):
    """metric entries of 1e±90: coefficients stay quotients of edge measures,
    as the reference's volume ratios.  (The oracle forms the determinant of
    the Gram matrix, the square of a volume: 1e270 for three such edges, so
    entries much further out overflow there and not here.)"""
    import similie_amd.exterior as E

    extents = [9, 6, 5][:n]
    rng = np.random.default_rng(5)
    axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, e - 1)])) for e in extents]
    m = metric_of(rng, extents, n, "extreme")
    og = orc.Geometry(extents, axes=axes, metric_kind=orc.METRIC_DIAGONAL, metric=m.reshape(-1, n))
    gg = E.Grid(extents, axis_coords=axes, metric=cuda(m), metric_kind=orc.METRIC_DIAGONAL)
    for k in range(n + 1):
        w = rng.standard_normal(tuple(extents) + (comb(n, k),))
        o = torch.empty(tuple(extents) + (comb(n, n - k),), dtype=torch.float64, device="cuda")
        E.hodge_star(gg, k, o, cuda(w))
        ref = orc.hodge_star(og, k, w)
        assert np.all(np.isfinite(ref))
        assert close(o, ref, per_value=True)


def test_degenerate_spacings_take_the_general_kernels():
    """an edge below the reference's 1e-14 rule (its 2-form coefficients are
    zero): the grid is not regular, results follow the oracle"""
    import similie_amd.exterior as E

    axes = [np.array([0.0, 1e-9, 1.0, 2.0]), np.array([0.0, 1e-6, 1.0])]
    extents = [4, 3]
    og = orc.Geometry(extents, axes=axes)
    gg = E.Grid(extents, axis_coords=axes)
    rng = np.random.default_rng(9)
    for k in range(3):
        w = rng.standard_normal(tuple(extents) + (comb(2, k),))
        o = torch.empty(w.shape, dtype=torch.float64, device="cuda")
        E.laplacian(gg, k, o, cuda(w))
        assert close(o, orc.laplacian(og, k, w, extents)), k


MARCH = [
    ([2, 6, 62], (1, 2)),       # one full tile, one chunk
    ([9, 7, 63], (1, 2)),       # one node past the tile along y and z
    ([23, 13, 125], (1, 2)),    # chunks with a remainder
    ([131, 63, 64], (0, 3)),    # 0- and 3-forms march from 500 000 nodes on
]


@pytest.mark.parametrize("kind", ["identity", "diagonal", "singular"])
@pytest.mark.parametrize("extents,degrees", MARCH)
def test_marching_laplacian_matches_oracle(extents, degrees, kind):
    """Δ on 3D grids wide enough for the march (k_rect_lap3_march, and for
    index-last 1-forms the fused march at the chunk its size selects)."""
    import similie_amd.exterior as E

    rng = np.random.default_rng(sum(extents))
    axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, e - 1)])) for e in extents]
    m = metric_of(rng, extents, 3, kind)
    mk = orc.METRIC_IDENTITY if m is None else orc.METRIC_DIAGONAL
    og = orc.Geometry(extents, axes=axes, metric_kind=mk, metric=None if m is None else m.reshape(-1, 3))
    gg = E.Grid(extents, axis_coords=axes, metric=None if m is None else cuda(m), metric_kind=mk)
    for k in degrees:
        w = rng.standard_normal(tuple(extents) + (comb(3, k),))
        for oext in (extents, [e - 1 for e in extents]):
            ref = orc.laplacian(og, k, w, oext)
            for order in orders(3):
                t = stored(w.shape, order)
                t.copy_(cuda(w))
                o = stored(tuple(oext) + (comb(3, k),), order)
                o.fill_(float("nan"))
                E.laplacian(gg, k, o, t, comp_dim=3)
                assert close(o, ref), (k, oext, order)


def test_default_stream_is_the_current_one():
    """calls without a stream go to torch's current stream, inside and outside
    a stream context and under capture"""
    import similie_amd._lib as L

    def same():
        return (L.stream_handle().value or 0) == torch.cuda.current_stream().cuda_stream

    assert same()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert same() and L.stream_handle().value == side.cuda_stream
    graph = torch.cuda.CUDAGraph()
    t = torch.zeros(4, device="cuda")
    with torch.cuda.graph(graph):
        t.add_(1.0)
        assert same()
    assert L.stream_handle(side).value == side.cuda_stream


def edge_lengths(axes):
    h = [np.append(np.diff(a), a[-1] - a[-2]) for a in axes]
    return np.stack(np.meshgrid(*[np.abs(x) for x in h], indexing="ij"), axis=-1)


def star_quotients(h, m, src, real):
    """Π_tgt s / Π_src s at every node, s_a = √|m_a| h_a, in the arithmetic `real`"""
    s = h.astype(real) if m is None else np.sqrt(np.abs(m).astype(real)) * h.astype(real)
    num, den = np.ones(h.shape[:-1], dtype=real), np.ones(h.shape[:-1], dtype=real)
    for a in range(h.shape[-1]):
        if a in src:
            den = den * s[..., a]
        else:
            num = num * s[..., a]
    return num / den


def device_star(axes, m, k):
    """|⋆| of a k-form of ones: {source axes: coefficient per node}"""
    import similie_amd.exterior as E

    n, extents = len(axes), tuple(len(a) for a in axes)
    gg = E.Grid(extents, axis_coords=axes, metric=None if m is None else cuda(m),
                metric_kind=orc.METRIC_IDENTITY if m is None else orc.METRIC_DIAGONAL)
    w = torch.ones(extents + (comb(n, k),), dtype=torch.float64, device="cuda")
    o = torch.empty(extents + (comb(n, n - k),), dtype=torch.float64, device="cuda")
    E.hodge_star(gg, k, o, w)
    o = np.abs(o.cpu().numpy())
    return {tuple(a for a in range(n) if a not in tgt): o[..., q]
            for q, tgt in enumerate(combinations(range(n), n - k))}


@pytest.mark.parametrize("kind", ["identity", "diagonal"])
@pytest.mark.parametrize("extents", [[60000], [300, 200], [40, 40, 40]])
def test_star_rounds_no_more_than_quotients_of_products(extents, kind):
    """The rms rounding of every coefficient against 64-bit mantissas, and that
    of quotients of FP64 products, as the general kernels form them.  Over
    64 000 nodes the two rms figures are known to about 0.5 %: 2 % apart is a
    difference in the arithmetic."""
    n = len(extents)
    rng = np.random.default_rng(n)
    axes = [np.cumsum(np.concatenate([[0.0], np.exp(rng.uniform(-4.0, 2.0, e - 1))])) for e in extents]
    m = None if kind == "identity" else np.exp(rng.uniform(-8.0, 8.0, tuple(extents) + (n,)))
    h = edge_lengths(axes)
    for k in range(n + 1):
        got, plain, sq = device_star(axes, m, k), 0.0, 0.0
        for src, c in got.items():
            exact = star_quotients(h, m, src, np.longdouble)
            sq += float(np.mean(((c - exact) / exact) ** 2))
            plain += float(np.mean(((star_quotients(h, m, src, np.float64) - exact) / exact) ** 2))
        print(f"star {extents} {kind} k={k}: rms {np.sqrt(sq / len(got)):.3e}, "
              f"quotients {np.sqrt(plain / len(got)):.3e}", flush=True)
        assert sq <= 1.02 ** 2 * plain, k


@pytest.mark.parametrize("n", [1, 2, 3])
def test_metric_entries_without_a_finite_measure(n):
    """zero, infinite, NaN, subnormal and huge entries: what the quotients of
    products give (zero where the metric is singular or the source measure
    vanishes)"""
    rng = np.random.default_rng(n)
    axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, e - 1)])) for e in [40, 9, 7][:n]]
    extents = tuple(len(a) for a in axes)
    m = rng.choice([1.0, 2.5, -3.0, 0.0, np.inf, np.nan, 5e-324, 1e-200, 1e200, 1.7e308], extents + (n,))
    h = edge_lengths(axes)
    with np.errstate(all="ignore"):
        for k in range(n + 1):
            for src, c in device_star(axes, m, k).items():
                want = np.abs(star_quotients(h, m, src, np.float64))
                s = np.sqrt(np.abs(m)) * h
                measure = np.prod([s[..., a] for a in src], axis=0) if src else np.ones(extents)
                want = np.where(np.any(m == 0.0, axis=-1) | (measure == 0.0), 0.0, want)
                np.testing.assert_allclose(c, want, rtol=1e-15 * 8, atol=0.0, err_msg=str(src))


@pytest.mark.parametrize("kind", ["identity", "diagonal"])
@pytest.mark.parametrize("extents,oext,degrees", [([23, 13, 125], [10, 12, 100], (1, 2)),
                                                  ([23, 13, 125], [1, 13, 124], (1, 2)),
                                                  ([9, 70, 66], [7, 61, 62], (1, 2)),
                                                  ([131, 69, 70], [128, 64, 62], (0, 3))])
def test_march_on_output_domains_well_inside_the_grid(extents, oext, degrees, kind):
    """output domains several nodes shorter than the grid along each axis: the
    last tiles and chunks read nodes that none of them writes"""
    import similie_amd.exterior as E

    rng = np.random.default_rng(sum(extents))
    axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, e - 1)])) for e in extents]
    m = metric_of(rng, extents, 3, kind)
    mk = orc.METRIC_IDENTITY if m is None else orc.METRIC_DIAGONAL
    og = orc.Geometry(extents, axes=axes, metric_kind=mk, metric=None if m is None else m.reshape(-1, 3))
    gg = E.Grid(extents, axis_coords=axes, metric=None if m is None else cuda(m), metric_kind=mk)
    for k in degrees:
        w = rng.standard_normal(tuple(extents) + (comb(3, k),))
        ref = orc.laplacian(og, k, w, oext)
        for order in orders(3):
            t = stored(w.shape, order)
            t.copy_(cuda(w))
            o = stored(tuple(oext) + (comb(3, k),), order)
            o.fill_(float("nan"))
            E.laplacian(gg, k, o, t, comp_dim=3)
            assert close(o, ref), (k, order)
