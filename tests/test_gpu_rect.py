"""The compile-time kernels of d, ⋆, δ and Δ on regular rectilinear grids
(dec_rect.hip) against the CPU oracle, at the sizes, strides and metrics where
their rule can go wrong: one- and two-node axes (the general kernels), grids
that leave a partial workgroup, component-first and permuted storage, output
domains shorter than the grid, singular and extreme metric entries."""
from math import comb

import numpy as np
import pytest
import torch

import oracle_lib as orc

pytestmark = pytest.mark.gpu

# every coefficient is a product of N factors each within about 4 ulp, every
# result a sum of at most 30 products: 30 · (3·4 + 2) ulp ≈ 1e-13
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
