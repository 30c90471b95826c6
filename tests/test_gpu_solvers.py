"""GPU parity of the magnetostatics / Poisson operators and of the CG solve
(FP64 and mixed precision) against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import similie_amd.solvers as S

    return S


def cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def ms_problem(shape, rng, stretch=True):
    coords = []
    for n in shape:
        h = rng.uniform(0.5, 1.5, n - 1) if stretch else np.ones(n - 1)
        coords.append(np.concatenate([[0.0], np.cumsum(h)]) / (n - 1))
    nx, ny, nz = shape
    cells = (nx - 1) * (ny - 1) * (nz - 1)
    cell_mu = np.where(rng.random(cells) < 0.3, 1000.0, 1.0) * 4e-7 * np.pi
    cell_j = rng.standard_normal((cells, 3))
    return coords, cell_mu, cell_j


@pytest.mark.parametrize("shape", [(6, 5, 7), (17, 9, 12), (70, 15, 41)])
def test_magnetostatics_assembly_and_apply(S, shape):
    rng = np.random.default_rng(sum(shape))
    coords, cell_mu, cell_j = ms_problem(shape, rng)
    mu0 = 4e-7 * np.pi
    mu = S.MagnetostaticsOperator3D.nodal_mu(shape, cuda(cell_mu), mu0)
    mu_ref = orc.ms_nodal_mu(shape, cell_mu, mu0)
    np.testing.assert_allclose(mu.cpu().numpy(), mu_ref, rtol=1e-15)
    op = S.MagnetostaticsOperator3D(*coords, mu, gauge_penalty=1e7)
    b = op.rhs(cuda(cell_j))
    b_ref = orc.ms_rhs(coords, cell_j)
    assert np.max(np.abs(b.cpu().numpy() - b_ref)) <= 1e-14 * np.max(np.abs(b_ref))
    x = rng.standard_normal(op.size())
    y = op.apply(cuda(x)).cpu().numpy()
    y_ref = orc.ms_apply(coords, mu_ref, 1e7, x)
    assert np.max(np.abs(y - y_ref)) <= 1e-12 * np.max(np.abs(y_ref))
    y32 = op.apply_f32(cuda(x).float()).double().cpu().numpy()
    assert np.max(np.abs(y32 - y_ref)) <= 1e-5 * np.max(np.abs(y_ref))
    d = op.diagonal().cpu().numpy()
    d_ref = orc.ms_diagonal(coords, mu_ref, 1e7)
    assert np.max(np.abs(d - d_ref)) <= 1e-12 * np.max(np.abs(d_ref))


def poisson_problem(nx, ny, rng, varcoef=True):
    xc = np.linspace(0.0, 1.0, nx)
    yc = np.linspace(0.0, 1.0, ny)
    kappa = np.exp(rng.standard_normal((nx, ny))) if varcoef else None
    b = np.zeros((nx, ny))
    b[1:-1, 1:-1] = rng.standard_normal((nx - 2, ny - 2))
    return xc, yc, kappa, b


def test_poisson_apply_and_diagonal(S):
    rng = np.random.default_rng(4)
    xc, yc, kappa, b = poisson_problem(33, 29, rng)
    op = S.Poisson2D(xc, yc, cuda(kappa))
    u = rng.standard_normal((33, 29))
    got = op.apply(cuda(u).reshape(-1)).cpu().numpy().reshape(33, 29)
    hx = np.concatenate([np.diff(xc), [xc[-1] - xc[-2]]])
    hy = np.concatenate([np.diff(yc), [yc[-1] - yc[-2]]])
    ref = orc.poisson2d_apply(hx, hy, kappa, u * np.pad(np.ones((31, 27)), 1))
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("precond", ["identity", "jacobi"])
def test_cg_fp64_poisson_matches_oracle(S, precond):
    rng = np.random.default_rng(5)
    xc, yc, kappa, b = poisson_problem(65, 65, rng)
    op = S.Poisson2D(xc, yc, cuda(kappa))
    st = S.StrongFormulationSolverSettings(max_iterations=5000, relative_tolerance=1e-10, preconditioner=precond)
    x, dg = S.minimize_strong_formulation_residual(op, cuda(b).reshape(-1), settings=st)
    assert dg["converged"] == 1 and dg["true_relative_residual"] <= 1.5e-10
    if precond == "identity":
        hx = np.full(65, 1 / 64)
        xr, it, rn, bn = orc.poisson2d_cg(hx, hx, kappa, b, 1e-10, 5000)
        # the count at a fixed tolerance moves with the rounding order of the
        # dot products (the GPU's block partials and the oracle's fixed
        # 4096-blocks are both deterministic, and different): ±1 %
        assert abs(it - dg["iterations"]) <= max(2, it // 100), (it, dg["iterations"])
        err = np.max(np.abs(x.cpu().numpy().reshape(65, 65) - xr)) / np.max(np.abs(xr))
        assert err <= 1e-8


@pytest.mark.parametrize("precond", ["identity", "jacobi"])
def test_cg_fp64_magnetostatics(S, precond):
    rng = np.random.default_rng(6)
    shape = (14, 12, 16)
    coords, cell_mu, cell_j = ms_problem(shape, rng, stretch=False)
    mu0 = 4e-7 * np.pi
    mu = S.MagnetostaticsOperator3D.nodal_mu(shape, cuda(cell_mu), mu0)
    op = S.MagnetostaticsOperator3D(*coords, mu, gauge_penalty=1e7)
    b = op.rhs(cuda(cell_j))
    st = S.StrongFormulationSolverSettings(max_iterations=20000, relative_tolerance=1e-10, preconditioner=precond)
    x, dg = S.minimize_strong_formulation_residual(op, b, settings=st)
    assert dg["converged"] == 1 and dg["true_relative_residual"] <= 1.5e-10
    r = b.cpu().numpy() - orc.ms_apply(coords, mu.cpu().numpy(), 1e7, x.cpu().numpy())
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b.cpu().numpy())
    x2, dg2 = S.minimize_strong_formulation_residual(op, b, settings=st)
    assert torch.equal(x, x2) and dg2["iterations"] == dg["iterations"]  # reproducible


@pytest.mark.parametrize("precond", ["identity", "jacobi"])
def test_cg_mixed_precision_reaches_fp64_verified_tolerance(S, precond):
    rng = np.random.default_rng(7)
    shape = (14, 12, 16)
    coords, cell_mu, cell_j = ms_problem(shape, rng, stretch=False)
    mu = S.MagnetostaticsOperator3D.nodal_mu(shape, cuda(cell_mu), 4e-7 * np.pi)
    op = S.MagnetostaticsOperator3D(*coords, mu, gauge_penalty=1e7)
    b = op.rhs(cuda(cell_j))
    st = S.StrongFormulationSolverSettings(max_iterations=20000, relative_tolerance=1e-10, preconditioner=precond,
                                           precision="mixed")
    x, dg = S.minimize_strong_formulation_residual(op, b, settings=st)
    assert dg["converged"] == 1 and dg["true_relative_residual"] <= 1e-10
    r = b.cpu().numpy() - orc.ms_apply(coords, mu.cpu().numpy(), 1e7, x.cpu().numpy())
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b.cpu().numpy())
    rng2 = np.random.default_rng(8)
    xc, yc, kappa, bp = poisson_problem(97, 81, rng2)
    opp = S.Poisson2D(xc, yc, cuda(kappa))
    xp, dgp = S.minimize_strong_formulation_residual(opp, cuda(bp).reshape(-1), settings=st)
    assert dgp["converged"] == 1 and dgp["true_relative_residual"] <= 1e-10


def test_cg_zero_rhs_and_iteration_cap(S):
    rng = np.random.default_rng(9)
    xc, yc, kappa, b = poisson_problem(33, 33, rng)
    op = S.Poisson2D(xc, yc, cuda(kappa))
    zero = torch.zeros(33 * 33, dtype=torch.float64, device="cuda")
    x, dg = S.minimize_strong_formulation_residual(op, zero)
    assert dg["iterations"] == 0 and dg["converged"] == 1 and torch.count_nonzero(x) == 0
    st = S.StrongFormulationSolverSettings(max_iterations=5, relative_tolerance=1e-14, preconditioner="identity")
    x, dg = S.minimize_strong_formulation_residual(op, cuda(b).reshape(-1), settings=st)
    assert dg["iterations"] == 5 and dg["converged"] == 0


def _numpy_cg(apply, diag, b, iterations):
    """Jacobi CG, a fixed number of iterations"""
    x, r = np.zeros_like(b), b.copy()
    z = r / diag
    p, rz = z.copy(), float(np.dot(r, z))
    for _ in range(iterations):
        q = apply(p)
        if rz == 0.0:  # solved exactly: the iterates stay
            break
        alpha = rz / float(np.dot(p, q))
        x += alpha * p
        r -= alpha * q
        z = r / diag
        new = float(np.dot(r, z))
        p, rz = z + (new / rz) * p, new
    return x


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(3, 3), (5, 4), (33, 17), (61, 64, 1), (4, 3, 5), (9, 16, 7), (65, 9, 30)])
def test_cg_stops_at_the_iteration_limit(shape, precision):
    """The iterates after 1, 2, 3, 31, 32, 33 and 35 iterations (the first and
    last of a chunk, the first of the next) against plain CG: every kernel of
    an iteration finishes the one before, so a limit inside a chunk, at its
    end and just after it takes different paths.  Rows that are no multiple
    of the vector width, fewer rows than one workgroup's, one direction
    kernel (3D) and none (2D).  Stretched axes of a small 3D grid keep 35
    iterations below convergence."""
    from similie_amd import solvers as S

    rng = np.random.default_rng(sum(shape))
    if len(shape) == 2:
        hx = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, n - 1)])) for n in shape]
        kappa = np.exp(rng.standard_normal(shape))
        op = S.Poisson2D(*hx, kappa=torch.from_numpy(kappa.reshape(-1)).cuda())
    else:
        shape = tuple(max(s, 3) for s in shape)
        axes = [np.cumsum(np.concatenate([[0.0], rng.uniform(0.5, 1.5, n - 1)])) for n in shape]
        mu = np.exp(rng.standard_normal(int(np.prod(shape))))
        op = S.MagnetostaticsOperator3D(*axes, torch.from_numpy(mu).cuda(), gauge_penalty=0.5)
    n = op.size()
    dense = torch.stack([op.apply(e) for e in torch.eye(n, dtype=torch.float64, device="cuda")]).cpu().numpy().T \
        if n <= 600 else None
    diag = op.diagonal().cpu().numpy()

    def apply(v):
        return dense @ v if dense is not None else op.apply(torch.from_numpy(v).cuda()).cpu().numpy()

    b = rng.standard_normal(n)
    if len(shape) == 2:
        b = b.reshape(shape)
        b[0, :] = b[-1, :] = 0.0
        b[:, 0] = b[:, -1] = 0.0
        b = b.reshape(-1)
    bt = torch.from_numpy(b).cuda()
    # k steps of a recurrence rounded to u amplify by at most the operator's
    # condition (below 1e3 here): 35 · 1e3 · u, 4e-12 in FP64 and 2e-3 in FP32;
    # a reduction in another order counts as one more rounding
    for limit in (1, 2, 3, 31, 32, 33, 35):
        x, dg = S.minimize_strong_formulation_residual(
            op, bt, settings=S.StrongFormulationSolverSettings(max_iterations=limit, relative_tolerance=1e-9,
                                                               precision=precision, check_interval=32))
        assert dg["iterations"] <= limit
        if not dg["converged"]:
            assert dg["iterations"] == limit
        r = b - apply(x.cpu().numpy())
        rel_true = np.linalg.norm(r) / max(np.linalg.norm(b), 1e-300)
        assert abs(rel_true - dg["true_relative_residual"]) <= 1e-9 + 1e-6 * rel_true
        if dg["converged"]:
            assert rel_true <= 1e-9 * (1 + 1e-3)
        else:
            ref = _numpy_cg(apply, diag, b, limit)
            tol = 1e-10 if precision == "fp64" else 2e-3
            assert np.linalg.norm(x.cpu().numpy() - ref) <= tol * np.linalg.norm(ref), limit


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_cg_with_more_partial_sums_than_a_workgroup_adds(precision):
    """From 2049 workgroups of a product on (524 288 nodes of a 2D Poisson
    grid) α comes from a kernel of its own: the iterates after 1, 2 and 5
    iterations against plain CG (5 steps of a recurrence that the operator's
    condition of these few steps amplifies by less than 1e3: 5e3 · u)."""
    from similie_amd import solvers as S

    rng = np.random.default_rng(21)
    shape = (1027, 515)
    assert (np.prod(shape) + 255) // 256 > 2048
    kappa = torch.from_numpy(np.exp(rng.standard_normal(shape)).reshape(-1)).cuda()
    op = S.Poisson2D(np.linspace(0.0, 2.0, shape[0]), np.linspace(0.0, 1.0, shape[1]), kappa=kappa)
    b = np.zeros(shape)
    b[1:-1, 1:-1] = rng.standard_normal((shape[0] - 2, shape[1] - 2))
    b = b.reshape(-1)
    diag = op.diagonal().cpu().numpy()
    for limit in (1, 2, 5):
        x, dg = S.minimize_strong_formulation_residual(
            op, torch.from_numpy(b).cuda(), settings=S.StrongFormulationSolverSettings(
                max_iterations=limit, relative_tolerance=1e-9, precision=precision))
        assert dg["iterations"] == limit and dg["converged"] == 0
        ref = _numpy_cg(lambda v: op.apply(torch.from_numpy(v).cuda()).cpu().numpy(), diag, b, limit)
        tol = 1e-12 if precision == "fp64" else 3e-4
        assert np.linalg.norm(x.cpu().numpy() - ref) <= tol * np.linalg.norm(ref), limit
