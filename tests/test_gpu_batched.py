"""GPU checks of the batched persistent Poisson solver: every problem
reaches an FP64-verified 1e-10 relative residual (recomputed here with the
CPU oracle's operator), for every workgroup size the autotuner chooses from."""
import numpy as np
import pytest
import torch

import oracle_lib as orc

pytestmark = pytest.mark.gpu


def problems(seed, count, lo=8, hi=70):
    rng = np.random.default_rng(seed)
    sides = np.round(np.exp(rng.uniform(np.log(lo), np.log(hi), count))).astype(int)
    kap, rhs = [], []
    for n in sides:
        kap.append(np.exp(rng.standard_normal((n, n))))
        b = np.zeros((n, n))
        b[1:-1, 1:-1] = rng.standard_normal((n - 2, n - 2))
        rhs.append(b)
    return sides, kap, rhs


@pytest.mark.parametrize("block", [256, 512, 1024])
def test_batched_solve_reaches_fp64_verified_tolerance(block):
    from similie_amd.batched import BatchedPoisson2D

    sides, kap, rhs = problems(3, 24)
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    solver = BatchedPoisson2D(sides, kappa)
    solver.set_block(block)
    x, results, secs = solver.solve(b)
    xh = x.cpu().numpy()
    for p, n in enumerate(sides):
        assert results[p]["converged"] == 1, (p, n, results[p])
        assert results[p]["true_relative_residual"] <= 1e-10
        o = solver.offset(p)
        xp = xh[o:o + n * n].reshape(n, n)
        ones = np.ones(n)
        r = rhs[p] - orc.poisson2d_apply(ones, ones, kap[p], xp)
        assert np.linalg.norm(r) <= 1.0001e-10 * np.linalg.norm(rhs[p])


def test_autotune_picks_a_candidate_and_solves():
    from similie_amd.batched import BatchedPoisson2D

    sides, kap, rhs = problems(4, 40, 16, 120)
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    solver = BatchedPoisson2D(sides, kappa)
    block, secs = solver.autotune(b, probe_iterations=10)
    assert block in (256, 512, 1024) and all(v > 0 for v in secs.values())
    x, results, _ = solver.solve(b)
    assert all(r["converged"] == 1 and r["true_relative_residual"] <= 1e-10 for r in results)


@pytest.mark.parametrize("wide_side", ["3", "40", "100000"])
def test_wide_path_reaches_fp64_verified_tolerance(wide_side, monkeypatch):
    """Problems at or above the wide side are spread over many workgroups
    (kernel boundaries as the only barriers); the rest stay one workgroup
    each.  Every split — all wide, mixed, none wide — solves every problem."""
    from similie_amd.batched import BatchedPoisson2D

    monkeypatch.setenv("SIL_BATCH_WIDE_SIDE", wide_side)
    sides, kap, rhs = problems(5, 18, 8, 90)
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    solver = BatchedPoisson2D(sides, kappa)
    x, results, _ = solver.solve(b)
    xh = x.cpu().numpy()
    for p, n in enumerate(sides):
        assert results[p]["converged"] == 1, (p, n, results[p])
        assert results[p]["true_relative_residual"] <= 1e-10
        o = solver.offset(p)
        xp = xh[o:o + n * n].reshape(n, n)
        ones = np.ones(n)
        r = rhs[p] - orc.poisson2d_apply(ones, ones, kap[p], xp)
        assert np.linalg.norm(r) <= 1.0001e-10 * np.linalg.norm(rhs[p])
    # a second solve on the same handle reuses the captured graphs
    x2, results2, _ = solver.solve(b)
    assert [r["iterations"] for r in results2] == [r["iterations"] for r in results]


def test_shape_autotune_keeps_every_problem_solved():
    """The shape autotuner re-partitions the batch (wide-path threshold,
    workgroups per wide problem, workgroup size) between timed probes; the
    shape it leaves behind still solves every problem to the verified
    tolerance, and a second solve repeats the first bit for bit."""
    from similie_amd.batched import BatchedPoisson2D

    sides, kap, rhs = problems(6, 30, 8, 260)
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    solver = BatchedPoisson2D(sides, kappa)
    shape = solver.autotune_shape(b, probe_iterations=8)
    assert shape["block"] in (256, 512, 1024) and shape["probe_seconds"] > 0
    assert shape["wide_side"] in (96, 128, 192, 256, 384, int(max(sides)) + 1)
    assert shape["wide_problems"] == sum(int(n) >= shape["wide_side"] for n in sides)
    assert shape["wide_workgroups"] >= 1
    x, results, _ = solver.solve(b)
    xh = x.cpu().numpy()
    for p, n in enumerate(sides):
        assert results[p]["converged"] == 1, (p, n, results[p])
        assert results[p]["true_relative_residual"] <= 1e-10
        o = solver.offset(p)
        xp = xh[o:o + n * n].reshape(n, n)
        ones = np.ones(n)
        r = rhs[p] - orc.poisson2d_apply(ones, ones, kap[p], xp)
        assert np.linalg.norm(r) <= 1.0001e-10 * np.linalg.norm(rhs[p])
    x2, results2, _ = solver.solve(b)
    assert torch.equal(x, x2) and [r["iterations"] for r in results2] == [r["iterations"] for r in results]


@pytest.mark.parametrize("limit", [1, 7, 8, 9, 17])
@pytest.mark.parametrize("replace", [0, 3])
def test_wide_and_persistent_paths_take_the_same_iterations(limit, replace, monkeypatch):
    """A limit on the iterations inside, at the end of and just after a chunk
    of steps, with and without replacement steps of their own in between:
    the wide path counts and iterates as the persistent kernel does (FP32
    recurrences of at most 17 iterations, sums in another order: 1e-4)."""
    from similie_amd.batched import BatchedPoisson2D
    from similie_amd.solvers import StrongFormulationSolverSettings

    sides, kap, rhs = problems(7, 9, 3, 70)
    sides[0], sides[1] = 3, 33  # one unknown; 1089 nodes: a second workgroup of 65
    rng = np.random.default_rng(3)
    kap = [np.exp(rng.standard_normal((n, n))) for n in sides]
    rhs = [np.pad(rng.standard_normal((n - 2, n - 2)), 1) for n in sides]
    rhs[4][:] = 0.0  # solved before the first step
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    st = StrongFormulationSolverSettings(relative_tolerance=1e-10, precision="mixed", preconditioner="jacobi",
                                         max_iterations=limit, replace_interval=replace)
    got = []
    for side in ("3", "100000"):
        monkeypatch.setenv("SIL_BATCH_WIDE_SIDE", side)
        x, results, _ = BatchedPoisson2D(sides, kappa).solve(b, settings=st)
        got.append((x.cpu().numpy(), results))
    (xw, rw), (xp, rp) = got
    for p, n in enumerate(sides):
        assert rw[p]["iterations"] == rp[p]["iterations"] <= limit, p
        assert rw[p]["converged"] == rp[p]["converged"], p
        assert abs(rw[p]["true_relative_residual"] - rp[p]["true_relative_residual"]) <= \
            1e-4 * rp[p]["true_relative_residual"] + 1e-10
    assert np.linalg.norm(xw - xp) <= 1e-4 * np.linalg.norm(xp)


def test_second_direction_buffer_is_the_wide_problems_alone():
    """6000 problems of the persistent kernel and one wide one: a handle holds
    six FP32 and four FP64 values a node, and the wide path's own arrays for
    the wide problem only (an FP32 value a node of all would be 194 MB; 64 MB
    are left for the rounding of some twenty allocations)"""
    import gc

    from similie_amd.batched import BatchedPoisson2D

    sides = [90] * 6000 + [96]
    nodes = sum(n * n for n in sides)
    kappa = torch.ones(nodes, dtype=torch.float64, device="cuda")
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    solver = BatchedPoisson2D(sides, kappa)
    torch.cuda.synchronize()
    held = before - torch.cuda.mem_get_info()[0]
    assert 56 * nodes <= held <= 56 * nodes + (64 << 20), held / nodes
    del solver


def test_the_workgroup_size_is_the_one_in_use():
    """few small problems: 16 wavefronts each; many: eight; set or autotuned:
    that"""
    from similie_amd import _lib as L
    from similie_amd.batched import BatchedPoisson2D

    compute_units = torch.cuda.get_device_properties(0).multi_processor_count
    for count, block in ((4, 1024), (2 * compute_units, 1024), (2 * compute_units + 1, 512)):
        solver = BatchedPoisson2D([5] * count, torch.ones(25 * count, dtype=torch.float64, device="cuda"))
        assert solver.block == block == L.lib().sil_batched_poisson2d_block(solver.handle)
        solver.set_block(256)
        assert solver.block == 256 == L.lib().sil_batched_poisson2d_block(solver.handle)
        chosen, _ = solver.autotune(torch.ones(25 * count, dtype=torch.float64, device="cuda"), probe_iterations=2)
        assert solver.block == chosen == L.lib().sil_batched_poisson2d_block(solver.handle)


@pytest.mark.parametrize("limit,replace", [(24, 0), (41, 7)])
def test_wide_problems_that_finish_at_different_times(limit, replace, monkeypatch):
    """Wide problems whose right-hand sides hold 1, 6, 14 or 22 eigenvectors
    finish after about as many iterations, and the map of workgroups is
    rebuilt while a problem of side 517 still runs, whose 256 workgroups take
    a second, partial pass (267 289 nodes).  The persistent kernel does the
    same arithmetic with its FP64 sums in another order: the solved problems
    stop within an iteration of it on a verified residual, the others hold
    its iterates (FP32 recurrences, 1e-4 as in the test above)."""
    from similie_amd.batched import BatchedPoisson2D
    from similie_amd.solvers import StrongFormulationSolverSettings

    rng = np.random.default_rng(4)
    modes = {96: 1, 160: 1, 161: 6, 200: 6, 130: 14, 201: 14, 162: 22, 97: 22}
    sides, kap = [517], [np.exp(0.5 * rng.standard_normal((517, 517)))]
    rhs = [np.pad(rng.standard_normal((515, 515)), 1)]
    for n, count in modes.items():  # of middle wavelengths: eigenvalues that FP32 products resolve
        t = np.pi * np.arange(n) / (n - 1)
        b = np.zeros((n, n))
        for m in range(1, count + 1):
            b += rng.uniform(0.5, 1.5) * np.outer(np.sin((n // 8 + 2 * m) * t), np.sin((n // 6 + m) * t))
        b[0], b[-1], b[:, 0], b[:, -1] = 0.0, 0.0, 0.0, 0.0
        sides.append(n), kap.append(np.ones((n, n))), rhs.append(b)
    kappa = torch.from_numpy(np.concatenate([k.ravel() for k in kap])).cuda()
    b = torch.from_numpy(np.concatenate([r.ravel() for r in rhs])).cuda()
    st = StrongFormulationSolverSettings(relative_tolerance=1e-5, precision="mixed", preconditioner="identity",
                                         max_iterations=limit, replace_interval=replace)
    got = []
    for side in ("96", "100000"):
        monkeypatch.setenv("SIL_BATCH_WIDE_SIDE", side)
        x, results, _ = BatchedPoisson2D(sides, kappa).solve(b, settings=st)
        got.append((x.cpu().numpy(), results))
    (xw, rw), (xp, rp) = got
    print([r["iterations"] for r in rw], [r["iterations"] for r in rp], flush=True)
    assert len({r["iterations"] for r in rw if r["converged"]}) >= 3 and not rw[0]["converged"]
    at = 0
    for p, n in enumerate(sides):
        xi, xr = xw[at:at + n * n], xp[at:at + n * n]
        at += n * n
        assert rw[p]["converged"] == rp[p]["converged"], p
        if rw[p]["converged"]:
            assert abs(rw[p]["iterations"] - rp[p]["iterations"]) <= 1, p
            r = rhs[p] - orc.poisson2d_apply(np.ones(n), np.ones(n), kap[p], xi.reshape(n, n))
            assert np.linalg.norm(r) <= 1.0001e-5 * np.linalg.norm(rhs[p]), p
        else:
            assert rw[p]["iterations"] == rp[p]["iterations"] == limit, p
        assert np.linalg.norm(xi - xr) <= 1e-4 * np.linalg.norm(xr), p
