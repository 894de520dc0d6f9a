"""Batched solves whose products read the symmetric slice storage, where a slice of 64 rows holds rows of two
instances and zero padding that points from one into the other."""
import numpy as np
import pytest
import torch

from nonlocal_amd import _abi as A
from nonlocal_amd import api, batch, configs
from tests.helpers import direct_solution, oracle_assembly, rel_l2

pytestmark = pytest.mark.gpu

SIDES = [140, 97, 113, 89]                 # 792 slices of 64 rows: a batch reads them from 600 at the latest
BAD = 1
TOL = 1e-12
BOUND = 4 * 140 ** 2 * TOL                 # the error of a solution: the condition number times its residual


def _instances(lam=1.0):
    """Four uneven instances, no size a multiple of 64; the second one's conductivity is given."""
    return [configs.thermal_q4(n, 0.3 + 0.1 * k, 2.5 / n, lam if k == BAD else 1.0 + 0.2 * k, name=f"s{k}")
            for k, n in enumerate(SIDES)]


@pytest.fixture(scope="module")
def references():
    refs = []
    for p in _instances():
        om, K, f, xD, inner = oracle_assembly(p)
        refs.append(direct_solution(K, f))
    return refs


@pytest.mark.parametrize("mode", [A.NLF_MODE_FP64, A.NLF_MODE_MIXED])
@pytest.mark.parametrize("precond", [A.NLF_PRECOND_JACOBI, A.NLF_PRECOND_ILLT])
def test_graph_replays_and_solutions(gpu_ctx, references, precond, mode):
    """The oracle's solutions from graph replays, the same bits from eager launches and from a second graph."""
    print(f"[batch slices] graph, precond {precond} mode {mode}", flush=True)
    solver = batch.BatchSolver(_instances(), gpu_ctx, precond=precond)
    assert solver.K.symv_info() is not None
    x, its, res, st = solver.solve(tol=TOL, mode=mode)
    assert res.max() <= TOL and st.preconditioner == precond
    for i, (xi, ref) in enumerate(zip(solver.split(x), references)):
        assert rel_l2(xi.cpu().numpy(), ref) < BOUND, f"instance {i}"
    eager, its_e, _, _ = solver.solve(tol=TOL, mode=mode, use_graph=False)
    torch.cuda.synchronize()
    again, its_a, _, _ = solver.solve(tol=TOL, mode=mode)
    assert torch.equal(x, eager) and torch.equal(x, again)
    assert np.array_equal(its, its_e) and np.array_equal(its, its_a)


# (no ILLT with the conductivity: one factorisation serves the batch, fails and says so)
@pytest.mark.parametrize("precond,what", [(A.NLF_PRECOND_JACOBI, "load"), (A.NLF_PRECOND_JACOBI, "start"),
                                          (A.NLF_PRECOND_JACOBI, "conductivity"), (A.NLF_PRECOND_ILLT, "load"),
                                          (A.NLF_PRECOND_ILLT, "start")])
@pytest.mark.parametrize("mode", [A.NLF_MODE_FP64, A.NLF_MODE_MIXED])
def test_instances_stay_apart(gpu_ctx, references, precond, mode, what):
    """One instance with a not-a-number in its load or its start value, or an infinite conductivity: the others'
    solutions are the oracle's."""
    print(f"[batch slices] {what} precond {precond} mode {mode}", flush=True)
    solver = batch.BatchSolver(_instances(np.inf if what == "conductivity" else 1.0), gpu_ctx, precond=precond)
    assert solver.K.symv_info() is not None
    begin, end = solver.node_begin[BAD], solver.node_begin[BAD + 1]
    x0 = torch.zeros_like(solver.b)
    if what != "conductivity":
        (solver.b if what == "load" else x0)[(begin + end) // 2] = float("nan")
        (solver.b if what == "load" else x0)[[begin, end - 1]] = float("nan")
    x, its, res, st = solver.solve(tol=TOL, mode=mode, x0=x0)
    for i, (xi, ref) in enumerate(zip(solver.split(x), references)):
        if i != BAD:
            assert res[i] <= TOL, f"instance {i}"
            assert rel_l2(xi.cpu().numpy(), ref) < BOUND, f"instance {i}"


@pytest.mark.parametrize("sides,slices", [([32] * 35, False), ([32] * 36, True), ([72] * 4, False), ([64] * 7, True)])
def test_storage_by_size(gpu_ctx, sides, slices):
    """Small batches read the full storage, larger ones (600 slices; 400 with 4096 rows an instance) the slices: the
    bits tell which, and the solutions are the same."""
    problems = [configs.thermal_q4(n, 0.5, 3.3 / n, 1.0 + 0.01 * k, name=f"t{k}") for k, n in enumerate(sides)]
    solver = batch.BatchSolver(problems, gpu_ctx)
    rows = int(solver.node_begin[-1])
    print(f"[batch slices] {len(sides)} of {sides[0]}: {(rows + 63) // 64} slices, {rows // len(sides)} rows each", flush=True)
    x, its, res, st = solver.solve(tol=TOL, mode=A.NLF_MODE_MIXED)
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        y, its_y, res_y, _ = solver.solve(tol=TOL, mode=A.NLF_MODE_MIXED)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)
    assert max(res.max(), res_y.max()) <= TOL
    # the slices add in another order; the full storage gives the same bits again
    assert torch.equal(x, y) == (not slices)
    assert float((x - y).norm() / y.norm()) < BOUND


def test_autotuner_has_nothing_to_choose(gpu_ctx, tmp_path):
    """Where the solve reads the slices, the autotuner times and writes nothing; with them off it does."""
    solver = batch.BatchSolver(_instances(), gpu_ctx)
    cache = tmp_path / "tune.txt"
    assert solver.autotune(str(cache)) == 4.0 and not cache.exists()
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        chosen = solver.autotune(str(cache))
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)
    assert chosen in (1.0, 2.0, 4.0, 8.0, 16.0) and len(cache.read_text().split()) == 2
    assert solver.autotune(str(cache)) == chosen                # a stored choice is taken either way


def test_product_of_a_vector_with_nan(gpu_ctx):
    """nlf_spmv on the slices: not-a-number exactly in the rows with an entry for it, with windows of more than
    2048 values (radius of 21 elements on a 182 x 182 mesh)."""
    problem = configs.thermal_q4(182, 0.5, 21.3 / 182)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    api._search(g, problem.models)
    f, xD, inner = api.boundary_data(g, 1, problem.bcs)
    Kg = api._assemble(g, 0, problem.models, problem.materials, inner)
    slots, strips = Kg.symv_info()
    print(f"[batch slices] {slots} slots, {strips} strip values in {(f.size + 63) // 64} slices", flush=True)
    assert strips > 2048 * ((f.size + 63) // 64)
    x = np.random.default_rng(5).standard_normal(f.size)
    y = Kg.spmv(torch.from_numpy(x).to(gpu_ctx.device)).cpu().numpy()
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        assert rel_l2(y, Kg.spmv(torch.from_numpy(x).to(gpu_ctx.device)).cpu().numpy()) <= 1e-14
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)
    col = f.size // 2 + 3
    x[col] = np.nan
    bad = Kg.spmv(torch.from_numpy(x).to(gpu_ctx.device)).cpu().numpy()
    c = Kg.export(0)                                           # the upper triangle
    rows = np.repeat(np.arange(f.size), np.diff(c.outer))
    touched = np.zeros(f.size, dtype=bool)
    nz = c.val != 0.0
    touched[rows[nz & (c.inner == col)]] = True
    touched[c.inner[nz & (rows == col)]] = True
    assert np.array_equal(np.isnan(bad), touched)
    assert np.array_equal(bad[~touched], y[~touched])
