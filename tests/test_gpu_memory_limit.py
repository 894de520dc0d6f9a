"""Storage that is only there to be faster is left out where there is no memory for it: the same solve as without
it, to the bit.  NLF_OPT_ALLOC_LIMIT_MIB makes the one block fail that is to be left out."""
import contextlib

import numpy as np
import pytest
import torch

from nonlocal_amd import _abi as A
from nonlocal_amd import api, batch, configs, learned, meshgen
from tests import helpers as H

pytestmark = pytest.mark.gpu

MODES = [A.NLF_MODE_FP64, A.NLF_MODE_MIXED, A.NLF_MODE_SPLIT]


@contextlib.contextmanager
def option(ctx, which, value, normal):
    ctx.set_option(which, value)
    try:
        yield
    finally:
        ctx.set_option(which, normal)


def full_storage(ctx):
    return option(ctx, A.NLF_OPT_SPMV_SYMMETRIC, 0, 1)


def limit(ctx, too_large):
    """A limit that a block of `too_large` bytes exceeds, by less than a MiB."""
    assert too_large > 2 << 20
    return option(ctx, A.NLF_OPT_ALLOC_LIMIT_MIB, (too_large - 1) >> 20, 0)


def without_slices(ctx, make, solve, reduced):
    """solve(K) with the full storage, then without memory for the slices (`reduced`: for their reduced values)."""
    K = make()
    with full_storage(ctx):
        want = solve(K)
    slots = make().symv_info()[0]
    if reduced:
        assert K.symv_info() is not None
    with limit(ctx, slots * 64 * (4 if reduced else 8)):
        got = solve(K)
        assert K.symv_info() is None
    assert torch.equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    return want


@pytest.mark.parametrize("mode,reduced", [(m, False) for m in MODES] + [(m, True) for m in MODES[1:]])
def test_cg(gpu_ctx, mode, reduced):
    print(f"[memory limit] cg mode {mode} reduced {reduced}", flush=True)
    n = {A.NLF_MODE_FP64: 100, A.NLF_MODE_MIXED: 270, A.NLF_MODE_SPLIT: 380}[mode]     # sizes that take the slices
    problem = configs.thermal_q4(n, 0.5, 9.3 / n)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    api._search(g, problem.models)
    f, xD, inner = api.boundary_data(g, 1, problem.bcs)
    b = torch.from_numpy(f).to(gpu_ctx.device)

    def make():
        K = api._assemble(g, 0, problem.models, problem.materials, inner)
        if mode == A.NLF_MODE_MIXED:
            K.make_fp32()
        if mode == A.NLF_MODE_SPLIT:
            K.make_split()
        return K

    def solve(K):
        cg = api.conjugate_gradient(K)
        cg.init_preconditioner(A.NLF_PRECOND_JACOBI)
        cg.set_tolerance(1e-12)
        return cg.solve(b, mode=mode), cg.iterations()

    without_slices(gpu_ctx, make, solve, reduced)


@pytest.mark.parametrize("mode,reduced", [(A.NLF_MODE_FP64, False), (A.NLF_MODE_MIXED, False), (A.NLF_MODE_MIXED, True)])
def test_flexible_cg(gpu_ctx, mode, reduced):
    print(f"[memory limit] flexible cg mode {mode} reduced {reduced}", flush=True)

    def make():
        n = 96 if mode == A.NLF_MODE_FP64 else 270
        tp = learned.TrainingProblem(n, seed=1, ctx=gpu_ctx, count=3, r=(5.3 if n == 96 else 11.3) / n)
        tp.K.make_fp32()
        tp.K.problem = tp
        return tp.K

    def solve(K):
        x, st = learned.fcg_solve(K, K.problem.learned, K.problem.b, tol=1e-10, max_it=20000, mode=mode)
        assert st.true_residual <= 1e-10
        return x, st.iterations

    without_slices(gpu_ctx, make, solve, reduced)


@pytest.mark.parametrize("mode,reduced", [(A.NLF_MODE_FP64, False), (A.NLF_MODE_MIXED, False), (A.NLF_MODE_MIXED, True)])
def test_batch(gpu_ctx, mode, reduced):
    print(f"[memory limit] batch mode {mode} reduced {reduced}", flush=True)
    problems = [configs.thermal_q4(n, 0.5, 5.3 / n, name=f"m{n}") for n in (150, 128, 141)]

    def make():
        solver = batch.BatchSolver(problems, gpu_ctx)
        solver.K.solver = solver
        return solver.K

    def solve(K):
        x, its, res, st = K.solver.solve(tol=1e-11, mode=mode)
        assert res.max() <= 1e-11
        return x, its

    without_slices(gpu_ctx, make, solve, reduced)


@pytest.mark.parametrize("build", [lambda: configs.cfg1(0.2), lambda: configs.cfg2(0.2)], ids=["q8", "elastic_q4"])
def test_factorisation(gpu_ctx, build):
    """The incomplete factorisation without the lists that its chunks work from: the same preconditioner."""
    problem = build()
    print(f"[memory limit] factorisation of {problem.mesh.n_nodes} rows", flush=True)
    om, KL, f, xD, inner = H.oracle_assembly(problem, part=A.NLF_PART_LOCAL)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    K = api._assemble(g, problem.physics, problem.models, problem.materials, inner, part=A.NLF_PART_LOCAL)
    upper = KL.export(0)
    above = np.diff(upper.outer) - 1                                    # entries beside the diagonal
    below = np.bincount(upper.inner, minlength=f.size) - 1
    entries = max(above.max(), below.max())
    width, lanes = next((w, l) for w, l in [(4, 4), (8, 8), (12, 16), (16, 16), (24, 32), (32, 32)] if entries <= w)
    r = torch.from_numpy(np.random.default_rng(2).standard_normal(f.size)).to(gpu_ctx.device)
    P = api.preconditioner(K, A.NLF_PRECOND_ILLT)
    z = P.solve(r).cpu().numpy()
    with limit(gpu_ctx, f.size * width * lanes * 4):
        Q = api.preconditioner(K, A.NLF_PRECOND_ILLT)
    assert Q.info()["ok"] and Q.info()["shift"] == P.info()["shift"] and Q.sweep_info() == P.sweep_info()
    assert H.rel_l2(Q.solve(r).cpu().numpy(), z) <= 1e-12            # as every layout against the oracle's


@pytest.mark.parametrize("q8", [True, False], ids=["q8", "q4"])
def test_assembly(gpu_ctx, q8):
    """Nonlocal heat matrices without the element-pair blocks: the node-centric contraction's values."""
    n = 14 if q8 else 40
    mesh = meshgen.structured_q8(n, jitter=0.2, seed=n) if q8 else meshgen.structured_q4(n, jitter=0.2, seed=n)
    print(f"[memory limit] assembly of {mesh.n_nodes} nodes", flush=True)
    models, mats = [configs.bell(0.4, 4.3 / n)], [A.thermal_material()]
    g = api.mesh_2d(mesh, gpu_ctx)
    api.find_neighbours(g, H.radii(models))
    inner = np.ones(mesh.n_nodes, dtype=np.uint8)
    inner[:n] = 0
    with option(gpu_ctx, A.NLF_OPT_ASSEMBLY_PAIRS, 0, 1):
        want = api._assemble(g, 0, models, mats, inner)
    with limit(gpu_ctx, int(g.neighbours()[0][-1]) * mesh.nn ** 2 * 8):
        got = api._assemble(g, 0, models, mats, inner)
    for part in (1, 2):
        a, b = got.export(part), want.export(part)
        assert np.array_equal(a.inner, b.inner) and np.array_equal(a.val, b.val)
