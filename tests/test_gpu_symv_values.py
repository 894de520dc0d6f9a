"""Which storage the products of a mixed or split solve read: the slices from the size at which they are faster,
the full storage below it, with the same solution."""

import pytest
import torch

from nonlocal_amd import _abi as A
from nonlocal_amd import api, configs

pytestmark = pytest.mark.gpu

TOL = 1e-11


# FP32 values take the slices from 1024 of them and 80 MiB in the full storage or from 512 and 256 MiB, split ones from
# 1024 and 256 MiB, FP64 ones at any size, but with windows over 2048 values (the last two) from 512
@pytest.mark.parametrize("mode,n,reach,slices", [
    (A.NLF_MODE_MIXED, 250, 9.3, False), (A.NLF_MODE_MIXED, 260, 9.3, True), (A.NLF_MODE_MIXED, 400, 3.1, False),
    (A.NLF_MODE_MIXED, 190, 22.3, False), (A.NLF_MODE_MIXED, 190, 25.3, True),
    (A.NLF_MODE_SPLIT, 250, 15.3, False), (A.NLF_MODE_SPLIT, 260, 13.3, True), (A.NLF_MODE_SPLIT, 330, 8.3, False),
    (A.NLF_MODE_FP64, 40, 9.3, True), (A.NLF_MODE_FP64, 178, 21.3, False), (A.NLF_MODE_FP64, 182, 21.3, True)])
def test_storage_by_size(gpu_ctx, mode, n, reach, slices):
    problem = configs.thermal_q4(n, 0.5, reach / n)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    api._search(g, problem.models)
    f, xD, inner = api.boundary_data(g, 1, problem.bcs)
    K = api._assemble(g, 0, problem.models, problem.materials, inner)
    K.make_split()
    size = {A.NLF_MODE_FP64: 8, A.NLF_MODE_MIXED: 4, A.NLF_MODE_SPLIT: 6}[mode]
    print(f"[storage] mode {mode} n {n}: {(f.size + 63) // 64} slices, {K.info()['nnz_full'] * size / 2 ** 20:.1f} MiB", flush=True)
    cg = api.conjugate_gradient(K)
    cg.init_preconditioner(A.NLF_PRECOND_JACOBI)
    cg.set_tolerance(TOL)
    b = torch.from_numpy(f).to(gpu_ctx.device)
    x = cg.solve(b, mode=mode)
    read = cg.stats.spmv_bytes
    assert cg.stats.true_residual <= (TOL if mode != A.NLF_MODE_FP64 else 10 * TOL)
    slots, strips = K.symv_info() or (0, 0)
    assert (read == slots * 64 * size + 2 * strips * 8 + 32 * f.size) == slices
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        y = cg.solve(b, mode=mode)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)
    # each solution is within the condition number, about n^2, times its residual of the exact one
    assert float((x - y).norm() / y.norm()) <= 4 * n ** 2 * TOL
