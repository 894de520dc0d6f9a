"""Which storage the products of a mixed or split solve read: the slices from the size at which they are faster,
the full storage below it, with the same solution."""

import pytest
import torch

from nonlocal_amd import _abi as A
from nonlocal_amd import api, configs

pytestmark = pytest.mark.gpu

TOL = 1e-11


# 9.3 elements' reach: 24.6 and 26.7 million nonzeros around 96 MiB of FP32 values, 41.5 and 47.1 around 256 MiB of split ones
@pytest.mark.parametrize("mode,n,slices", [(A.NLF_MODE_MIXED, 240, False), (A.NLF_MODE_MIXED, 250, True),
                                           (A.NLF_MODE_SPLIT, 310, False), (A.NLF_MODE_SPLIT, 330, True),
                                           (A.NLF_MODE_FP64, 40, True)])
def test_storage_by_size(gpu_ctx, mode, n, slices):
    problem = configs.thermal_q4(n, 0.5, 9.3 / n)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    api._search(g, problem.models)
    f, xD, inner = api.boundary_data(g, 1, problem.bcs)
    K = api._assemble(g, 0, problem.models, problem.materials, inner)
    K.make_split()
    size = {A.NLF_MODE_FP64: 8, A.NLF_MODE_MIXED: 4, A.NLF_MODE_SPLIT: 6}[mode]
    print(f"[storage] mode {mode} n {n}: {K.info()['nnz_full'] * size / 2 ** 20:.1f} MiB", flush=True)
    cg = api.conjugate_gradient(K)
    cg.init_preconditioner(A.NLF_PRECOND_JACOBI)
    cg.set_tolerance(TOL)
    b = torch.from_numpy(f).to(gpu_ctx.device)
    x = cg.solve(b, mode=mode)
    read = cg.stats.spmv_bytes
    assert cg.stats.true_residual <= (TOL if mode != A.NLF_MODE_FP64 else 10 * TOL)
    slots, strips = K.symv_info()
    assert (read == slots * 64 * size + 2 * strips * 8 + 32 * f.size) == slices
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        y = cg.solve(b, mode=mode)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)
    # each solution is within the condition number, about n^2, times its residual of the exact one
    assert float((x - y).norm() / y.norm()) <= 4 * n ** 2 * TOL
