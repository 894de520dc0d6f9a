"""CG with sweeps on the full matrix storage below and above the size from which its values bypass the caches:
the residual of the solution, formed with the product that reads 32-bit columns one nonzero at a time."""
import pytest
import torch

from nonlocal_amd import _abi as A, _lib, api, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale,above", [(0.6, False), (0.7, True)])
def test_residual_on_both_sides(gpu_ctx, scale, above):
    gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 0)
    try:
        _check(gpu_ctx, scale, above)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_SPMV_SYMMETRIC, 1)


def _check(ctx, scale, above):
    p = configs.cfg1(scale)
    g = api.mesh_2d(p.mesh, ctx)
    api.find_neighbours(g, api._radii(p.models))
    _, _, inner = api.boundary_data(g, p.dof, p.bcs)
    K = api._assemble(g, p.physics, p.models, p.materials, inner)
    L = api._assemble(g, p.physics, p.models, p.materials, inner, part=A.NLF_PART_LOCAL)
    assert (K.info()["nnz_full"] * 8 > 256 << 20) == above
    cg = api.conjugate_gradient(K)
    cg.init_preconditioner(A.NLF_PRECOND_ILLT, L)
    cg.set_tolerance(1e-9)
    b = torch.ones(K.info()["rows"], dtype=torch.float64, device=ctx.device)
    x = cg.solve(b)
    y = torch.empty_like(b)
    assert _lib.load().nlf_spmv_lpr(K.h, 0x4200 | 16, 0, x.data_ptr(), y.data_ptr()) == 0
    ctx.synchronize()
    # CG stops at 1e-9 by its recurrence; the true residual follows it to rounding, far below 1e-9
    assert float((b - y).norm() / b.norm()) < 2e-9
