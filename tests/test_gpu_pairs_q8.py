"""Thermal Q8 pair blocks on the matrix cores against the node-centric contraction of the same entries (the
1e-13 relative to the largest entry that the Q4 pair blocks are held to), for every conductivity kind and
influence class, several groups and Dirichlet nodes, with the blocks in one pass and in node chunks."""
import numpy as np
import pytest

from nonlocal_amd import _abi as A
from nonlocal_amd import api, configs, meshgen
from oracle import oracle as O
from tests import helpers as H

pytestmark = pytest.mark.gpu

INFLUENCE = {"bell": dict(p=2.0, q=2.0), "fast": dict(p=2.0, q=1.0), "quartic": dict(p=4.0, q=3.0),
             "exponential": dict(influence=A.NLF_INFLUENCE_EXPONENTIAL, p=2.0, q=0.5),
             "constant": dict(influence=A.NLF_INFLUENCE_CONSTANT)}


def _problem(n, reach, influence, kind, groups=1):
    mesh = meshgen.structured_q8(n, jitter=0.2, seed=n)
    cut = [0, mesh.n_elems] if groups == 1 else [0, mesh.n_elems // 3, mesh.n_elems]
    mesh.group_begin = np.array(cut, dtype=np.int64)
    mesh.group_names = [f"g{k}" for k in range(groups)]
    models = [A.model(0.3 + 0.2 * k, reach / n, **INFLUENCE[influence]) for k in range(groups)]
    mats = [A.thermal_material(kind, (1.0 + k, 0.4, 0.1)) for k in range(groups)]
    return configs.Problem(f"q8_{n}_{influence}_{kind}_{groups}", mesh, 0, models, mats, configs.thermal_bcs(), {})


CASES = [_problem(1, 0.7, "bell", A.NLF_CONDUCTIVITY_ISOTROPIC), _problem(5, 1.3, "fast", A.NLF_CONDUCTIVITY_ORTHOTROPIC),
         _problem(14, 4.3, "bell", A.NLF_CONDUCTIVITY_ANISOTROPIC), _problem(13, 5.2, "quartic", A.NLF_CONDUCTIVITY_ANISOTROPIC, 2),
         _problem(9, 3.1, "exponential", A.NLF_CONDUCTIVITY_ISOTROPIC), _problem(11, 2.4, "constant", A.NLF_CONDUCTIVITY_ORTHOTROPIC, 2)]


@pytest.mark.parametrize("problem", CASES, ids=[c.name for c in CASES])
def test_pairs_match_node_contraction(gpu_ctx, problem):
    print(f"[q8 pairs] {problem.name}", flush=True)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    api.find_neighbours(g, H.radii(problem.models))
    inner = O.OracleMesh(problem.mesh).boundary(problem.bcs, 1)[2]
    whole = api._assemble(g, 0, problem.models, problem.materials, inner)
    gpu_ctx.set_option(A.NLF_OPT_ASSEMBLY_PAIRS, 0)
    try:
        node = api._assemble(g, 0, problem.models, problem.materials, inner)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_ASSEMBLY_PAIRS, 1)
    gpu_ctx.set_option(A.NLF_OPT_PAIR_BUDGET_MIB, 1)
    try:
        chunked = api._assemble(g, 0, problem.models, problem.materials, inner)
    finally:
        gpu_ctx.set_option(A.NLF_OPT_PAIR_BUDGET_MIB, 0)
    for part in (1, 2):
        a, b, c = whole.export(part), node.export(part), chunked.export(part)
        assert np.array_equal(a.inner, b.inner)
        assert np.array_equal(a.val, c.val), "chunked blocks are the same bits"
        if a.val.size:
            assert np.abs(a.val - b.val).max() <= 1e-13 * np.abs(b.val).max()
