"""The chunked ILLT sweeps where their plan can go wrong, against the oracle's IC(0) apply at the 1e-12
that every sweep layout is held to: chunk edges (64 rows of nodes), one chunk longer than the LDS
window, node numbers in random order (dependencies from everywhere, most of them read through memory),
rows with up to 32 entries on one side of the diagonal and few on the other, and one row with more (the
packed sweep)."""
import ctypes as C

import numpy as np
import pytest
import torch

from nonlocal_amd import _abi as A
from nonlocal_amd import api, configs, meshgen
from nonlocal_amd._lib import load
from oracle import oracle as O
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _mesh(xy, elems, edges):
    """A one-group Q4 mesh whose first boundary group holds `edges` (the others are empty)."""
    begin = np.array([0] + [len(edges)] * 4, dtype=np.int64)
    return meshgen.Mesh2D(xy=np.ascontiguousarray(xy, dtype=np.float64), elems=np.ascontiguousarray(elems, dtype=np.int32),
                          nn=4, group_begin=np.array([0, len(elems)], dtype=np.int64), group_names=["m"],
                          bedges=np.asarray(edges, dtype=np.int32), bgroup_begin=begin)


def _problem(mesh):
    return configs.Problem("sweep", mesh, 0, [A.model(1.0, 0.0)], [A.thermal_material()],
                           [A.boundary(A.NLF_BC_FIRST_KIND, 0.0), A.boundary(), A.boundary(), A.boundary()], {})


def grid(nx, ny, seed=None):
    x, y = np.meshgrid(np.arange(nx + 1) / nx, np.arange(ny + 1) / nx)
    j, i = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    b = (j * (nx + 1) + i).ravel()
    elems = np.stack([b, b + 1, b + nx + 2, b + nx + 1], axis=1)
    edges = np.array([[k * (nx + 1), (k + 1) * (nx + 1)] for k in range(ny)])
    xy = np.stack([x.ravel(), y.ravel()], axis=1)
    if seed is not None:
        new = np.random.default_rng(seed).permutation(len(xy))
        moved = np.empty_like(xy)
        moved[new] = xy
        xy, elems, edges = moved, new[elems], new[edges]
    return _problem(_mesh(xy, elems, edges))


def fan(m, hub_first=False):
    """m quads around one node of 2 m neighbours, numbered last or first; two outer nodes are fixed."""
    t = np.linspace(0.0, 2.0 * np.pi, 2 * m, endpoint=False)
    r = np.where(np.arange(2 * m) % 2, 1.0, 0.9)
    xy = np.concatenate([np.stack([r * np.cos(t), r * np.sin(t)], axis=1), [[0.0, 0.0]]])
    k = 2 * np.arange(m)
    elems = np.stack([np.full(m, 2 * m), k, k + 1, (k + 2) % (2 * m)], axis=1)
    edges = np.array([[0, 1]])
    if hub_first:
        xy, elems, edges = np.roll(xy, 1, axis=0), (elems + 1) % (2 * m + 1), edges + 1
    return _problem(_mesh(xy, elems, edges))


def elastic_q8(n):
    p = configs.cfg2(n / 300)
    p.mesh = meshgen.structured_q8(n, jitter=0.2, seed=3)
    return p


CASES = [
    ("one_row", lambda: grid(70, 1), 2),
    ("long_strip", lambda: grid(400, 3), 2),
    ("chunk_edge_63", lambda: grid(70, 62), 2),
    ("chunk_edge_65", lambda: grid(70, 65), 2),
    ("three_chunks", lambda: grid(150, 131), 2),
    ("random_numbers", lambda: grid(90, 80, seed=5), 2),
    ("q8_elastic", lambda: elastic_q8(15), 2),
    ("fan_32", lambda: fan(17), 2),
    ("fan_34", lambda: fan(18), 0),
    ("fan_6_hub_first", lambda: fan(4, hub_first=True), 2),
    ("fan_32_hub_first", lambda: fan(17, hub_first=True), 2),
]


@pytest.mark.parametrize("name,build,kernel", CASES, ids=[c[0] for c in CASES])
def test_sweep_matches_oracle(gpu_ctx, name, build, kernel):
    problem = build()
    om, KL, f, xD, inner = H.oracle_assembly(problem, part=A.NLF_PART_LOCAL)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    K = api._assemble(g, problem.physics, problem.models, problem.materials, inner, part=A.NLF_PART_LOCAL)
    P, Pg = O.OraclePrecond(A.NLF_PRECOND_ILLT, KL), api.preconditioner(K, A.NLF_PRECOND_ILLT)
    assert P.ok()[0] and Pg.info()["ok"]
    info = Pg.sweep_info()
    print(f"[sweep] {name}: {f.size} rows, {info}", flush=True)
    assert info["forward"]["kernel"] == kernel and info["backward"]["kernel"] == kernel
    rng = np.random.default_rng(3)
    for k in range(3):                       # again and again: the buffers are emptied for the next apply
        r = rng.standard_normal(f.size)
        z = Pg.solve(torch.from_numpy(r).to(gpu_ctx.device)).cpu().numpy()
        assert H.rel_l2(z, P.apply(r)) <= 1e-12
    # not-a-number in, not-a-number out (and no wait for it), and the next apply is untouched by it
    bad = r.copy()
    bad[int(np.flatnonzero(inner)[0])] = np.nan
    assert np.isnan(Pg.solve(torch.from_numpy(bad).to(gpu_ctx.device)).cpu().numpy()).any()
    assert np.array_equal(z, Pg.solve(torch.from_numpy(r).to(gpu_ctx.device)).cpu().numpy())


def test_shifted_factorisation(gpu_ctx):
    """Couplings enlarged until the unshifted IC(0) meets a non-positive pivot: the retries find the oracle's
    shift, the factor is emptied in between, and the apply matches."""
    problem = grid(70, 66)
    om, KL, f, xD, inner = H.oracle_assembly(problem, part=A.NLF_PART_LOCAL)
    g = api.mesh_2d(problem.mesh, gpu_ctx)
    K = api._assemble(g, 0, problem.models, problem.materials, inner, part=A.NLF_PART_LOCAL)
    c = KL.export(0)
    rows = np.repeat(np.arange(len(c.outer) - 1), np.diff(c.outer))
    add = np.where(rows != c.inner, 0.6 * c.val, 0.0)
    KL.set_values(c.val + add)
    rc = np.ascontiguousarray(np.stack([rows, c.inner], axis=1), dtype=np.int64)
    gpu_ctx.check(load().nlf_matrix_add_pairs(K.h, len(add), rc.ctypes.data_as(C.POINTER(C.c_int64)),
                                              np.ascontiguousarray(add).ctypes.data_as(C.POINTER(C.c_double))))
    P, Pg = O.OraclePrecond(A.NLF_PRECOND_ILLT, KL), api.preconditioner(K, A.NLF_PRECOND_ILLT)
    ok, shift = P.ok()
    assert ok and shift > 0.0
    assert Pg.info()["ok"] and Pg.info()["shift"] == shift
    r = np.random.default_rng(4).standard_normal(f.size)
    z = Pg.solve(torch.from_numpy(r).to(gpu_ctx.device)).cpu().numpy()
    print(f"[sweep] shift {shift}, rel err {H.rel_l2(z, P.apply(r)):.2e}", flush=True)
    # the shifted factor is ill conditioned: an error of 1e-16 in the pivots grows by 1 / shift and more
    assert H.rel_l2(z, P.apply(r)) <= 1e-10
