"""Gradient of the learned preconditioner's loss where the backward kernels' blocks take more than one trip over
the nodes (16 x 256 and 32 x 256 of them) and end in a remainder, against the FP64 oracle."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from nonlocal_amd import learned
from oracle import learned_oracle as LO
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [5, 64, 100])     # 36, 4225 and 10201 nodes
def test_gradient_over_several_trips(gpu_ctx, side):
    tp = learned.TrainingProblem(side, seed=1, ctx=gpu_ctx, count=3, r=1.5 / side)
    n = tp.problem.mesh.n_nodes
    csr = tp.K.export(2)
    K = sp.csr_matrix((csr.val, csr.inner, csr.outer), shape=(n, n))
    outer, cols, feat, s = tp.learned.graph()
    rng = np.random.default_rng(side)
    w = learned.init_weights(side).astype(np.float64)
    w[LO.P_WOUT:LO.P_WOUT + LO.H] = rng.uniform(-0.2, 0.2, LO.H)
    w = w.astype(np.float32)
    tp.learned.set_weights(w)
    e = rng.standard_normal(n)
    r = K @ e
    dev = gpu_ctx.device
    loss, g = tp.learned.loss_grad(torch.from_numpy(r).to(dev), torch.from_numpy(e).to(dev))
    lo, go = LO.loss_grad(w.astype(np.float64), outer, cols, feat.astype(np.float64), s.astype(np.float64), K, r, e)
    assert abs(loss - lo) <= 1e-5 * abs(lo)
    assert rel_l2(g, go) < 1e-4
