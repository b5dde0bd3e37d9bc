"""The network's gradients at the sizes where their sums differ: fewer rows than
a tile, rows that no tile divides, fewer and more workgroups than the partials
are capped at.

Bar: as in the fixed-size test against the oracle's bf16 model, 1e-2 normwise
(bf16 roundings of intermediate values land on different sides of a tie when
float sums are taken in another order).
"""
import numpy as np
import pytest

import pympnn as M
from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2, 3, 7, 13, 22])
def test_gradients_match_oracle(N):
    case = mesh.box_case(N, mach=0.3, kspace=5)
    g = M.periodic_graph(case)
    rng = np.random.default_rng(N)
    p = M.init_params(5)
    n = case.nshg
    bd = np.asfortranarray(rng.standard_normal((n, 5, 5)))
    v = np.asfortranarray(rng.standard_normal((n, 5)))
    t = np.asfortranarray(v + 0.3 * rng.standard_normal((n, 5)))
    dscale = np.full(25, 2.0, dtype=np.float32)
    gpu = solver.GpuSolver(case)
    try:
        gpu.mpnn_init(dscale)
        gpu.mpnn_set_weights(solver.mpnn_flatten(p))
        loss, grad = gpu.mpnn_train_step(bd, v, t, lr=0.0, want_grad=True)
    finally:
        gpu.close()
    x, s = M.features(bd, v, dscale, g.active)
    ystar = ((t - v) * s).astype(np.float32)
    loss_ref, ref, _ = M.loss_and_grad(p, g, x, ystar)
    assert abs(loss - loss_ref) <= 1e-2 * loss_ref
    got = solver.mpnn_unflatten(grad)
    for k, _ in solver.MPNN_SHAPES:
        assert np.linalg.norm(got[k] - ref[k]) < 1e-2 * np.linalg.norm(ref[k]), k
