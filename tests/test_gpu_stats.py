"""What the solver reports about its own work.

* ms_spmv counts the cycle's products and nothing else, also where the network's acceptance
  test (two products, four inner products and a wait for the host) stands before the first
  Gram-Schmidt step: at most twice the time per product of the plain solve, the factor of
  two for the event pair around the test's two products, whose packets take some 5 us each,
  as long as a product on this mesh.
"""
import os

import numpy as np
import pytest

from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(solver.__file__)), "weights",
                       "mpnn_box64.npz")


def test_product_time_with_the_network():
    case = mesh.box_case(6, mach=0.3, kspace=1, grade=1.1, cfl=3.0)
    w = np.load(WEIGHTS)
    gpu = solver.GpuSolver(case)
    per = {}
    try:
        gpu.mpnn_init(w["dscale"])
        gpu.mpnn_set_weights(w["weights"])
        for use_pc in (0, 1):
            gpu.mpnn_enable(use_pc=use_pc)
            per[use_pc] = 1e9
            for _ in range(20):
                gpu.upload_state(case.yold)
                gpu.predict()
                st = gpu.newton_iteration()
                per[use_pc] = min(per[use_pc], st["ms_spmv"] / st["n_spmv"])
    finally:
        gpu.close()
    print(f"[stats] us per product: plain {1e3 * per[0]:.2f}, network {1e3 * per[1]:.2f} "
          f"(of {st['n_spmv']})", flush=True)
    assert 0.0 < per[1] <= 2.0 * per[0]
