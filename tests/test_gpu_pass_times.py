"""Device-clock times of the solver's passes against each other.

* The FP64 block pass with discontinuity capturing beside the matrix tau: per point and
  block DC adds six values to the 25 of W PTau and the point record's 8, and some forty
  operations (weight, sums of A0's entries) to the matrix product's three hundred, so the
  pass may take at most 1.4 times the time without DC, bytes and operations together.
"""
import pytest

from phasta_amd import config, mesh, solver

pytestmark = pytest.mark.gpu


def test_dc_beside_the_matrix_tau():
    N = 33
    case = mesh.box_case(N, mach=0.3, kspace=5)
    ms = {}
    for idc in (0, 1):
        gpu = solver.GpuSolver(case, params=config.solver_params(N, 0.3, 5, idc=idc, itau=10))
        try:
            ms[idc] = 1e9
            for _ in range(8):
                gpu.upload_state(case.yold)
                gpu.predict()
                ms[idc] = min(ms[idc], gpu.newton_iteration()["ms_blocks"])
        finally:
            gpu.close()
    print(f"[passes] blocks {1e3 * ms[0]:.0f} us, with DC {1e3 * ms[1]:.0f} us", flush=True)
    assert ms[0] > 0.0
    assert ms[1] <= 1.4 * ms[0]
