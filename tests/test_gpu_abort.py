"""What an aborted Newton iteration (tnanq, rstatCheck) leaves resident: the state as it
was and a zero Dy, not the increment of an earlier iteration."""
import numpy as np
import pytest

from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [solver.PHG_FP64, solver.PHG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("abort", ["nan", "divergence"])
def test_aborted_iteration_leaves_no_increment(abort, precision):
    case = mesh.box_case(4, mach=0.3, kspace=10)
    zero = np.zeros((case.nshg, 5), order="F")
    gpu = solver.GpuSolver(case, precision=precision)
    try:
        # an iteration with an increment: from the box's state, or from it scaled down
        # to 1e-6 of its residual (a rest state disturbed by 1e-6)
        rest = zero.copy(order="F")
        rest[:, 3], rest[:, 4] = 1.0e5, 300.0
        first = case.yold if abort == "nan" else rest + 1e-6 * (case.yold - rest)
        gpu.upload_state(np.asfortranarray(first))
        gpu.predict()
        gpu.newton_iteration()
        assert np.linalg.norm(gpu.download_state()[2]) > 0.0
        y = case.yold.copy(order="F")
        if abort == "nan":
            y[case.nshg // 2, 3] = np.nan
        gpu.upload_current(y, zero)
        with pytest.raises(solver.PhgError) as ei:
            gpu.newton_iteration()
        assert ei.value.code == (10 if abort == "nan" else 11)
        after, _, dy = gpu.download_state()
    finally:
        gpu.close()
    assert np.array_equal(after, y, equal_nan=True)
    assert np.array_equal(dy, zero)
