"""Host arrays to the device and back, where their ways differ.

* Several arrays of one call are asked for together whatever their sizes: with a large and
  two small ones the call takes at most three times the call for the large one alone.
"""
import os
import time

import numpy as np
import pytest

from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(solver.__file__)), "weights",
                       "mpnn_box64.npz")


def test_arrays_of_one_call_share_their_wait():
    case = mesh.box_case(9, mach=0.3, kspace=3)  # BDiag 200 KB, the vectors 40 KB
    n = case.nshg
    w = np.load(WEIGHTS)
    bd = np.zeros((n, 5, 5), order="F")
    b, z = (np.zeros((n, 5), order="F") for _ in range(2))
    gpu = solver.GpuSolver(case)
    try:
        gpu.mpnn_init(w["dscale"])
        gpu.mpnn_set_weights(w["weights"])
        gpu.mpnn_enable(use_pc=0, keep_pair=True)
        gpu.upload_state(case.yold)
        gpu.predict()
        gpu.newton_iteration()
        want = gpu.mpnn_last_pair()
        call, p = solver.lib().phg_mpnn_last_pair, solver._p
        us = []
        for args in ((bd, b, z), (bd, None, None)):
            ts = []
            for _ in range(300):
                t = time.perf_counter()
                rc = call(gpu.h, *(p(a) for a in args))
                ts.append(1e6 * (time.perf_counter() - t))
                assert rc == 0
            us.append(float(np.median(ts)))
        # absent arrays, each alone
        for k in range(3):
            got = [np.full_like(a, -1.0) if i != k else None for i, a in enumerate(want)]
            assert call(gpu.h, *(p(a) for a in got)) == 0
            assert all(np.array_equal(g, a) for g, a in zip(got, want) if g is not None)
    finally:
        gpu.close()
    print(f"[host] three arrays {us[0]:.1f} us, the largest {us[1]:.1f}", flush=True)
    assert all(np.array_equal(x, y) for x, y in zip((bd, b, z), want))
    assert us[0] <= 3.0 * us[1]


# nodes: 1000 (both small), 1331 (downloads large), 1728 (both large), 74088 (no ring),
# 85184 and 97336 (ring)
@pytest.mark.parametrize("N", [3, 9, 10, 11, 41, 43, 45])
def test_state_arrays_round_trip(N):
    case = mesh.box_case(N, mach=0.3, kspace=1)
    n = case.nshg
    print(f"[host] N={N} nodes {n}", flush=True)
    rng = np.random.default_rng(N)
    up = [np.asfortranarray(rng.standard_normal((n, 5))) for _ in range(4)]
    gpu = solver.GpuSolver(case)
    L, p = solver.lib(), solver._p

    def down(call, want):
        """every subset of the call's results"""
        for mask in range(1 << len(want)):
            got = [np.full((n, 5), np.nan, order="F") if mask >> k & 1 else None
                   for k in range(len(want))]
            assert call(gpu.h, *(p(a) for a in got)) == 0
            for k, a in enumerate(got):
                if a is not None and want[k] is not None:
                    assert np.array_equal(a, want[k]), (mask, k)

    try:
        gpu.upload_state(up[0], up[1])
        gpu.upload_current(up[2], up[3])
        down(L.phg_state_download_old, up[:2])
        # (Dy is not set yet; its place among the others is taken all the same)
        down(L.phg_state_download, up[2:] + [None])
        # many uploads in a row without a download: the pinned buffer runs full
        for k in range(12):
            gpu.upload_current(up[k % 4], up[(k + 1) % 4])
        down(L.phg_state_download, [up[3], up[0], None])
        down(L.phg_state_download_old, up[:2])
    finally:
        gpu.close()
