"""The block pass at the sizes where its wavefronts differ: few blocks and many,
lanes without a block, elements loaded past the last one, entries of several
lanes, every stored type and tau.

Bar, norm of the difference over the norm: an entry is a sum of products of up
to eight rounded factors, and a row's elements and points are added one after
the other, at most some hundred additions whose errors partly cancel: 16 units
of rounding for the products and as many for the additions, 32 units in all
(float 2^-24: 1.9e-6; double 2^-53: 3.6e-15, where the oracle's own sums round
as much again, so 7.1e-15 there).
"""
import numpy as np
import pytest

import pyoracle
from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision", [solver.PHG_FP64, solver.PHG_MIXED])
@pytest.mark.parametrize("N,itau,idc", [(2, 0, 0), (3, 0, 0), (5, 1, 0), (7, 0, 1), (6, 10, 0),
                                        (5, 10, 1), (13, 0, 0)])
def test_blocks_against_oracle(N, itau, idc, precision):
    # (a graded box has an even number of cells)
    case = mesh.box_case(N, mach=0.3, kspace=5, grade=1.0 if N % 2 else 1.1, cfl=3.0)
    params = dict(case.params, itau=itau, idc=idc)
    o = pyoracle.Oracle(case, params=params)
    y, ac = o.itr_predict_bc(case.yold)
    rng = np.random.default_rng(N)
    ac = np.asfortranarray(ac + 1e3 * rng.standard_normal(ac.shape))
    res, _, bdiag, lhsk = o.elmgmrs(y, ac)
    g = solver.GpuSolver(case, params=params, precision=precision)
    gres, _, gbdiag, glhsk = g.elmgmrs(y, ac)
    g.close()
    tol = 1.9e-6 if precision == solver.PHG_MIXED else 7.1e-15
    assert rel(glhsk, lhsk) < tol
    assert rel(gbdiag, bdiag) < tol
    assert rel(gres, res) < 1e-12
