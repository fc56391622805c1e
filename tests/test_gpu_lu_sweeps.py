"""The triangular solves of FP64 factors, one launch a sweep (rf_lu.hip), at
their edges: one block, partial last blocks, one and several blocks per CU's
worth of rows; against numpy on matrices whose rows have to be exchanged.

Bound: a solution with partial pivoting is within about n eps cond(A); numpy's
own is too.  The factors' own part is tested elsewhere; here 4 n eps cond(A).
"""
import numpy as np
import pytest

import rigidfibers_kth_amd as rf
from rigidfibers_kth_amd.layouts import layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(1, 2), (1, 21), (7, 3), (1, 22), (5, 13), (2, 171), (4, 97), (5, 300), (3, 911)])
def test_direct_solves(M, N):
    pos, ori = layout(N, 5e-2 if N > 2 else 1e-3, 5 + N)
    p = rf.default_params(num_terms=M, num_quad_intervals=4, use_direct_solver=1, use_analytical_integration=0)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        got = []
        for _ in range(2):  # the scratch of the sweeps is used again
            sim.assemble_system()
            sim.solve_system()
            got.append(sim.coefficients())
        A, b = sim.matrix(), sim.rhs()
    want = np.linalg.solve(A, b)
    bound = 4.0 * b.size * np.finfo(float).eps * np.linalg.cond(A)
    err = np.linalg.norm(got[0] - want) / np.linalg.norm(want)
    print("n=%d: %.2e, bound %.2e" % (b.size, err, bound))
    assert err <= bound
    assert np.array_equal(got[0], got[1])
