"""The neighbour preconditioner's cluster inverses (Gauss-Jordan in registers,
rf_precond.hip) for every thread layout and at its edges, against numpy.

Bound: elimination with partial pivoting solves a cluster system to about
dim eps cond(A_CC) of the solution; numpy's own solve the same: 4 of these.
The layouts allow fibers a thousandth apart; some clusters of the eight-term
systems then hold entries above the diagonal's, so the pivot rows change.
"""
import numpy as np
import pytest

import rigidfibers_kth_amd as rf
from rigidfibers_kth_amd.layouts import layout

pytestmark = pytest.mark.gpu

# clusters of 6 to 126 rows
SHAPES = [(1, 1), (1, 6), (2, 4), (3, 2), (4, 2), (3, 6), (7, 2), (5, 4), (6, 3), (8, 2), (3, 1), (5, 6), (7, 4),
          (8, 3), (6, 6), (7, 5), (8, 4)]


@pytest.mark.parametrize("precision", [rf.PREC_FP64, rf.PREC_MIXED])
@pytest.mark.parametrize("M,K", SHAPES)
def test_cluster_inverses(M, K, precision):
    N = 40
    pos, ori = layout(N, 0.1, 7 * M + K, min_gap=1e-3)
    p = rf.default_params(num_terms=M, precond=1, precond_neighbours=K, precision=precision, gmres_restart=30,
                          gmres_max_iters=3000, gmres_tol=1e-8)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        A = sim.matrix()
        nbr, _ = sim.neighbours(K)
        r = np.random.default_rng(M).normal(size=sim.n)
        sim.solve_system()
        z = sim.precond_apply(r)
    m = 3 * M
    worst, moved = 0.0, 0
    for i in range(N):
        idx = np.concatenate([np.arange(c * m, (c + 1) * m) for c in np.concatenate([[i], nbr[i]])])
        B = A[np.ix_(idx, idx)]
        x = np.linalg.solve(B, r[idx])
        bound = 4.0 * idx.size * np.finfo(float).eps * np.linalg.cond(B) * np.linalg.norm(x)
        worst = max(worst, np.abs(z[i * m:(i + 1) * m] - x[:m]).max() / bound)
        moved += np.abs(B - np.eye(idx.size)).max() > 1.0
    print("M=%d K=%d: %d rows, %.2e of the bound, %d clusters with entries above the diagonal" % (
        M, K, m * (K + 1), worst, moved))
    assert worst <= 1.0


@pytest.mark.parametrize("M,K", [(7, 6), (8, 5)])
def test_clusters_beyond_the_largest_are_refused(M, K):
    pos, ori = layout(20, 2e-2, 3)
    p = rf.default_params(num_terms=M, precond=1, precond_neighbours=K)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        with pytest.raises(rf.RigidFibersError):
            sim.solve_system()
