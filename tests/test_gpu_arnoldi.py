"""The one-launch Arnoldi step (rf_linalg.hip) through rf_solve: GMRES on the
stored matrix against the same iteration in numpy, at the edges of its forms:
one workgroup, a row a thread to 32 workgroups (16384 rows), more rows than
that, more than 16 and more than 32 basis vectors, restarts in between.

Classical Gram-Schmidt applied twice keeps the basis orthogonal to rounding,
so both runs build the same Krylov space: the true backward error meets the
tolerance and the iteration counts agree to one (a residual that lies within
rounding of the tolerance may decide either way).
"""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import rigidfibers_kth_amd as rf
from rigidfibers_kth_amd.layouts import layout

pytestmark = pytest.mark.gpu


def _gmres(A, b, m, tol, maxit):
    x, total, bn = np.zeros_like(b), 0, np.linalg.norm(b)
    while True:
        r = b - A @ x
        V = [r / np.linalg.norm(r)]
        H = np.zeros((m + 1, m))
        beta = np.linalg.norm(r)
        for j in range(m):
            w = A @ V[j]
            Q = np.array(V)
            for _ in range(2):
                h = Q @ w
                w = w - h @ Q
                H[:j + 1, j] += h
            H[j + 1, j] = np.linalg.norm(w)
            V.append(w / H[j + 1, j])
            total += 1
            e = np.zeros(j + 2)
            e[0] = beta
            y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)
            if np.linalg.norm(e - H[:j + 2, :j + 1] @ y) <= tol * bn or total >= maxit or j == m - 1:
                xt = x + y @ np.array(V[:j + 1])
                if np.linalg.norm(b - A @ xt) <= tol * bn or total >= maxit:
                    return xt, total
        x = xt


@pytest.mark.parametrize("M,N,phi,restart,tol", [
    (1, 2, 1e-3, 30, 1e-11),      # 6 rows: one workgroup, breakdown of the space near its size
    (1, 170, 2e-2, 30, 1e-11),    # 510 and 513 rows: either side of one workgroup
    (1, 171, 2e-2, 5, 1e-11),     # restarts
    (5, 100, 5e-2, 60, 1e-12),
    (3, 911, 2e-2, 30, 1e-11),    # 8199 rows: 32 workgroups
    (8, 682, 1e-2, 40, 1e-12),    # 16368 rows: the last size with a row a thread
    (8, 683, 1e-2, 12, 1e-10),    # 16392 rows: several rows a thread, at most 16 vectors
    (8, 683, 1e-2, 60, 1e-12),    # and more than 16
])
def test_gmres_follows_the_same_iteration(M, N, phi, restart, tol):
    pos, ori = layout(N, phi, 40 + N)
    p = rf.default_params(num_terms=M, num_quad_intervals=4, use_direct_solver=0, use_analytical_integration=0,
                          gmres_restart=restart, gmres_max_iters=400, gmres_tol=tol)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        sim.solve_system()
        A, b, x, st = sim.matrix(), sim.rhs(), sim.coefficients(), sim.stats()
    be = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    want, iters = _gmres(A, b, restart, tol, 400)
    diff = np.linalg.norm(x - want) / np.linalg.norm(want)
    print("n=%d restart %d: %d iterations (numpy %d), backward error %.2e, x %.2e" % (
        b.size, restart, st.last_gmres_iters, iters, be, diff))
    assert st.last_solver == rf.SOLVER_GMRES
    assert be <= tol * (1 + 1e-3) + 1e-15
    assert abs(st.last_gmres_iters - iters) <= 1


def test_more_than_32_basis_vectors():
    """Fibers in near contact: several cycles of 60 vectors.  The iteration's
    estimate and the true residual agree only while the basis is orthogonal."""
    N = 300
    pos, ori = layout(N, 5e-2, 0x5EED0003)
    p = rf.default_params(gmres_restart=60, gmres_max_iters=3000, gmres_tol=1e-10)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.step()
        sim.step()
        sim.assemble_system()
        sim.solve_system()
        A, b, x, st = sim.matrix(), sim.rhs(), sim.coefficients(), sim.stats()
    be = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    print("%d iterations, backward error %.2e" % (st.last_gmres_iters, be))
    assert st.last_solver == rf.SOLVER_GMRES and st.last_gmres_iters > 60
    assert be <= 1e-10 * (1 + 1e-3)


def test_solvers_on_their_own_threads():
    """Steps that wait for each other's workgroups, from several streams at a
    time: the results of one after the other, bit for bit."""
    p = rf.default_params(gmres_restart=30, gmres_max_iters=300, gmres_tol=1e-11)

    def solve(seed):
        pos, ori = layout(120, 2e-2, seed)
        with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
            for _ in range(3):
                sim.assemble_system()
                sim.solve_system()
            return sim.coefficients()

    seeds = list(range(60, 66))
    want = [solve(s) for s in seeds]
    with ThreadPoolExecutor(len(seeds)) as pool:
        got = list(pool.map(solve, seeds))
    for w, g in zip(want, got):
        assert np.array_equal(w, g)
