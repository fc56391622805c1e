"""The analytic assembly (a wavefront per group of targets, near and far pairs
in turn; rf_assemble.hip) at its edges: fiber counts around the groups of 5 to
20 targets, odd and large numbers of outer points (self-mirrored middle point,
one pair at a time), every number of terms, all pairs near, all far, mixed.

Rows of A x against a 64-bit sum of the integrals themselves, to be as close
as the oracle's matrix up to a factor of three for the different rounding, and
1e-12 of max |y| (a far pair's sums are within 2e-13 of its largest entry).
FP32 storage adds 6e-8 of |A| |x|, and its recurrences for |R|^2 >= 10 a few
FP32 roundings of a moment: 4e-6 of |A - I| |x| with the rounding of A.
"""
import numpy as np
import pytest

import oracle
import rigidfibers_kth_amd as rf
from rigidfibers_kth_amd.layouts import layout
from test_gpu_operator_far import EPS, _rows, _shell

pytestmark = pytest.mark.gpu


def _check(pos, ori, M, noqi, precision, fibers, panels):
    N = pos.size // 3
    x = np.random.default_rng(M + N).normal(size=3 * M * N)
    p = rf.default_params(use_analytical_integration=1, num_terms=M, num_quad_intervals=noqi, slenderness=EPS,
                          precision=precision)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        A, b = sim.matrix(), sim.rhs()
        bo = sim.operator(rf.OP_RHS)
        pos, ori = (np.asarray(v).ravel() for v in sim.state()[:2])
    Ao = oracle.assemble_matrix(1, EPS, pos, ori, M, noqi)
    y, yo = A @ x, Ao @ x
    scale = np.abs(yo).max()
    err = closed = 0.0
    for i in fibers:
        rows = slice(3 * M * i, 3 * M * (i + 1))
        want = _rows(i, pos, ori, M, noqi, x, panels=panels)
        err = max(err, np.abs(y[rows] - want).max() / scale)
        closed = max(closed, np.abs(yo[rows] - want).max() / scale)
    fp32 = 4e-6 * (np.abs(Ao - np.eye(x.size)) @ np.abs(x)).max() / scale if precision == rf.PREC_MIXED else 0.0
    print("N=%d M=%d NoQI=%d: %.2e, oracle's matrix %.2e" % (N, M, noqi, err, closed))
    assert err <= 3.0 * closed + 1e-12 + fp32
    for i in range(N):  # the diagonal blocks are exactly the identity
        block = slice(3 * M * i, 3 * M * (i + 1))
        assert np.array_equal(A[block, block], np.eye(3 * M))
    # the right-hand side's part: the operator's, summed from the same pairs
    # (mixed: its far points pass the FP32 recurrences too, so FP64 only)
    if precision == rf.PREC_FP64:
        assert np.abs(b - bo).max() <= (3.0 * closed + 1e-12) * max(scale, np.abs(bo).max())


@pytest.mark.parametrize("precision", [rf.PREC_FP64, rf.PREC_MIXED])
@pytest.mark.parametrize("N,M,noqi,phi", [
    (2, 1, 1, 1e-3), (5, 2, 3, 1e-2), (6, 3, 32, 1e-2), (19, 4, 5, 2e-2), (20, 5, 7, 2e-2), (21, 5, 8, 1e-4),
    (41, 6, 4, 2e-2), (64, 7, 11, 1e-3), (33, 8, 21, 1e-2), (130, 5, 8, 2e-3), (290, 2, 4, 5e-3), (330, 1, 2, 2e-3)])
def test_rows_against_the_integrals(N, M, noqi, phi, precision):
    pos, ori = layout(N, phi, 700 + N)
    _check(pos, ori, M, noqi, precision, sorted({0, N // 2, N - 1}), 40)


@pytest.mark.parametrize("M,noqi,dmin", [(1, 8, 4.2), (4, 3, 4.2), (5, 8, 4.2), (5, 1, 4.2), (6, 8, 5.2), (8, 16, 5.2)])
def test_far_pairs(M, noqi, dmin):
    N = 48
    pos, ori = _shell(N, dmin + 1e-6, dmin + 2.0, 31 * M + noqi)
    _check(pos, ori, M, noqi, rf.PREC_FP64, [0], 1)


@pytest.mark.parametrize("M,noqi,N", [(1, 3, 23), (5, 8, 101), (6, 5, 47), (8, 4, 40)])
def test_velocity_operator(M, noqi, N):
    """W through the velocities of the solved system against the matrix-free
    sums (closed forms in both: 1e-11 to M = 5, beyond that their recurrences'
    own 6e-9 of a moment)."""
    pos, ori = layout(N, 1e-3, N)
    p = rf.default_params(use_analytical_integration=1, num_terms=M, num_quad_intervals=noqi, slenderness=EPS,
                          external_force=(0.2, -0.1, -1.0))
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        sim.solve_system()
        sim.update_velocities()
        v, w = sim.velocities()
        vo, wo = sim.operator(rf.OP_VELOCITY, sim.coefficients())
    tol = 1e-11 if M <= 5 else 1e-8
    assert np.abs(v - vo).max() <= tol * np.abs(vo).max()
    assert np.abs(w - wo).max() <= tol * max(np.abs(wo).max(), np.abs(vo).max())


@pytest.mark.parametrize("precision", [rf.PREC_FP64, rf.PREC_MIXED])
@pytest.mark.parametrize("N,M,noqi,phi", [
    (2, 1, 1, 1e-3), (5, 2, 3, 1e-2), (6, 3, 32, 1e-2), (19, 4, 5, 2e-2), (21, 5, 8, 1e-4), (41, 6, 4, 2e-2),
    (33, 8, 21, 1e-2), (64, 7, 11, 5e-2), (150, 5, 8, 5e-2)])
def test_numeric_against_the_oracle(N, M, noqi, phi, precision):
    """The same sums of the same products, so rounding alone: 1e-12 of the
    largest entry, as the parity tests; FP32 storage 6e-8 of an entry."""
    pos, ori = layout(N, phi, 50 + N)
    p = rf.default_params(use_analytical_integration=0, num_terms=M, num_quad_intervals=noqi, slenderness=EPS,
                          precision=precision, external_force=(0.2, -0.1, -1.0))
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        A, b = sim.matrix(), sim.rhs()
        pos, ori = (np.asarray(v).ravel() for v in sim.state()[:2])
    Ao = oracle.assemble_matrix(0, EPS, pos, ori, M, noqi)
    bo = oracle.assemble_rhs(0, EPS, pos, ori, np.tile([0.2, -0.1, -1.0], N), M, noqi)
    scale = np.abs(Ao - np.eye(Ao.shape[0])).max()
    err_b = np.abs(b - bo).max() / np.abs(bo).max()
    print("numeric N=%d M=%d NoQI=%d: A %.2e, b %.2e" % (N, M, noqi, np.abs(A - Ao).max() / scale, err_b))
    if precision == rf.PREC_MIXED:
        assert np.all(np.abs(A - Ao) <= 6e-8 * np.abs(Ao) + 1e-12 * scale)
    else:
        assert np.abs(A - Ao).max() <= 1e-12 * scale
    assert err_b <= 1e-12
