"""The LU at sizes where its wide trailing update and its edges are in play
(rf_selftest_lu), against LAPACK getrf."""
import numpy as np
import pytest
import scipy.linalg as sl

import rigidfibers_kth_amd as rf
from rigidfibers_kth_amd.layouts import layout
from test_gpu_lu import _dominant_with_block_swaps, _random

pytestmark = pytest.mark.gpu


# trailing matrices of 14 to 17 tiles of 128 rows, whole and ragged, odd n
# (the last row pair reaches the padding), super-panels of 512 and of 480
# columns (48-column panels), and of 495 (45: no whole K chunks, the narrow
# kernel throughout)
@pytest.mark.parametrize("n,nb", [(2304, 0), (2305, 0), (2433, 0), (2560, 48), (2401, 45)])
def test_fp64_wide_update_matches_lapack(n, nb):
    A = _dominant_with_block_swaps(n, nb if nb else 64, n)
    lu_ref, piv_ref = sl.lu_factor(A)
    LU, ipiv, info, fb = rf.selftest_lu(A, 8, nb)
    assert info == 0 and fb == 0
    np.testing.assert_array_equal(ipiv, piv_ref)
    assert np.abs(LU - lu_ref).max() <= 1e-12 * np.abs(lu_ref).max()


def test_fp64_wide_update_on_a_matrix_that_pivots_everywhere():
    n = 2311
    A = _random(n, 23)
    lu_ref, piv_ref = sl.lu_factor(A)
    LU, ipiv, info, fb = rf.selftest_lu(A, 8, 0)
    assert info == 0 and fb == (n - 1) // 64
    np.testing.assert_array_equal(ipiv, piv_ref)
    # growth and conditioning of a random matrix: n eps times the factors' size, with room for both
    assert np.abs(LU - lu_ref).max() <= 1e-10 * np.abs(lu_ref).max()


@pytest.mark.parametrize("N,terms,mixed", [(10, 5, 0), (34, 5, 0), (35, 5, 1), (69, 5, 1), (103, 5, 0), (53, 7, 1),
                                           (171, 3, 0), (177, 4, 1)])
def test_fp32_factor_solve_at_block_edges(N, terms, mixed):
    """(LU)^-1 r with FP32 factors against numpy, for systems below, at and
    just past multiples of the 512-row diagonal blocks and the 64-row blocks
    they are merged from; FP32 factors of a well-conditioned system."""
    pos, ori = layout(N, 1e-2, 4000 + N)
    p = rf.default_params(num_terms=terms, precond=rf.PRECOND_LU, lu_factor_fp32=1, precision=mixed, gmres_tol=1e-10,
                          gmres_restart=30, gmres_max_iters=300)
    with rf.Simulation(rf.Configuration(p, pos, ori)) as sim:
        sim.assemble_system()
        sim.solve_system()
        assert sim.stats().last_backward_error <= 1e-10
        A = sim.matrix()
        r = np.random.default_rng(N).normal(size=sim.n)
        z = sim.precond_apply(r)
        again = sim.precond_apply(r)
    ref = np.linalg.solve(A, r)
    assert np.array_equal(z, again)
    assert np.linalg.norm(z - ref) <= 1e-5 * np.linalg.norm(ref)


# With more than 1024 columns beyond the next super-panel (512 columns in FP64,
# 1024 in FP32) their update runs on the side stream beside the factorisation
# of that super-panel: 2048 + 512, FP32 from 3072 + 1024 on, with whole and ragged ends, panels
# redone column by column in between, and the fp16 update's tiles.
@pytest.mark.parametrize("n,es,fp16", [(2049, 8, 0), (3100, 8, 0), (3073, 4, 0), (4300, 4, 0), (4611, 4, 1),
                                       (6200, 4, 1)])
def test_overlapped_updates_give_partial_pivoting(n, es, fp16):
    A = _dominant_with_block_swaps(n, 64, n + 1)
    if es == 4:
        A = A.astype(np.float32).astype(np.float64)
    lu_ref, piv_ref = sl.lu_factor(A)
    LU, ipiv, info, fb = rf.selftest_lu(A, es, 0, update_fp16=fp16)
    again, _, _, _ = rf.selftest_lu(A, es, 0, update_fp16=fp16)
    assert info == 0 and fb == 0
    np.testing.assert_array_equal(ipiv, piv_ref)
    np.testing.assert_array_equal(LU, again)
    # FP64 and FP32 rounding of sums over n of a diagonally dominant matrix; fp16 operands
    tol = 1e-12 if es == 8 else (2e-3 if fp16 else 1e-5)
    assert np.abs(LU - lu_ref).max() <= tol * np.abs(lu_ref).max()


def test_overlapped_updates_with_redone_panels():
    n = 3200
    A = _random(n, 29)
    lu_ref, piv_ref = sl.lu_factor(A)
    LU, ipiv, info, fb = rf.selftest_lu(A, 8, 0)
    assert info == 0 and fb == (n - 1) // 64
    np.testing.assert_array_equal(ipiv, piv_ref)
    assert np.abs(LU - lu_ref).max() <= 1e-10 * np.abs(lu_ref).max()
