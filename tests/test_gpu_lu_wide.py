"""The LU at sizes where its wide trailing update and its edges are in play
(rf_selftest_lu), against LAPACK getrf."""
import numpy as np
import pytest
import scipy.linalg as sl

import rigidfibers_kth_amd as rf
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
