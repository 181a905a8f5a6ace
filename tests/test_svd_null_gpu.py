"""One-sided Jacobi SVD (the LDS and global-memory kernels) of square and
nearly square blocks with null singular values: the missing directions have
to be completed although no unit vector comes near them.

Tolerance: backward stability and the pair test's cosines, both within
4 max(m, n) eps."""
import numpy as np
import pytest

from test_svd_eig_gpu import check_orthonormal, with_null_values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,null", [(2, 2, 1), (12, 12, 1), (13, 13, 1), (14, 15, 1), (15, 15, 1), (15, 15, 2),
                                      (23, 23, 1), (23, 22, 1), (21, 22, 2), (23, 23, 2), (19, 20, 1), (24, 24, 1),
                                      (31, 31, 2), (30, 31, 1), (24, 24, 20), (40, 40, 9), (400, 30, 1), (200, 200, 9),
                                      (193, 193, 30)])
def test_null_columns_are_completed(m, n, null):
    """LDS kernel up to 15 columns and with more than eight null ones,
    global-memory kernel from 193 rows; the eigenvector path for the others."""
    check_orthonormal(with_null_values(m, n, null), "D")

