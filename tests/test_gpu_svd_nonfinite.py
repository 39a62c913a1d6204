"""Jacobi SVD in one workgroup of matrices that hold a NaN: every value stands in S once, the NaN first, and the columns
without one (rows, for a wide matrix) are decomposed as if they stood alone, because a pair with a NaN is not rotated.

Tolerance: the singular values' of test_gpu_svd_resident.py, 1e-12 S[0].
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("bad", [[0], [2], [-1], [1, 3]], ids=str)
@pytest.mark.parametrize("m,n", [(4, 4), (32, 20), (100, 32), (64, 63), (20, 32), (60, 64)])
def test_nan_stays_in_the_singular_values(m, n, bad, cplx):
    print(f"[case] svd nan {m}x{n} {bad} cplx={cplx}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(m * n)
    A = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0)
    k = min(m, n)
    G.svd_truncate(np.asfortranarray(1e3 * A), 0.0, 0, 3)  # other values in the buffers that are kept between calls
    B = A.copy()
    for j in bad:
        if m < n:
            B[j, n // 2] = np.nan
        else:
            B[m // 2, j] = np.nan
    rest = np.linalg.svd(np.delete(A, bad, axis=0 if m < n else 1), compute_uv=False)
    r = G.svd_truncate(np.asfortranarray(B), 0.0, 0, 3)
    S = r["S"]
    assert len(S) == k
    assert np.all(np.isnan(S[:len(bad)]))
    assert np.max(np.abs(S[len(bad):] - rest)) <= 1e-12 * rest[0]
    assert np.isnan(r["U"]).any() == (m >= n) and np.isnan(r["Vt"]).any() == (m < n)
