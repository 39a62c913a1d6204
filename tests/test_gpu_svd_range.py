"""Jacobi SVD of matrices whose columns' squared norms are in range but whose products are not (norms of about 1e130 and
1e-130), in each of its paths: one workgroup for everything, LDS-resident columns, one launch per round, block pairs.

Tolerances: those of test_gpu_svd_resident.py.
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from test_gpu_svd_resident import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("scale", [1e130, 1e-130])
@pytest.mark.parametrize("m,n", [(9, 7), (32, 32), (80, 32), (81, 31), (128, 20), (64, 64), (32, 128), (200, 24), (700, 32), (32, 700), (129, 64), (140, 140)])
def test_scaled_far_from_one(m, n, scale, cplx):
    print(f"[case] svd {m}x{n} scale={scale} cplx={cplx}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(10 * m + n)
    A = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0)
    check(scale * A, scale * np.linalg.norm(A, 2))
    k = min(m, n)
    u, _, vt = np.linalg.svd(A, full_matrices=False)
    check(scale * ((u * np.exp(-np.arange(k) / 2)) @ vt), scale)  # graded, as Schmidt values are
