"""One-sided Jacobi SVD at the edges of its single-workgroup kernel (up to 128 x 64, 16 lanes per column pair, 2 to 8 elements
per lane) and just beyond it, with exact zeros and equal singular values, against LAPACK.

Tolerances: singular values <= 1e-12 S[0], U and Vt orthonormal and the product back to A to 1e-12 sqrt(k) and 1e-12 S[0]
(a rotation errs by a few eps; a column meets at most a few thousand of them, whose errors do not add up coherently).
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G

pytestmark = pytest.mark.gpu

SIZES = [(3, 2), (17, 15), (32, 32), (33, 33), (64, 63), (65, 64), (64, 128), (128, 64), (33, 128), (129, 32), (32, 129), (129, 64)]


def check(A, scale):
    S_ref = np.linalg.svd(A, compute_uv=False)
    r = G.svd_truncate(np.asfortranarray(A), 0.0, int(np.sum(S_ref > 1e-14 * S_ref[0])), 3)
    S, k, U, Vt = r["S"], r["rank"], r["U"], r["Vt"]
    assert np.all(np.diff(S) <= 0)
    assert np.max(np.abs(S - S_ref)) <= 1e-12 * scale
    assert np.linalg.norm(U.conj().T @ U - np.eye(k)) <= 1e-12 * np.sqrt(k)
    assert np.linalg.norm(Vt @ Vt.conj().T - np.eye(k)) <= 1e-12 * np.sqrt(k)
    assert np.linalg.norm(A - (U * S[:k]) @ Vt) <= 1e-12 * scale * np.sqrt(k)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("m,n", SIZES)
def test_svd_resident_edges(m, n, cplx):
    print(f"[case] svd {m}x{n} cplx={cplx}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(100 * m + n)
    A = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0)
    check(A, np.linalg.norm(A, 2))
    check(1e-130 * A, 1e-130 * np.linalg.norm(A, 2))
    k = min(m, n)
    u, _, vt = np.linalg.svd(A, full_matrices=False)
    s = np.repeat(np.exp(-np.arange((k + 1) // 2)), 2)[:k]  # pairs of equal values
    check((u * s) @ vt, 1.0)
    Z = A.copy()
    Z[:, ::3] = 0  # columns of zeros
    Z[m // 2:, :] = 0
    check(Z, np.linalg.norm(Z, 2))
