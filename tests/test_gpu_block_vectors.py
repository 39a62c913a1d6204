"""Eigensolver block-vector kernels at sizes around their dispatch lines: one row, one and several row blocks, the switch
between short and long reductions (2^17 rows) and between folds in the last workgroup and in a launch of their own. A
solve on an operator with known spectrum exercises projection, update, Ritz and correction kernels together; its residual
is checked on the host in 64 bits, with the solver's own tolerance."""
import sys

import numpy as np
import pytest

import dmrg_amd as G

pytestmark = pytest.mark.gpu


def diagonal_operator(chiL, chiR, cplx, seed):
    """H = 1 (x) (A + B) with diagonal A on the left and B on the right bond plus a small Hermitian left block: d = 2,
    D = 2 MPO that adds the two environments."""
    rng = np.random.default_rng(seed)
    W = np.zeros((2, 2, 2, 2), order="F")
    W[0, 0] = W[1, 1] = np.eye(2)
    W[0, 1] = np.diag([0.0, 0.5])
    L = np.zeros((chiL, chiL, 2), complex)
    R = np.zeros((chiR, chiR, 2), complex)
    A = rng.standard_normal((chiL, chiL)) + (1j * rng.standard_normal((chiL, chiL)) if cplx else 0)
    L[:, :, 1] = np.diag(np.linspace(0.0, 4.0, chiL)) + 0.01 * (A + A.conj().T) / np.sqrt(chiL)
    L[:, :, 0] = np.eye(chiL)
    R[:, :, 1] = np.eye(chiR)
    R[:, :, 0] = np.diag(np.linspace(0.0, 5.0, chiR))
    return W, L, R


# n = 2 chiL chiR: 8, 254, 258, 1022, 8192, 2^17 - 1024, 2^17, 2^17 + 512.
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("chiL,chiR", [(2, 2), (127, 1), (129, 1), (73, 7), (64, 64), (256, 254), (256, 256), (256, 257)])
def test_solve_residual(chiL, chiR, cplx):
    W, L, R = diagonal_operator(chiL, chiR, cplx, chiL + chiR)
    op = G.MatVecMPOS([W], L, R, dtype=np.complex128 if cplx else np.float64)
    n = 2 * chiL * chiR
    for mixed in (False, True):
        print(f"[case] n={n} cplx={cplx} mixed={mixed}", file=sys.stderr, flush=True)
        w, v, info = op.eigs(tol=1e-10, mixed=mixed)
        v = v[:, 0] if v.ndim == 2 else v
        r = op.MultAx(v) - w[0] * v
        assert info["nconv"] == 1
        assert abs(np.linalg.norm(v) - 1) <= 1e-12
        assert np.linalg.norm(r) <= 1e-9 * max(1.0, info["anorm"])  # ten times the solver's tolerance
    op.close()


@pytest.mark.parametrize("ncv", [4, 15, 16, 17, 33, 40, 64])
def test_basis_sizes(ncv):
    """Basis sizes around the column groups (4, 16) and the number of Ritz coefficients passed with the launch (32)."""
    W, L, R = diagonal_operator(48, 40, False, 3)
    op = G.MatVecMPOS([W], L, R, dtype=np.float64)
    print(f"[case] ncv={ncv}", file=sys.stderr, flush=True)
    w, v, info = op.eigs(tol=1e-11, ncv=ncv)
    assert info["nconv"] == 1
    v = v[:, 0] if v.ndim == 2 else v
    assert np.linalg.norm(op.MultAx(v) - w[0] * v) <= 1e-10 * max(1.0, info["anorm"])
    op.close()
