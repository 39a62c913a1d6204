"""The eigensolver's expansion step at its dispatch lines: one workgroup with the vector in LDS (32 KiB of it, 32 columns),
three launches up to 2^17 rows (folds in the last workgroup up to 128 of them, one or two rows a thread), and the separate
launches beyond; with the residual and with a preconditioned one, which makes the second Gram-Schmidt pass run.

Tolerances: the solver's own (residual norm tol * max(1, |H|)) with a factor of ten for the norm estimate, unit norm to 1e-12.
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from test_gpu_block_vectors import diagonal_operator

pytestmark = pytest.mark.gpu


def solve(chiL, chiR, cplx, seed=7, **kw):
    W, L, R = diagonal_operator(chiL, chiR, cplx, seed)
    op = G.MatVecMPOS([W], L, R, dtype=np.complex128 if cplx else np.float64)
    print(f"[case] n={2 * chiL * chiR} cplx={cplx} {kw}", file=sys.stderr, flush=True)
    try:
        w, v, info = op.eigs(tol=1e-10, **kw)
        v = v[:, 0] if v.ndim == 2 else v
        assert info["nconv"] == 1
        assert abs(np.linalg.norm(v) - 1) <= 1e-12
        assert np.linalg.norm(op.MultAx(v) - w[0] * v) <= 1e-9 * max(1.0, info["anorm"])
    finally:
        op.close()
    return w[0]


# n: 2, 6, 2046, 2048, 2050, 4096, 4098, 8192, 8198, 32768, 33024, 65536, 66048.
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("chiL,chiR", [(1, 1), (3, 1), (33, 31), (32, 32), (41, 25), (64, 32), (683, 3), (64, 64), (4099, 1), (128, 128),
                                       (129, 128), (256, 128), (129, 256)])
def test_sizes(chiL, chiR, cplx):
    e = solve(chiL, chiR, cplx)
    assert abs(solve(chiL, chiR, cplx, mixed=True) - e) <= 1e-9 * max(1.0, abs(e))


@pytest.mark.parametrize("chiL,chiR", [(20, 20), (64, 64), (200, 200)])
@pytest.mark.parametrize("ncv", [31, 32, 33, 34, 60])
def test_columns(chiL, chiR, ncv):
    solve(chiL, chiR, False, ncv=ncv, target="SA")


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("chiL,chiR", [(24, 20), (64, 64), (150, 150)])
def test_preconditioned(chiL, chiR, cplx):
    e = solve(chiL, chiR, cplx)
    assert abs(solve(chiL, chiR, cplx, precond=1) - e) <= 1e-9 * max(1.0, abs(e))
