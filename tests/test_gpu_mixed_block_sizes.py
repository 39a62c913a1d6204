"""Optimally mixed block at the line between the one-workgroup Gram-Schmidt (128 KiB a vector) and the separate launches, and
where H1 psi is parallel to psi (its column of the block is at the rounding level), against the block's own definition:
alpha combines an orthonormal basis of {psi, H1 psi, H2 psi}, so the result has the norm of alpha and lies in their span.

Tolerance: 1e-11 relative (three projections of vectors of condition up to about 1e3, 1e-16 each, with room for 2^13 terms).
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from dmrg_amd.workloads import random_heff_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("d,chiL,chiR", [(2, 1, 1), (2, 5, 7), (4, 64, 32), (4, 64, 63), (4, 64, 64), (4, 65, 64), (4, 96, 70)])
def test_sizes(d, chiL, chiR, cplx):
    print(f"[case] d={d} chi={chiL}x{chiR} cplx={cplx}", file=sys.stderr, flush=True)
    dt = np.complex128 if cplx else np.float64
    ops = []
    for seed, D in ((1, 3), (2, 4)):
        th, W, L, R = random_heff_problem(d, chiL, chiR, D, D, seed=seed, complex_=cplx)
        ops.append(G.MatVecMPOS([W], L if cplx else L.real, R if cplx else R.real, dtype=dt))
    psi = th.astype(dt).reshape(-1, order="F")
    psi /= np.linalg.norm(psi)
    x, alpha, _ = G.optimally_mixed_block(ops[0], ops[1], psi, 3)
    x = np.asarray(x).reshape(-1, order="F")
    span = np.stack([psi, ops[0].MultAx(psi), ops[1].MultAx(psi)], axis=1)
    c, *_ = np.linalg.lstsq(span, x, rcond=None)
    if psi.size >= 3:  # two components hold no three orthonormal vectors
        assert abs(np.linalg.norm(x) - np.linalg.norm(alpha)) <= 1e-11
    assert np.linalg.norm(span @ c - x) <= 1e-11
    for op in ops:
        op.close()
