"""Grouped matvecs over the kernels that one leg's GEMMs can be split over: MPO legs of K and M up to 64 on the streaming
kernel beside larger ones on the pipelined tiles, by the size rule (tuning off) and by timing (tuning on), with extents at
and around the edges of the 16-, 32- and 64-wide tiles.

Tolerances: relative 2-norm error of the double-precision result <= 1e-12, of the single-precision one <= 1e-5 (sums of at
most a few hundred terms: eps sqrt(K) is 4e-15 and 2e-6).
"""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from dmrg_amd.workloads import random_heff_problem
from oracle import heff as O

pytestmark = pytest.mark.gpu

# (d, chi_l, chi_r, D_l, D_r): K of the MPO leg is d D_l, M is d D_r.
SETS = {
    "tiny": [(2, 1, 1, 2, 2), (1, 1, 3, 1, 1), (2, 2, 1, 3, 2)],
    "edges": [(2, 16, 32, 5, 5), (2, 17, 31, 5, 5), (2, 33, 15, 4, 8), (2, 65, 63, 3, 5)],
    "streamed_and_tiled": [(4, 24, 20, 17, 16), (4, 20, 24, 16, 16), (2, 30, 41, 5, 40), (2, 70, 9, 33, 3)],
    "one": [(3, 130, 129, 5, 5)],
}


@pytest.mark.parametrize("tuned", [0, 1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("name", list(SETS))
def test_group_kinds(name, fp32, cplx, tuned):
    print(f"[case] group {name} fp32={fp32} cplx={cplx} tuned={tuned}", file=sys.stderr, flush=True)
    dt = np.complex128 if cplx else np.float64
    vt = {(0, 0): np.float64, (0, 1): np.complex128, (1, 0): np.float32, (1, 1): np.complex64}[fp32, cplx]
    probs = []
    for i, (d, cl, cr, dl, dr) in enumerate(SETS[name]):
        th, W, L, R = random_heff_problem(d, cl, cr, dl, dr, seed=40 + i, complex_=cplx)
        probs.append((th.astype(dt), W.astype(dt), (L if cplx else L.real).astype(dt), (R if cplx else R.real).astype(dt)))
    G._lib.call("dmrg_autotune_enable", tuned)
    ops = [G.MatVecMPOS([W], L, R, dtype=dt) for th, W, L, R in probs]
    xs = [G.DeviceArray.from_numpy(th.astype(vt).reshape(-1, order="F")) for th, *_ in probs]
    ys = [G.DeviceArray((x.shape[0],), vt) for x in xs]
    try:
        grp = G.MatvecGroup(ops, xs, ys, fp32=fp32, graph=True)
        try:
            for _ in range(2):
                grp.run()
                G._lib.call("dmrg_synchronize")
                for (th, W, L, R), y in zip(probs, ys):
                    ref = O.matrix_vector_product(th, W, L, R).reshape(-1, order="F")
                    err = np.linalg.norm(y.to_numpy() - ref) / np.linalg.norm(ref)
                    assert err <= (1e-5 if fp32 else 1e-12), th.shape
                    y.zero()
        finally:
            grp.close()
    finally:
        G._lib.call("dmrg_autotune_enable", 1)
        for a in xs + ys:
            a.close()
        for op in ops:
            op.close()
