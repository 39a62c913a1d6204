"""NaN and infinity in an operand of the pipelined and streaming kernels stay in the rows or columns of the result that they belong
to, at tile edges and under padding too: one column of an environment reaches one column of the matvec, the rest equals the result
without it (relative 2-norm 1e-12, FP32 1e-5: the matvec's tolerances)."""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from dmrg_amd import _lib
from test_gpu_gemm_pipe import TOL32, TOL64, general, rel, single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("plan", [(-1, 0), (0, 1), (2, 3), (5, 1), (6, 1)], ids=str)
@pytest.mark.parametrize("d,chiL,chiR,D", [(2, 5, 3, 3), (2, 33, 31, 5), (3, 65, 17, 4), (2, 64, 64, 16)])
def test_confined_to_its_column(d, chiL, chiR, D, plan, cplx):
    print(f"[case] d={d} {chiL}x{chiR} D={D} {plan} cplx={cplx}", file=sys.stderr, flush=True)
    th, W, L, R = general(np.random.default_rng(chiL + D), d, chiL, chiR, D, D, cplx)
    _lib.call("dmrg_gemm_plan_override", *plan)
    try:
        for conv, tol in ((lambda a: a, TOL64), (single, TOL32)):
            clean = G.matrix_vector_product(*(conv(x) for x in (th, W, L, R)))
            for bad in (np.nan, np.inf):
                for a in (0, chiL - 1):
                    Lb = L.copy(order="F")
                    Lb[chiL // 2, a, D - 1] = bad
                    out = G.matrix_vector_product(*(conv(x) for x in (th, W, Lb, R)))
                    assert not np.isfinite(out[:, a, :]).any()
                    assert rel(np.delete(out, a, 1), np.delete(clean, a, 1)) <= tol
                for b in (0, chiR - 1):
                    Rb = R.copy(order="F")
                    Rb[chiR // 2, b, 0] = bad
                    out = G.matrix_vector_product(*(conv(x) for x in (th, W, L, Rb)))
                    assert not np.isfinite(out[:, :, b]).any()
                    assert rel(np.delete(out, b, 2), np.delete(clean, b, 2)) <= tol
    finally:
        _lib.call("dmrg_gemm_plan_override", -1, 0)
