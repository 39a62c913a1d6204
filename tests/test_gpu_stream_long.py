"""The streaming GEMM where a wavefront walks several blocks of 16 columns (more than 65536 columns on 256 CUs), with a ragged last
block and wavefronts that end early: the MPO leg of 263 x 257 bonds (67591 columns), K of 6 and of 40, all types.
Tolerances: those of test_gpu_gemm_pipe.py."""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from dmrg_amd import _lib
from oracle import heff as O
from test_gpu_gemm_pipe import TOL32, TOL64, general, rel, single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("chiL,chiR,D", [(263, 257, 3), (263, 257, 20), (300, 331, 4)])
def test_several_blocks_per_wavefront(chiL, chiR, D, cplx):
    _lib.call("dmrg_gemm_plan_override", 6, 1)
    try:
        print(f"[case] chi={chiL}x{chiR} D={D} cplx={cplx}", file=sys.stderr, flush=True)
        th, W, L, R = general(np.random.default_rng(chiR + D), 2, chiL, chiR, D, D, cplx)
        ref = O.matrix_vector_product(th, W, L, R)
        assert rel(G.matrix_vector_product(th, W, L, R), ref) <= TOL64
        assert rel(G.matrix_vector_product(single(th), single(W), single(L), single(R)), ref) <= TOL32
    finally:
        _lib.call("dmrg_gemm_plan_override", -1, 0)
