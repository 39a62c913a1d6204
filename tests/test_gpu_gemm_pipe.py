"""The pipelined GEMM kernels at the sizes where they can go wrong: tile edges and remainders, K chunks shorter than,
equal to and just past a stage, operands whose 16-byte units run along K, along the other index or along neither, and
operands that are not 16-byte aligned. Checked against the oracle's contractions; tolerances are the matvec's (relative
2-norm): the products are summed in another order, with error bounds of a few hundred eps at these sizes."""
import ctypes as C
import sys

import numpy as np
import pytest

import dmrg_amd as G
from dmrg_amd import _lib
from oracle import heff as O

pytestmark = pytest.mark.gpu
TOL64, TOL32 = 1e-12, 1e-5


def general(rng, d, chiL, chiR, DL, DR, cplx):
    def t(*s):
        a = rng.standard_normal(s)
        return np.asfortranarray(a + 1j * rng.standard_normal(s) if cplx else a)

    return t(d, chiL, chiR), t(DL, DR, d, d), t(chiL, chiL, DL), t(chiR, chiR, DR)


def rel(a, b):
    return np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel())


def single(a):
    return a.astype(np.complex64 if np.iscomplexobj(a) else np.float32)


@pytest.fixture(params=[(0, 1), (0, 3), (2, 2), (4, 1), (5, 1), (5, 4)], ids=lambda p: f"cfg{p[0]}-ks{p[1]}")
def plan(request):
    _lib.call("dmrg_gemm_plan_override", *request.param)
    yield request.param
    _lib.call("dmrg_gemm_plan_override", -1, 0)


# d = 1, 2, 3: units along the physical index or none; bonds around 8, 16, 32, 64, 128 and odd; D = 1 (plain K) and more.
SHAPES = [(2, 1, 1, 1, 1), (1, 7, 9, 2, 3), (2, 8, 16, 3, 3), (3, 15, 17, 2, 4), (2, 16, 15, 5, 5), (2, 31, 33, 3, 5), (2, 64, 63, 5, 3),
          (2, 65, 66, 4, 4), (4, 32, 128, 2, 2), (2, 129, 36, 3, 3), (3, 34, 130, 2, 2)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matvec_and_env_at_tile_edges(shape, plan):
    rng = np.random.default_rng(sum(shape))
    for cplx in (False, True):
        th, W, L, R = general(rng, *shape, cplx)
        ref = O.matrix_vector_product(th, W, L, R)
        print(f"[case] {shape} {plan} cplx={cplx}", file=sys.stderr, flush=True)
        assert rel(G.matrix_vector_product(th, W, L, R), ref) <= TOL64
        assert rel(G.matrix_vector_product(single(th), single(W), single(L), single(R)), ref) <= TOL32
        for side, E in (("L", L), ("R", R)):
            ref = O.env_build_block(side, E, th, W)
            assert rel(G.env_build_block(side, E, th, W), ref) <= TOL64
            assert rel(G.env_build_block(side, single(E), single(th), single(W)), ref) <= TOL32


@pytest.mark.parametrize("dtype,off", [(np.float64, 8), (np.complex128, 8), (np.float32, 4), (np.float32, 8), (np.complex64, 8)])
def test_operands_off_16_byte_alignment(dtype, off):
    """Device pointers aligned to their element's parts only."""
    rng = np.random.default_rng(off)
    ts = [np.asfortranarray(t.astype(dtype)) for t in general(rng, 2, 48, 40, 4, 4, np.issubdtype(dtype, np.complexfloating))]
    ref = O.matrix_vector_product(*(t.astype(np.complex128) for t in ts))
    out = np.empty(ts[0].shape, dtype, order="F")
    bufs, ptrs = [], []
    for t in ts + [out]:
        p = C.c_void_p()
        _lib.call("dmrg_malloc", C.byref(p), t.nbytes + 16)
        bufs.append(p)
        ptrs.append(C.c_void_p(p.value + off))
    try:
        for t, p in zip(ts, ptrs):
            _lib.call("dmrg_memcpy_htod", p, t.ctypes.data_as(C.c_void_p), t.nbytes)
        th, W, L, R = ts
        dims = [(C.c_int64 * len(t.shape))(*t.shape) for t in ts]
        print(f"[case] offset {off} {dtype.__name__}", file=sys.stderr, flush=True)
        _lib.call("dmrg_matrix_vector_product", G.dtype_code(dtype), ptrs[4], ptrs[0], dims[0], ptrs[1], dims[1], ptrs[2], dims[2],
                  ptrs[3], dims[3], None)
        _lib.call("dmrg_memcpy_dtoh", out.ctypes.data_as(C.c_void_p), ptrs[4], out.nbytes)
    finally:
        for p in bufs:
            _lib.call("dmrg_free", p)
    assert rel(out, ref) <= (TOL64 if np.dtype(dtype).itemsize // (2 if np.issubdtype(dtype, np.complexfloating) else 1) == 8 else TOL32)


# The streaming kernel of the MPO leg (M = d D', K = d D): row blocks of 16 and K steps of 4 and their remainders, the
# largest sizes it takes (64) and the next ones, columns around one block and one workgroup (16, 64).
@pytest.mark.parametrize("d,DL,DR", [(1, 1, 1), (1, 2, 5), (2, 2, 8), (2, 6, 3), (3, 3, 5), (2, 8, 9), (4, 8, 8), (2, 16, 17), (2, 25, 25), (2, 32, 32),
                                     (2, 33, 32), (4, 16, 16)])
def test_streaming_leg_edges(d, DL, DR):
    _lib.call("dmrg_gemm_plan_override", 6, 1)
    try:
        rng = np.random.default_rng(d * 1000 + DL * 10 + DR)
        for chiL, chiR in ((1, 1), (3, 5), (4, 4), (17, 8), (9, 23)):
            for cplx in (False, True):
                print(f"[case] d={d} D={DL},{DR} chi={chiL}x{chiR} cplx={cplx}", file=sys.stderr, flush=True)
                th, W, L, R = general(rng, d, chiL, chiR, DL, DR, cplx)
                ref = O.matrix_vector_product(th, W, L, R)
                assert rel(G.matrix_vector_product(th, W, L, R), ref) <= TOL64
                assert rel(G.matrix_vector_product(single(th), single(W), single(L), single(R)), ref) <= TOL32
                for side, E in (("L", L), ("R", R)):
                    assert rel(G.env_build_block(side, E, th, W), O.env_build_block(side, E, th, W)) <= TOL64
    finally:
        _lib.call("dmrg_gemm_plan_override", -1, 0)
