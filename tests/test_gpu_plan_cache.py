"""More GEMM shapes on one thread than the plan cache holds (4096): first and later calls of shapes that were kept, given up and met
again give the same bits, and agree with the oracle to the matvec's tolerance (relative 2-norm 1e-12)."""
import sys

import numpy as np
import pytest

import dmrg_amd as G
from oracle import heff as O

pytestmark = pytest.mark.gpu


def test_more_shapes_than_the_cache_holds():
    rng = np.random.default_rng(5)
    shapes = [(a, b, D) for a in range(1, 31) for b in range(1, 31) for D in (1, 2)]  # three GEMMs each, 5400
    print(f"[case] {len(shapes)} shapes", file=sys.stderr, flush=True)
    flat = rng.standard_normal((4, 2 * 30 * 30 * 2))

    def tensors(a, b, D):
        dims = (2, a, b), (D, D, 2, 2), (a, a, D), (b, b, D)
        return [np.asfortranarray(flat[i, : int(np.prod(s))].reshape(s, order="F")) for i, s in enumerate(dims)]

    first = {s: G.matrix_vector_product(*tensors(*s)) for s in shapes}
    for s in shapes[::7] + shapes[:40] + shapes[-40:]:
        assert np.array_equal(G.matrix_vector_product(*tensors(*s)), first[s])
    for s in shapes[::151]:
        ref = O.matrix_vector_product(*tensors(*s))
        assert np.linalg.norm((first[s] - ref).ravel()) <= 1e-12 * np.linalg.norm(ref.ravel())
