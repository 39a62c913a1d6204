"""The eigensolver's expansion step on both sides of the line between one workgroup and several launches within one solve (n m =
40960 basis elements): the same pair as from a basis that stays below it, residual and norm as in test_gpu_expand_step.py."""
import pytest

from test_gpu_expand_step import solve

pytestmark = pytest.mark.gpu


# n = 2 chiL chiR; the line: 10, 10.01, 20, 20.02 and 39.996 columns.
@pytest.mark.parametrize("chiL,chiR,ncv,cplx", [(64, 32, 14, False), (31, 66, 14, False), (32, 32, 24, False), (32, 32, 24, True), (33, 31, 24, True),
                                                (16, 32, 32, True)])
def test_columns_across_the_line(chiL, chiR, ncv, cplx):
    e = solve(chiL, chiR, cplx, ncv=ncv)
    assert abs(solve(chiL, chiR, cplx, ncv=8) - e) <= 1e-9 * max(1.0, abs(e))
