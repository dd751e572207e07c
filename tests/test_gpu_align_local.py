"""The local gauge alignment against the oracle at the edges of its products'
tiles (32 and 64 outputs, 16 steps of k), its groups of four rows and its
batches of eight images.

FP64 1e-11 norm-wise per image.  Mixed precision: the potential differences
carry float rounding of A, a bond's gradient of the phase no more than that,
and the phase itself at most the sum over a path of N bonds and F images:
2^-24 max|A| N dx F, on top of the fields' own rounding, 1e-6."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("N,F,rows", [(2, 2, 4), (5, 3, 4), (16, 9, 5), (17, 10, 7), (31, 3, 4),
                                      (32, 17, 16), (33, 4, 9), (48, 3, 48), (64, 3, 13),
                                      (65, 4, 4), (96, 2, 19), (128, 3, 16), (130, 2, 7)])
def test_local_alignment(N, F, rows, precision, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=F, multicomponent=F % 2 == 0, seed=N + F)
    ref = oracle.OracleString(s)
    ref.gauge_align_local()
    tol = 1e-11
    if precision == "mixed":
        tol = 1e-6 + 2.0 ** -24 * np.max(np.abs(s.a)) * N * s.dx * F
    with Solver([s], precision=precision, segment_rows=rows) as sv:
        sv.gauge_align_local()
        a, p1, p2 = sv.download(0)
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if s.multicomponent:
        assert normwise(p2, ref.psi_2) < tol
