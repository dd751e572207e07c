"""Host arrays in and out of the device planes: every value arrives (exactly
in FP64, rounded to float32 in mixed precision), at the sizes where the cut
into chunks and workers changes: one chunk, chunk ends inside an image and a
row, several workers, and the smallest grid."""
import numpy as np
import pytest

from conftest import small_string

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("N,F,two", [(2, 1, False), (65, 3, True), (128, 4, False), (131, 9, True),
                                     (257, 20, True), (300, 13, False)])
def test_round_trip(N, F, two, precision):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=F, multicomponent=two, seed=N)
    kept = (lambda v: v.astype(np.float32).astype(np.float64)) if precision == "mixed" else (lambda v: v)
    with Solver([s], precision=precision) as sv:
        a, p1, p2 = sv.download(0)
        assert np.array_equal(a, kept(s.a)) and np.array_equal(p1, kept(s.psi_1))
        assert np.array_equal(p2, kept(s.psi_2) if two else np.zeros_like(a))
        # The three solver buffers, each from its own values.
        for k, which in enumerate(("g", "g_old", "d")):
            f = [(k + 2.5) * v[::-1] for v in (s.a, s.psi_1)] + [(k + 2.5) * s.psi_2[::-1] if two else None]
            sv.upload_state(0, which, *f)
        for k, which in enumerate(("g", "g_old", "d")):
            got = sv.download_state(0, which)
            assert np.array_equal(got[0], kept((k + 2.5) * s.a[::-1]))
            assert np.array_equal(got[1], kept((k + 2.5) * s.psi_1[::-1]))
            if two:
                assert np.array_equal(got[2], kept((k + 2.5) * s.psi_2[::-1]))
        # The fields are untouched by them, and the other field buffer holds
        # the uploaded values as well.
        assert np.array_equal(sv.download(0)[0], kept(s.a))
