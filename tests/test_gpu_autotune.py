"""The autotuner over strings of equal N whose partial sums have room for
different heights: a string that starts with one row per item, tuned beside
one that does not.  Tuning leaves the state as it was, and two steps at the
tuned heights agree with the oracle, FP64 to 1e-12 norm-wise per image, mixed
precision to 1e-5."""
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("uniform,planes", [(15, 40), (60, 8)])
def test_uniform_and_plane_string(uniform, planes, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    strings = [small_string(N=64, F=uniform, seed=1),
               small_string(N=64, F=planes, seed=2, planes=True)]
    with Solver(strings, precision=precision) as sv:
        assert sorted(sv.info(i)["tile_rows"] == 1 for i in (0, 1)) == [False, True]
        rows = sv.autotune(2)
        for i, r in enumerate(rows):
            assert r == sv.info(i)["tile_rows"]
            assert r >= 4 or (i == 0) == (uniform == 15)
        sv.nlcgSteps(2)
        for i, s in enumerate(strings):
            ref = oracle.OracleString(s)
            ref.nlcg_steps(2)
            a, p1, _ = sv.download(i)
            assert normwise(a, ref.a) < tol
            assert normwise(p1, ref.psi_1) < tol
