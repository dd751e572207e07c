"""The columns outside a strip in the step kernels: two NLCG steps against the
oracle where they come from memory, from the neighbouring strip's wavefront or
from the grid's edge: one to six strips, a last strip of one column or none
missing, domains with holes, the A of a film shared by the images or not.

Tolerances: FP64 1e-12 norm-wise per image, as for every single step; mixed
precision 1e-5 (float rounding of the fields)."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu

CASES = [(N, two, film) for N in (64, 65, 192, 257, 384) for two in (False, True)
         for film in ("", "shared", "own")]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("N,two,film", CASES)
def test_two_steps(N, two, film, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=2, multicomponent=two, masked=N % 2 == 1, seed=N,
                     no_self_field=bool(film))
    if film == "shared":
        s.a = np.broadcast_to(s.a[:1], s.a.shape).copy()
    ref = oracle.OracleString(s)
    ref.nlcg_steps(2)
    with Solver([s], precision=precision, segment_rows=7) as sv:
        sv.nlcgSteps(2)
        a, p1, p2 = sv.download(0)
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if two:
        assert normwise(p2, ref.psi_2) < tol
