"""The step kernels' derived parameter planes: two NLCG steps and the loop
against the oracle with one, some or all parameters and the applied field as
planes; strips of one and of two columns, one and two components, films.

Tolerances: FP64 1e-12 norm-wise per image, as for every single step; mixed
precision 1e-5 (float rounding of the fields)."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu

ALL = ("a_1", "b_1", "m_xx_1", "m_yy_1", "a_2", "b_2", "m_xx_2", "m_yy_2", "h")


def plane_string(N, two, film, names):
    s = small_string(N=N, F=2, multicomponent=two, masked=N % 2 == 1, seed=N, no_self_field=film)
    rng = np.random.default_rng(N)
    for name in names:
        if name.endswith("_2") and not two:
            continue
        v = getattr(s, name)
        setattr(s, name, v + 0.1 * rng.random((N, N)))
    return s.validate()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("names", [("h",), ("a_1",), ("b_2", "m_yy_1"), ALL],
                         ids=["h", "a", "some", "all"])
@pytest.mark.parametrize("N,two,film", [(2, False, False), (65, True, False), (66, False, False),
                                        (130, True, True), (192, True, False)])
def test_two_steps(N, two, film, names, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    if names == ("b_2", "m_yy_1") and not two:
        names = ("b_1", "m_yy_1")
    s = plane_string(N, two, film, names)
    ref = oracle.OracleString(s)
    ref.nlcg_steps(2)
    with Solver([s], precision=precision, segment_rows=7) as sv:
        sv.nlcgSteps(2)
        a, p1, p2 = sv.download(0)
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if two:
        assert normwise(p2, ref.psi_2) < tol


def test_resampled_string(oracle):
    """The planes stay with a string whose image count changes."""
    from mepgl_amd.solver import Solver

    s = plane_string(40, True, False, ALL)
    out = []
    for grow in (False, True):
        with Solver([s], precision="fp64") as sv:
            if grow:
                sv.arcLength()
                sv.resample(0, 3)
                sv.arcLength()
                sv.resample(0, 2)
                sv.upload(0, s)
                sv.reset_solver()
            sv.nlcgSteps(2)
            out.append(sv.download(0))
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
