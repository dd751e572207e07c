"""The cubic reparametrisation where the arclength does not rise: set from
outside (the new images' nodes are those of the reference's incremental search
also where it falls), and over coincident images.  FP64 1e-11 norm-wise per image, as for the spline system elsewhere
(these systems have a condition number below 70); mixed precision 1e-5 times
that over the condition number of evenly spaced images, 3: 2.5e-4."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


def falling(F):
    """Evenly spaced images, but for two in the first half that lie further
    along than the two after them."""
    s = np.linspace(0.0, 1.0, F)
    s[F // 3:F // 3 + 2] += 2.6 / (F - 1)
    return s


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 2.5e-4)])
@pytest.mark.parametrize("F", [8, 12, 50, 130])
def test_falling_arclength(F, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=20, F=F, multicomponent=F % 4 == 0, seed=F)
    ref = oracle.OracleString(s)
    ref.s_jb = falling(F)
    ref.redistribute(cubic=True)
    with Solver([s], precision=precision) as sv:
        sv.set_scalars(0, "s_jb", falling(F))
        sv.redistributeCubic()
        a, p1, p2 = sv.download(0)
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if s.multicomponent:
        assert normwise(p2, ref.psi_2) < tol


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("first", [0, 3, 6])
def test_coincident_images(first, precision):
    """Two equal neighbours have no spline: every value is NaN, in LDS and,
    beside a string of 97 images, through memory."""
    from mepgl_amd.solver import Solver

    s = small_string(N=12, F=8, seed=5)
    for f in (s.a, s.psi_1):
        f[first + 1] = f[first]
    for others in ([], [small_string(N=12, F=97, seed=6)]):
        with Solver([s] + others, precision=precision) as sv:
            sv.arcLength()
            sv.redistributeCubic()
            a, p1, _ = sv.download(0)
            assert np.isnan(a).all() and np.isnan(p1).all()
            for i in range(len(others)):
                a, p1, _ = sv.download(1 + i)
                assert np.isfinite(a).all() and np.isfinite(p1).all()
