"""What lies outside the sample does not enter the energies: a mass plane that
is zero there, and a vector potential that is not finite outside both domains.
No bond and no plaquette of the sample holds such a site, so the energies
equal, bit for bit, those with ordinary values there; the entry point on
device arrays gives the same bits."""
import numpy as np
import pytest

from conftest import small_string
from test_zz_no_alloc import ROWS, context_energy, noalloc_energy

pytestmark = pytest.mark.gpu


def sample(N, two, film):
    """A masked sample with mass planes, finite everywhere; its sites."""
    s = small_string(N=N, F=3, seed=N, multicomponent=two, masked=True, no_self_field=film)
    rng = np.random.default_rng(N)
    for name in ("m_xx_1", "m_yy_1") + (("m_xx_2", "m_yy_2") if two else ()):
        setattr(s, name, getattr(s, name) + 0.1 * rng.random((N, N)))
    return s, s.sc_domain != 0


def masses_zero(s, inside):
    t = s.copy()
    for name in ("m_xx_1", "m_yy_1", "m_xx_2", "m_yy_2"):
        if not np.isscalar(getattr(t, name)):
            setattr(t, name, np.where(inside, getattr(t, name), 0.0))
    return t


def potential_not_finite(s, inside):
    t = s.copy()
    t.a = t.a.copy()
    out = np.argwhere(~inside)
    for k, (j, i) in enumerate(out):
        t.a[:, j, i] = (np.nan, np.inf, -np.inf)[k % 3]
    return t


CASES = [(24, False, False), (66, True, False), (65, True, True)]


@pytest.mark.parametrize("change", [masses_zero, potential_not_finite])
@pytest.mark.parametrize("N,two,film", CASES)
def test_energies(N, two, film, change):
    from mepgl_amd.solver import Solver

    s, inside = sample(N, two, film)
    t = change(s, inside)
    for precision in ("fp64", "mixed"):
        out = []
        for x in (s, t):
            with Solver([x], precision=precision) as sv:
                out.append(sv.computeFreeEnergy()[0])
        assert np.isfinite(out[0]).all()
        np.testing.assert_array_equal(out[1], out[0])


@pytest.mark.parametrize("change", [masses_zero, potential_not_finite])
@pytest.mark.parametrize("N,two,film", CASES)
def test_energies_on_device_arrays(N, two, film, change):
    s, inside = sample(N, two, film)
    t = change(s, inside)
    rc, e = noalloc_energy(t, ROWS)
    assert rc == 0
    np.testing.assert_array_equal(e, context_energy(s, ROWS))
    np.testing.assert_array_equal(e, context_energy(t, ROWS))
