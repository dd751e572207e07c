"""A string stepped and aligned at a new image count, against the oracle on
the resampled fields: what does not depend on the image count (parameter
planes and what is derived of them, the local alignment's cosine matrix)
stays in use.

Tolerances: FP64 1e-12 norm-wise per image for two steps, 1e-11 for the
local alignment; mixed precision 1e-5 for two steps (float rounding of the
fields), and for the alignment the bound of a path of N bonds and F images,
2^-24 max|A| N dx F, on top of the fields' own rounding, 1e-6."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


def plane_string(N, two, film, seed):
    s = small_string(N=N, F=3, multicomponent=two, masked=True, seed=seed, no_self_field=film)
    rng = np.random.default_rng(seed)
    for name in ("a_1", "b_1", "m_xx_1", "m_yy_1", "h") + \
            (("a_2", "b_2", "m_xx_2", "m_yy_2") if two else ()):
        setattr(s, name, getattr(s, name) + 0.1 * rng.random((N, N)))
    return s.validate()


def resident(sv, i, s):
    """String i as it is on the device."""
    t = s.copy()
    t.F = sv.F[i]
    t.a, t.psi_1, p2 = sv.download(i)
    t.psi_2 = p2 if s.multicomponent else None
    return t


def compare(got, ref, two, tol):
    a, p1, p2 = got
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if two:
        assert normwise(p2, ref.psi_2) < tol


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("N,two,film", [(200, True, False), (130, False, False), (66, True, True)])
def test_steps_at_the_new_count(N, two, film, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    strings = [plane_string(N, two, film, N), plane_string(40, not film, film, 7)]
    with Solver(strings, precision=precision) as sv:
        sv.nlcgSteps(1)
        for F in (5, 2):
            nbytes = sv.info(0)["bytes"]
            sv.resample(0, F)
            sv.resample(0, sv.F[0])
            assert (sv.info(0)["bytes"] > nbytes) == (F == 5)
            sv.reset_solver()
            refs = [oracle.OracleString(resident(sv, i, s)) for i, s in enumerate(strings)]
            sv.nlcgSteps(2)
            for i, (s, ref) in enumerate(zip(strings, refs)):
                ref.nlcg_steps(2)
                compare(sv.download(i), ref, s.multicomponent, tol)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("N", [65, 160])
def test_local_alignment_at_the_new_count(N, precision, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=4, multicomponent=True, seed=N)
    rng = np.random.default_rng(N)
    with Solver([s], precision=precision) as sv:
        sv.gauge_align_local()
        sv.resample(0, 7)
        t = resident(sv, 0, s)
        t.a = t.a + 0.05 * rng.standard_normal(t.a.shape)
        if precision == "mixed":
            t.a = t.a.astype(np.float32).astype(np.float64)
        sv.upload(0, t)
        ref = oracle.OracleString(t)
        ref.gauge_align_local()
        sv.gauge_align_local()
        tol = 1e-11 if precision == "fp64" else \
            1e-6 + 2.0 ** -24 * np.max(np.abs(t.a)) * N * s.dx * 7
        compare(sv.download(0), ref, True, tol)
