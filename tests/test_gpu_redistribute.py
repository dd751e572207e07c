"""The reparametrisation kernels against the oracle at the edges of their
tiles and batches: the spline kernel's image batches and its two paths (the
systems in LDS, and in memory for more than 96 images), the linear kernel's
groups of rows, the phase alignment's groups of rows.

Tolerances: FP64 1e-11 norm-wise per image for the spline system, 1e-12 for
the linear and phase kernels; mixed precision 1e-5 (float rounding of the
fields)."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


def compare(sv, ref, s, tol):
    a, p1, p2 = sv.download(0)
    assert normwise(a, ref.a) < tol
    assert normwise(p1, ref.psi_1) < tol
    if s.multicomponent:
        assert normwise(p2, ref.psi_2) < tol


def film_string(shared, **kw):
    s = small_string(multicomponent=True, no_self_field=True, **kw)
    if shared:
        s.a = np.broadcast_to(s.a[:1], s.a.shape).copy()
    return s


# F, N, rows: fewer images than a batch, whole batches and remainders in the
# forward sweep (F - 2 images), the back substitution (F - 1) and the new
# images (F); fewer (row, plane) pairs than images; both sides of the limit.
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 1e-5)])
@pytest.mark.parametrize("textbook", [False, True])
@pytest.mark.parametrize("F,N,rows", [(4, 65, 7), (5, 20, 1), (8, 24, 5), (9, 24, 5), (10, 24, 24),
                                      (13, 66, 4), (18, 20, 3), (64, 20, 19), (96, 16, 16),
                                      (97, 16, 16), (130, 12, 7)])
def test_cubic(F, N, rows, textbook, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=F, multicomponent=F % 2 == 0, seed=F)
    ref = oracle.OracleString(s, cubic_textbook=textbook)
    ref.arc_lengths()
    ref.redistribute(cubic=True)
    with Solver([s], precision=precision, segment_rows=rows, cubic_textbook=textbook) as sv:
        sv.arcLength()
        sv.redistributeCubic()
        compare(sv, ref, s, tol)


def test_cubic_strings_together(oracle):
    """One launch over strings of 4, 96 and 7 images, and one over strings of
    97 and 5, which go through memory."""
    from mepgl_amd.solver import Solver

    for counts in ((4, 96, 7), (97, 5)):
        strings = [small_string(N=20, F=F, seed=F) for F in counts]
        with Solver(strings, precision="fp64") as sv:
            sv.arcLength()
            sv.redistributeCubic()
            for i, s in enumerate(strings):
                ref = oracle.OracleString(s)
                ref.arc_lengths()
                ref.redistribute(cubic=True)
                a, p1, _ = sv.download(i)
                assert normwise(a, ref.a) < 1e-11
                assert normwise(p1, ref.psi_1) < 1e-11


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("film", ["", "shared", "own"])
@pytest.mark.parametrize("F,N,rows", [(2, 65, 1), (3, 20, 3), (5, 66, 4), (6, 64, 5), (7, 23, 19)])
def test_linear(F, N, rows, film, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    s = film_string(film == "shared", N=N, F=F, seed=F) if film else \
        small_string(N=N, F=F, multicomponent=F % 2 == 0, seed=F)
    ref = oracle.OracleString(s)
    ref.arc_lengths()
    ref.redistribute()
    with Solver([s], precision=precision, segment_rows=rows) as sv:
        sv.arcLength()
        sv.redistributeLinear()
        compare(sv, ref, s, tol)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("F,N,rows", [(2, 65, 1), (3, 20, 3), (6, 66, 4), (5, 64, 9), (4, 23, 19)])
def test_phase_alignment(F, N, rows, precision, tol, oracle):
    from mepgl_amd.solver import Solver

    s = small_string(N=N, F=F, multicomponent=F % 2 == 0, seed=F)
    ref = oracle.OracleString(s)
    ref.gauge_align()
    with Solver([s], precision=precision, segment_rows=rows) as sv:
        sv.gauge_align()
        compare(sv, ref, s, tol)
