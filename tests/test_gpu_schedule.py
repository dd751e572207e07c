"""The schedule a context starts with: the segment heights picked for a
string's size and whether its image parts run as sequences of their own.

Heights only change how sums over cells are grouped: FP64 results of the
default height and of 7 rows agree to 1e-12 norm-wise after two outer
iterations.  Mixed precision amplifies its rounding from one
reparametrisation to the next (at 2^2 sites a relative change of 1e-7 in A
alone moves the fields by 5e-6 after two), so there two steps are compared
with the oracle, to 1e-5."""
import numpy as np
import pytest

from conftest import normwise, small_string

pytestmark = pytest.mark.gpu


CASES = [(2, 3, True), (5, 3, True), (40, 5, True), (64, 4, True), (65, 4, False), (96, 3, False)]


def case_string(N, F):
    return small_string(N=N, F=F, multicomponent=F == 5, masked=N == 64, seed=N)


@pytest.mark.parametrize("N,F,one_row", CASES)
@pytest.mark.parametrize("mode", ["L", "C"])
def test_default_height(N, F, one_row, mode):
    from mepgl_amd.solver import Solver

    s = case_string(N, F)
    if mode == "C" and F < 4:
        mode = "S"
    out = []
    for rows in (0, 7):
        with Solver([s], precision="fp64", segment_rows=rows) as sv:
            if not rows:
                assert (sv.info(0)["tile_rows"] == 1) == one_row
            sv.loop(2, 3, mode)
            out.append(sv.download(0)[:2] + (sv.computeFreeEnergy()[0],))
    for x, y in zip(*out):
        x, y = (np.asarray(v).reshape(F, -1) for v in (x, y))
        assert normwise(x, y) < 1e-12


@pytest.mark.parametrize("N,F,one_row", CASES)
def test_default_height_mixed(N, F, one_row, oracle):
    from mepgl_amd.solver import Solver

    s = case_string(N, F)
    ref = oracle.OracleString(s)
    ref.nlcg_steps(2)
    with Solver([s], precision="mixed") as sv:
        assert (sv.info(0)["tile_rows"] == 1) == one_row
        sv.nlcgSteps(2)
        a, p1, _ = sv.download(0)
    assert normwise(a, ref.a) < 1e-5
    assert normwise(p1, ref.psi_1) < 1e-5


def test_one_row_string_changes():
    """A string that starts at one row per item: resampled to more images
    while it does, and after another height was set."""
    from mepgl_amd.solver import Solver

    s = small_string(N=40, F=4, seed=3)
    out = []
    for rows in (None, 0, 7):
        with Solver([s], precision="fp64") as sv:
            sv.loop(1, 3, "L")
            if rows:
                sv.set_segment_rows(0, rows)
            if rows == 0:
                sv.set_segment_rows(0, 1)  # clamped to four
                assert sv.info(0)["tile_rows"] == 4
            sv.arcLength()
            sv.resample(0, 11)
            sv.loop(1, 3, "L")
            out.append(sv.download(0)[:2])
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert normwise(x, y) < 1e-12


def test_small_strings_keep_one_sequence():
    """Few row strips: one sequence unless parts are asked for; the same
    results bit for bit."""
    from mepgl_amd import _lib
    from mepgl_amd.solver import Solver

    s = small_string(N=40, F=6, seed=4)
    out = []
    for ask in (None, 1, 3, 0):
        with Solver([s], precision="fp64") as sv:
            assert sv.get_control(_lib.CONTROL_SPLIT_IMAGES) == 0
            if ask is not None:
                sv.set_control(_lib.CONTROL_SPLIT_IMAGES, ask)
                assert sv.get_control(_lib.CONTROL_SPLIT_IMAGES) == {1: 2}.get(ask, ask)
            sv.loop(2, 5, "L")
            out.append(sv.download(0)[:2])
    for other in out[1:]:
        for x, y in zip(out[0], other):
            np.testing.assert_array_equal(x, y)
