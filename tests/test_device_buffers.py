"""Buffer management of a context, on the CPU: context.cpp is linked with a
stand-in for the HIP runtime (host_device.cpp) that checks, at every launch,
that all a kernel can reach lies inside live allocations of the size that it
would read or write."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT, small_string

TESTS = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libmepgl_host.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-isystem", "/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                    "-Wl,-Bsymbolic", os.path.join(ROOT, "mepgl_amd", "csrc", "context.cpp"),
                    os.path.join(TESTS, "host_device.cpp"), "-o", so], check=True)
    return so


class Host:
    def __init__(self, lib):
        self.lib = lib
        lib.host_device_faults.restype = ctypes.c_char_p
        lib.host_device_bytes.restype = ctypes.c_longlong
        lib.host_device_clear()

    def faults(self):
        return sorted(set(self.lib.host_device_faults().decode().splitlines()))

    def bytes(self):
        return self.lib.host_device_bytes()


@pytest.fixture
def host(built, monkeypatch):
    from mepgl_amd import _lib

    monkeypatch.setattr(_lib, "LIB_PATH", built)
    monkeypatch.setattr(_lib, "_lib", None)
    return Host(_lib.load())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("planes", [False, True])
def test_resample_keeps_what_is_not_per_image(host, precision, planes):
    """Derived parameter planes and the cosine matrix of the local alignment
    stay with a string whose image count changes; the per-image buffers are
    its only new ones."""
    from mepgl_amd.solver import Solver

    before = host.bytes()
    strings = [small_string(N=24, F=5, seed=1, planes=planes),
               small_string(N=20, F=4, seed=2, multicomponent=True, planes=planes)]
    with Solver(strings, precision=precision, use_graph=False) as sv:
        counted, held = sv.info(0)["bytes"], host.bytes()
        for F in (9, 2, 5):
            sv.resample(0, F)
            sv.nlcgSteps(2)
            sv.loop(1, 2, "L")
            sv.computeFreeEnergy()
        assert host.faults() == []
        assert sv.info(0)["bytes"] == counted
        assert host.bytes() == held
        sv.gauge_align_local()
        counted, held = sv.info(0)["bytes"], host.bytes()
        sv.resample(0, 7)
        sv.resample(0, 5)
        sv.gauge_align_local()
        sv.redistributeCubic()
        sv.gradient(0)
        sv.computeJB(0)
        sv.gradient(1)
        assert host.faults() == []
        assert sv.info(0)["bytes"] >= counted
    assert host.bytes() == before


def solver_with_rows(strings, rows, **kw):
    """A Solver whose strings take their segment heights from a list."""
    from mepgl_amd.solver import Solver

    class Uneven(Solver):
        def _fill_desc(self, d, s, _):
            super()._fill_desc(d, s, rows[[t is s for t in strings].index(True)])

    return Uneven(strings, **kw)


def square(F, planes, N=64):
    return small_string(N=N, F=F, seed=F, planes=planes)


# Strings of equal N of which one starts with one row per item and the other's
# partial sums have room for heights from four on.
UNEVEN = {
    "planes": ([square(15, False), square(40, True)], [0, 0]),
    "planes first": ([square(8, True), square(60, False)], [0, 0]),
    "asked for": ([square(6, False), square(6, False)], [0, 4]),
    "asked for, first": ([square(6, False), square(6, False)], [7, 0]),
}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("strings,rows", UNEVEN.values(), ids=UNEVEN)
def test_tuned_heights_fit_the_partial_sums(host, strings, rows, precision):
    with solver_with_rows(strings, rows, precision=precision, use_graph=False) as sv:
        assert sorted(sv.info(i)["tile_rows"] == 1 for i in (0, 1)) == [False, True]
        tuned = sv.autotune(2)
        assert tuned == [sv.info(i)["tile_rows"] for i in (0, 1)]
        sv.loop(1, 3, "L")
        sv.computeFreeEnergy()
        assert host.faults() == []


def test_tuned_heights_after_a_resample(host):
    """One string's partial sums are made anew at four rows, beside one that
    still has one row."""
    from mepgl_amd.solver import Solver

    with Solver([square(6, False), square(5, False)], use_graph=False) as sv:
        assert [sv.info(i)["tile_rows"] for i in (0, 1)] == [1, 1]
        sv.set_segment_rows(1, 1)  # raised to four
        sv.resample(1, 8)
        sv.autotune(2)
        sv.nlcgSteps(2)
        assert host.faults() == []
