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
