"""Host logic of the C-ABI runtime (oa_capi.cpp) on the CPU: compiled with g++ against stand-ins
for the HIP runtime and the kernel launchers (tests/cpp/capi_stub.cpp), which fail allocations on
request and check every launch's buffers."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from opticks_amd import _lib as L
from opticks_amd import configs
from opticks_amd.qsim import QSim, SEventConfig

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "opticks_amd", "csrc")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("no g++ or no HIP headers")
    out = tmp_path_factory.mktemp("stub") / "libcapi_stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I/opt/rocm/include", os.path.join(CSRC, "oa_capi.cpp"),
                    os.path.join(ROOT, "tests", "cpp", "capi_stub.cpp"), "-Wl,-Bsymbolic", "-o", str(out)], check=True)
    return str(out)


@pytest.fixture
def stub(built, monkeypatch):
    monkeypatch.setattr(L, "LIBPATH", built)
    monkeypatch.setattr(L, "_lib", None)
    lib = L.lib()
    lib.stub_limit.argtypes = [L.C.c_size_t]
    lib.stub_largest.restype = L.C.c_size_t
    lib.stub_reset()
    yield lib
    assert lib.stub_bad() == 0


def event(n):
    return configs.config0(num_photon=n).gensteps


def sim_of(**kw):
    w = configs.config0(num_photon=1)
    return QSim(w.geometry, w.physics, SEventConfig(seed=1, **kw))


def test_outputs_follow_the_handles_mask(stub):
    """simulate() gives the arrays that the handle was configured for, also where the caller's
    config object changed since, or the handle was configured by set_config_c."""
    sim = sim_of()
    sim.config.output_mask = L.MI_OUT_HIT                      # changed, not applied
    assert len(sim.simulate(event(100))) == 50
    assert sim.photon.shape == (100, 4, 4) and sim.seq.shape == (100, 2, 2)
    assert np.array_equal(sim.photon[:, 0, 0], np.arange(100)) and np.array_equal(sim.seq[:, 0, 0], np.arange(100))
    sim.config.output_mask = L.MI_OUT_PHOTON | L.MI_OUT_SEQ | L.MI_OUT_HIT
    c = sim.get_config_c()
    c.output_mask = L.MI_OUT_HIT
    sim.set_config_c(c)
    assert np.array_equal(sim.simulate(event(100))[:, 0, 0], np.arange(1, 100, 2))
    assert sim.photon is None and sim.seq is None
    sim.config.output_mask = L.MI_OUT_PHOTON
    assert sim.simulate(event(100)) is None
    sim.close()
