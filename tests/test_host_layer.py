"""The C-ABI layer's host logic without a GPU: lbf_api.cpp compiled over a HIP
runtime and kernels that do nothing (tests/host/host_stub.cpp)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from lbfast_amd import build, hip
from lbfast_amd.params import make_params, PREC_FP32

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libstub.so")
    subprocess.run([build.HIPCC, *build.FLAGS, "-O1", "-w", "--offload-host-only", "-shared", "-nogpulib",
                    "-no-hip-rt", "-Wl,-Bsymbolic", "-x", "hip", os.path.join(ROOT, "tests", "host", "host_stub.cpp"), "-o", out], check=True)
    return out


@pytest.fixture
def stub(stub_path, monkeypatch):
    monkeypatch.setattr(hip, "_lib", None)
    yield hip.load(stub_path)


def _wetting(L):
    out = (ctypes.c_long * 3)()
    L.stub_wetting(out)
    return list(out)


def test_failed_upload_of_isfluid_changes_nothing(stub):
    """The wetting list's allocation is the only one of an upload: where it fails
    the domain keeps the isfluid, the words and the list that it had."""
    n = (20, 12, 9)
    p = make_params(n, lattice=27, twocomponent=True, densratio=True, internal_obstacles=True, precision=PREC_FP32)
    a = np.ones(n[::-1], dtype=np.int8)
    b = a.copy()
    a[3:5, 4:6, 5:9] = 0
    b[2:7, 2:9, 3:15] = 0
    d = hip.Domain(p)
    d.upload_isfluid(a)
    d.init_state()
    d.step(1)
    had = _wetting(stub)
    assert had[0] == had[2] == 2 * 2 * 4
    stub.stub_fail_after(0)
    with pytest.raises(hip.LbfError):
        d.upload_isfluid(b)
    stub.stub_fail_after(-1)
    d.step(1)
    assert _wetting(stub) == had
    d.upload_isfluid(b)
    d.step(1)
    assert _wetting(stub)[0] == _wetting(stub)[2] == 5 * 7 * 12
    d.upload_isfluid(np.ones_like(a))
    d.step(1)
    assert _wetting(stub)[0] == _wetting(stub)[2] == 0
    d.close()
