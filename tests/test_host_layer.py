"""The C-ABI layer's host logic without a GPU: lbf_api.cpp compiled over a HIP
runtime and kernels that do nothing (tests/host/host_stub.cpp)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from lbfast_amd import build, hip
from lbfast_amd.params import make_params, PREC_FP32, PREC_FP64, PREC_MIXED

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


@pytest.mark.parametrize("n,prec,lattice,rows", [
    # one component in 64-bit arithmetic: the rows that were the fastest of 5, 8 and
    # 13, each with its best chunk (D3Q27 has 13 rows spill)
    ((176, 268, 32), PREC_FP64, 19, 13), ((50, 275, 85), PREC_FP64, 19, 13), ((100, 100, 100), PREC_FP64, 19, 5),
    ((192, 192, 192), PREC_FP64, 19, 5), ((64, 64, 64), PREC_FP64, 19, 8), ((36, 295, 114), PREC_FP64, 27, 8),
    ((150, 97, 75), PREC_FP64, 27, 5), ((176, 268, 32), PREC_MIXED, 19, 13), ((64, 64, 64), PREC_MIXED, 19, 8),
    ((192, 192, 192), PREC_MIXED, 19, 13), ((192, 192, 192), PREC_FP64, 27, 5), ((176, 268, 32), PREC_MIXED, 27, 8),
    ((335, 50, 237), PREC_MIXED, 27, 5)])
def test_rows_of_64_bit_domains(stub, n, prec, lattice, rows):
    p = make_params(n, lattice=lattice, highorder=lattice == 27, precision=prec)
    d = hip.Domain(p)
    d.init_state()
    d.step(1)
    ty, tz = ctypes.c_int(), ctypes.c_int()
    stub.stub_fused_tile(ctypes.byref(ty), ctypes.byref(tz))
    assert ty.value == rows
    d.close()


@pytest.mark.parametrize("prec,obstacles,n,fit", [
    # (measured 258 -> 250, 193 -> 188, 84.5 -> 82.8 and 72.8 -> 71.3 us a step)
    (PREC_FP64, 1, (131, 233, 48), 1), (PREC_FP64, 1, (171, 114, 67), 1), (PREC_MIXED, 0, (94, 245, 34), 2),
    (PREC_MIXED, 0, (58, 91, 169), 2), (PREC_FP64, 0, (94, 245, 34), 2), (PREC_FP32, 0, (94, 245, 34), 3)])
def test_prep_blocks_fit_one_round(stub, prec, obstacles, n, fit):
    """A domain small enough for it has the phase prep's blocks on the 256 CUs all at
    once: registers and LDS leave `fit` of them on each."""
    p = make_params(n, lattice=27, twocomponent=True, densratio=True, internal_obstacles=obstacles, precision=prec)
    d = hip.Domain(p)
    d.init_state()
    d.step(1)
    tiles = -(-n[0] // 64) * -(-n[1] // 12)
    assert tiles * -(-n[2] // stub.stub_prep_chunk()) <= 256 * fit
    d.close()


@pytest.mark.parametrize("n,prec,lattice,before", [
    # the tile before, and in turn with two others of its size: us a step with chunks
    # of 8 planes at least, with it, and now
    ((30, 49, 295), PREC_FP64, 19, (5, 12)),    # 26.7, 30.8
    ((39, 275, 37), PREC_FP64, 19, (5, 10)),    # 20.3, 24.0, 20.3
    ((156, 77, 56), PREC_FP64, 19, (8, 7)),     # 33.3, 36.0, 32.2
    ((37, 50, 228), PREC_FP32, 19, (13, 4)),    # 15.2, 15.9
    ((62, 325, 45), PREC_FP32, 27, (8, 8))])    # 22.7, 23.4
def test_chunks_leave_room_for_domains_in_turn(stub, n, prec, lattice, before):
    p = make_params(n, lattice=lattice, highorder=lattice == 27, precision=prec)
    d = hip.Domain(p)
    d.init_state()
    d.step(1)
    ty, tz = ctypes.c_int(), ctypes.c_int()
    stub.stub_fused_tile(ctypes.byref(ty), ctypes.byref(tz))

    # all planes that the blocks march, halo planes included, by the time of each
    plane = {8: 0.72, 13: 1.0} if prec == PREC_FP32 else {5: 0.64, 8: 1.0, 13: 1.4}

    def marched(rows, z):
        return -(-n[0] // 64) * -(-n[1] // rows) * -(-n[2] // z) * plane[rows] * (z + (4 if rows == 5 else 3))
    assert marched(ty.value, tz.value) < marched(*before)
    d.close()
