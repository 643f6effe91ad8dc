"""What a domain lays out from an uploaded isfluid (the wetting list, the fused
kernel's node words): a second upload replaces the first, down to no solid node."""
import numpy as np
import pytest

from lbfast_amd import hip
from lbfast_amd.params import PREC_FP32, PREC_FP64
from tests.cases import case, prepare, state_of

pytestmark = pytest.mark.gpu


def _run(d, f, isf):
    d.load(f, isf)
    d.step(3)
    st = state_of(d, d.p)
    return np.concatenate([st["h"].ravel(), st["phi"].ravel(), st["phiO"].ravel()])


@pytest.mark.parametrize("prec", [PREC_FP32, PREC_FP64])
def test_second_upload_replaces_the_first(prec):
    n = (40, 20, 24)
    starts = []
    for seed in (1, 2, None):
        p, f, raw = case("chan27h", n, prec, seed=seed or 1)
        if seed is None:  # no solid node at all: every axis periodic
            raw = np.ones((n[2], n[1], n[0]), dtype=np.int8)
            isf = raw
        else:
            f, isf = prepare(p, f, raw, hip.classify_isfluid)
        starts.append((f, isf))
    d = hip.Domain(p)
    for f, isf in starts + starts[:1]:
        fresh = hip.Domain(p)
        want = _run(fresh, f, isf)
        fresh.close()
        np.testing.assert_array_equal(_run(d, f, isf), want)
    d.close()
