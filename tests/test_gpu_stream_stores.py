"""Streaming stores of a state larger than the memory-side cache.

A domain of z-periodic content with period 16 and more than 256 MB of state
(read and written: 80 bytes a node with one component, 112 with two, 224 in
FP64) stores past the cache; the domain of one period does not.  The values are
the same, bit for bit, in every period.  (Next to a wall in y nothing defines
the moments of the wall's own layer.)
"""
import numpy as np
import pytest

from lbfast_amd import hip
from lbfast_amd.params import FIELD_PHI, HFIELDS, PREC_FP32, PREC_FP64
from tests.cases import case, prepare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,prec,copies", [("tg27h", PREC_FP32, 14), ("drop27h", PREC_FP32, 10),
                                              ("drop27h", PREC_FP64, 5), ("chan27h", PREC_FP32, 10)])
def test_same_values(name, prec, copies):
    n = (128, 128, 16)
    p, f, raw = case(name, n, prec)
    f, isf = prepare(p, f, raw, hip.classify_isfluid)
    out = []
    for c in (1, copies):
        q = type(p).from_buffer_copy(p)
        q.nz = c * n[2]
        d = hip.Domain(q)
        d.set_tile(8, 16)
        d.load({k: np.concatenate([v] * c) for k, v in f.items()}, None if isf is None else np.concatenate([isf] * c))
        d.step(3)
        out.append([d.download(k)[:, 1:-1] for k in HFIELDS + ((FIELD_PHI,) if "phi" in f else ())])
        d.close()
    for one, many in zip(*out):
        assert one.shape == (n[2], n[1] - 2, n[0]) and np.isfinite(one).all()
        for part in np.split(many, copies):
            assert np.array_equal(part, one)
