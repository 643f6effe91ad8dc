"""The row tiles that a caller may choose: 8 or 13, and 5 with 64-bit arithmetic,
whose default it is.  What lbf_batch_autotune and lbf_batch_tiles report,
lbf_batch_set_tile takes; the tile changes only which block computes a node, so
that results stay equal bit for bit."""
import numpy as np
import pytest

from lbfast_amd import hip
from lbfast_amd.params import FIELD_PHI, HFIELDS, PREC_FP32, PREC_FP64, PREC_MIXED
from tests.cases import case

pytestmark = pytest.mark.gpu

SIZES = [(40, 20, 24), (70, 14, 9)]


def _state(d):
    return np.stack([d.download(k) for k in HFIELDS + ((FIELD_PHI,) if d.p.twocomponent else ())])


def _load(name, prec):
    out = []
    for n in SIZES:
        p, f, _ = case(name, n, prec)
        d = hip.Domain(p)
        d.load(f)
        out.append(d)
    return out


@pytest.mark.parametrize("name,prec", [("drop27h", PREC_MIXED), ("tg27h", PREC_MIXED), ("tg19", PREC_FP64)])
def test_batch_takes_what_it_reports(name, prec):
    want = _load(name, prec)
    for d in want:
        d.step(6)
    doms = _load(name, prec)
    b = hip.Batch(doms)
    pair = b.autotune(2)
    assert pair[0] == b.tiles()[0]
    b.set_tile(*pair)
    b.step(2)
    for ty in (5, 13):
        b.set_tile(ty, 16)
        assert b.tiles()[0] == ty
        b.step(2)
    b.synchronize()
    for d, w in zip(doms, want):
        np.testing.assert_array_equal(_state(d), _state(w))
    b.close()
    for d in doms + want:
        d.close()


@pytest.mark.parametrize("name,prec", [("drop27h", PREC_FP64), ("drop27h", PREC_MIXED), ("tg27h", PREC_FP64)])
def test_domain_takes_five_rows(name, prec):
    a, b = _load(name, prec)[1], _load(name, prec)[1]
    a.set_tile(5, 4)
    a.step(3)
    b.step(3)
    np.testing.assert_array_equal(_state(a), _state(b))
    a.close()
    b.close()


def test_five_rows_stay_refused_in_32_bits():
    doms = _load("tg27h", PREC_FP32)
    b = hip.Batch(doms)
    for obj in (doms[0], b):
        for ty in (5, 7):
            with pytest.raises(hip.LbfError):
                obj.set_tile(ty, 8)
    b.close()
    for d in doms:
        d.close()
