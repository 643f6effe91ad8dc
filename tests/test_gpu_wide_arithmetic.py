"""The fast path in 64-bit arithmetic (FP64, MIXED) on its default tiles: the
prefetching fused kernel in 5-row blocks, whose x-halo nodes come as two dwords to
a value and whose completed plane is stored an iteration later; the streaming prep
with 64-bit rows (dwords where the row length is odd); D3Q19 in 13 rows.  The sizes
sit where the transfers can go wrong: segments a few nodes past a multiple of 64,
odd rows, domains thinner than a row tile.  Bars as in test_gpu_parity."""
import numpy as np
import pytest

from lbfast_amd import hip
from lbfast_amd.params import FIELD_PHI, HFIELDS, PREC_FP32, PREC_FP64, PREC_MIXED
from tests.cases import case, prepare
from tests.test_gpu_parity import run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("n", [(65, 7, 5), (131, 13, 5), (67, 6, 3), (3, 16, 5), (130, 11, 4)])
@pytest.mark.parametrize("name", ["drop27h", "drop19", "tg27h", "tg19"])
def test_rows(name, n, prec):
    res, bad = run_pair(name, prec, n, 4)
    assert not bad, bad


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("n", [(131, 18, 17), (67, 21, 16)])
@pytest.mark.parametrize("name", ["chan27h", "chan27h_bb", "pois27h_1c"])
def test_rows_obstacles(name, n, prec):
    res, bad = run_pair(name, prec, n, 6)
    assert not bad, bad


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("n", [(70, 27, 9), (131, 14, 5)])
def test_d3q19_thirteen_rows(n, prec):
    res, bad = run_pair("tg19", prec, n, 4, tile=(13, 4))
    assert not bad, bad


def _state(d):
    return np.stack([d.download(k) for k in HFIELDS + ((FIELD_PHI,) if d.p.twocomponent else ())])


@pytest.mark.parametrize("name", ["drop27h", "drop27h_smag", "tg27h"])
def test_mixed_batch_equals_single_domains(name):
    loads = [case(name, n, PREC_MIXED)[:2] for n in ((32, 32, 32), (48, 40, 36), (67, 24, 20), (21, 28, 44))]
    doms = []
    for p, f in loads:
        d = hip.Domain(p)
        d.load(f)
        doms.append(d)
    b = hip.Batch(doms)
    b.step(3)
    b.step(4)
    b.synchronize()
    for d, (p, f) in zip(doms, loads):
        one = hip.Domain(p)
        one.load(f)
        one.step(7)
        np.testing.assert_array_equal(_state(d), _state(one))
        one.close()
    b.close()
    for d in doms:
        d.close()


@pytest.mark.parametrize("name,prec,rows,copies", [
    ("drop27h", PREC_FP64, 5, 5), ("chan27h", PREC_FP64, 5, 5), ("tg27h", PREC_FP64, 5, 7),
    ("drop27h", PREC_MIXED, 5, 10), ("drop27h", PREC_FP32, 13, 10), ("chan27h", PREC_FP32, 13, 10)])
def test_streaming_stores_of_the_default_rows(name, prec, rows, copies):
    """As test_gpu_stream_stores, with the rows that a default takes: `copies`
    periods in z have more than 256 MB of state (80 bytes a node with one component,
    112 with two, twice that in FP64) and store past the cache, one does not; the
    values are the same bit for bit."""
    n = (128, 128, 16)
    p, f, raw = case(name, n, prec)
    f, isf = prepare(p, f, raw, hip.classify_isfluid)
    out = []
    for c in (1, copies):
        q = type(p).from_buffer_copy(p)
        q.nz = c * n[2]
        d = hip.Domain(q)
        d.set_tile(rows, 16)
        d.load({k: np.concatenate([v] * c) for k, v in f.items()}, None if isf is None else np.concatenate([isf] * c))
        d.step(3)
        out.append(_state(d)[:, :, 1:-1])
        d.close()
    assert np.isfinite(out[0]).all()
    for part in np.split(out[1], copies, axis=1):
        assert np.array_equal(part, out[0])
