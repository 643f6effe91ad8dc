"""Row segments of the fused kernel's transfers and its compiled-in switches.

The fused kernel fetches a 64-node row segment 16 bytes a lane, several fields
to a transfer, and away from the x faces the whole phi tile as one run; lanes
past a short row fetch what follows it.  The sizes sit where that can go wrong:
rows shorter than a lane's 16 bytes, segments of 1, 2 and 3 nodes past a
multiple of 64, the first size with a tile free of x wrap (130) and its
neighbours, one row or plane beside a full row tile.  FP32 against the oracle
with the bars of test_gpu_parity; 16-bit storage against the FP64 run with the
bar of test_gpu_precision (stochastic rounding to 2^-11 of a velocity that the
noise of the start makes 1e-4: 3e-3 after a few steps).
"""
import numpy as np
import pytest

from lbfast_amd import hip
from lbfast_amd.params import PREC_FP32, PREC_FP64, PREC_FP16S, HFIELDS
from tests.cases import case, prepare, rel_l2
from tests.test_gpu_parity import run_pair

pytestmark = pytest.mark.gpu

SIZES = [(129, 5, 4), (130, 14, 3), (131, 13, 5), (195, 4, 6), (66, 27, 2), (65, 3, 9), (3, 16, 5)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("name", ["drop27h", "tg19", "tg27h"])
def test_rows_fp32(name, n):
    res, bad = run_pair(name, PREC_FP32, n, 4)
    assert not bad, bad


@pytest.mark.parametrize("n", [(129, 20, 16), (131, 18, 17), (66, 27, 16)])
@pytest.mark.parametrize("name", ["chan27h", "chan19", "chan27h_bb", "pois27h_1c"])
def test_rows_obstacles_fp32(name, n):
    res, bad = run_pair(name, PREC_FP32, n, 6)
    assert not bad, bad


@pytest.mark.parametrize("n", [(129, 12, 12), (131, 13, 12), (67, 15, 14), (13, 14, 12)])
def test_rows_fp16s(n):
    vel = {}
    for prec in (PREC_FP64, PREC_FP16S):
        p, f, _ = case("drop27h", n, prec)
        d = hip.Domain(p)
        d.load(f)
        d.step(8)
        vel[prec] = np.stack([d.download(k) for k in HFIELDS[1:4]])
        d.close()
    assert rel_l2(vel[PREC_FP16S], vel[PREC_FP64]) < 3e-3


@pytest.mark.parametrize("name", ["drop27h", "drop27h_smag", "drop27h_nodens", "tg27h", "tg27h_smag"])
def test_batch_switches(name):
    """A batch launches the domains of the compiled-in switches and the others
    apart: equal to each domain stepped alone, bit for bit.  The two kernels of
    the SMAGORINSKI switch are compiled apart, so that their products may be
    contracted differently: every moment is a sum of 27 populations of up to
    0.05 (the velocity's scale), so sixteen roundings of 2^-24 of that bound it."""
    sizes = [(40, 20, 24), (70, 14, 9)]
    loads = [(*case(nm, n, PREC_FP32)[:2],) for nm in (name, name.split("_")[0]) for n in sizes]
    doms = []
    for p, f in loads:
        d = hip.Domain(p)
        d.load(f)
        doms.append(d)
    b = hip.Batch(doms)
    b.step(3)
    b.synchronize()
    for d, (p, f) in zip(doms, loads):
        one = hip.Domain(p)
        one.load(f)
        one.step(3)
        for k in HFIELDS:
            got, want = d.download(k), one.download(k)
            if p.smagorinsky:
                np.testing.assert_allclose(got, want, rtol=0, atol=16 * 2.0 ** -24 * 0.05)
            else:
                np.testing.assert_array_equal(got, want)
        one.close()
    b.close()
    for d in doms:
        d.close()
