"""Wick terms from segments at their edges: pixels in no order (segments of one pixel, more of
them in one bin than are sorted), one-pixel forests, one bin, a pair of a forest with itself.
Against the FP64 oracle, bars of test_gpu_wick."""
import numpy as np
import pytest

from oracle import cf_oracle as O
from picca_amd.engine import get_engine, params_from_globals
from picca_amd.store import ForestStore
from test_gpu_wick import _G, assert_close

pytestmark = pytest.mark.gpu


def forests(rng, lengths, shuffled):
    parts = []
    for n in lengths:
        r = 3800.0 + np.cumsum(rng.uniform(0.2, 1.0, n))
        parts.append(rng.permutation(r) if shuffled else r)
    r = np.concatenate(parts)
    off = np.concatenate([[0], np.cumsum(lengths)])
    n, m = len(r), len(lengths)
    return ForestStore(off, 2.0 + r / 1e4, r, r, rng.uniform(0.5, 2.0, n), rng.normal(size=n),
                       np.full(m, 3.0), np.linspace(0.01, 0.011, m), np.full(m, 0.01),
                       np.arange(m))


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("lengths,bins,r_max", [((130, 140), 1, 300.0), ((1, 2, 100), 1, 300.0),
                                                ((1, 2, 300), 7, 20.0),
                                                ((255, 256, 257, 65), 7, 20.0)])
def test_segments(lengths, shuffled, bins, r_max):
    rng = np.random.default_rng(len(lengths) + 10 * bins)
    store = forests(rng, lengths, shuffled)
    g = _G()
    g.num_bins_r_par = g.num_bins_r_trans = bins
    g.r_par_max = g.r_trans_max = r_max
    m = len(lengths)
    a, b = (x.ravel() for x in np.meshgrid(np.arange(m), np.arange(m), indexing="ij"))
    ang = rng.uniform(0.001, 0.01, len(a))
    off, mats = [0], []
    for k in range(m):
        n = lengths[k]
        q = rng.normal(size=(n, n))
        mats.append((0.01 * (q + q.T)).ravel())
        off.append(off[-1] + n * n)
    wx, wx_off = np.concatenate(mats), np.array(off[:-1], dtype=np.int64)
    zev1, zev2 = rng.uniform(0.5, 2.0, (2, store.num_pixels))
    eng = get_engine(0)
    eng.set_forests(store)
    mine = eng.wick_t123(params_from_globals(g), a, b, ang, zev1, zev2, wx_off, wx)
    nb = bins * bins
    ww, nw = np.zeros(nb), np.zeros(nb, dtype=np.int64)
    t = [np.zeros(nb * nb) for _ in range(3)]
    a32, b32 = a.astype(np.int32), b.astype(np.int32)
    params = O.params_from_module(g)
    O.lib().oracle_wick_t123(O.ctypes.byref(params), len(a), O._p(a32), O._p(b32), O._p(ang),
                             O._p(store.offsets), O._p(store.r_comov), O._p(store.weights),
                             O._p(zev1), O._p(zev2), O._p(wx_off), O._p(wx), O._p(ww), O._p(nw),
                             *[O._p(x) for x in t])
    assert nw.sum() > 0 and np.array_equal(mine[1], nw)
    n = nw.sum()
    assert_close(mine[0], ww, "weights_wick", rtol=1e-12)
    for k in range(3):
        assert_close(mine[2 + k], t[k].reshape(nb, nb), "t%d" % (k + 1))
    assert 0 < mine[5]["products"] <= n * (n - 1) // 2
