"""Bins and bin edges along a forest of the banded distortion matrix (dmat_band.h), on the CPU
against the reference's arithmetic (py/picca/cf.py:656-700) pixel by pixel: equal keys, and each
edge the first pixel of its key, on exact bin edges, gaps, repeated steps and single pixels."""
import numpy as np
import pytest

import walk_harness as H

GRIDS = {
    "lattice": 3800.0 + 1.0 * np.arange(400),
    "lattice_off": 3800.0 + 1e-10 + 0.5 * np.arange(300),
    "smooth": 3700.0 + np.cumsum(np.linspace(0.6, 0.4, 1500)),
    "gaps": np.concatenate([3700.0 + 0.3 * np.arange(50), 4100.0 + 0.3 * np.arange(50)]),
    "uneven": 3700.0 + np.cumsum(np.random.default_rng(1).uniform(0.01, 3.0, 257)),
    "two": np.array([3800.0, 3800.4]),
    "one": np.array([3812.0]),
}


@pytest.mark.parametrize("bins,span", [(50, 200.0), (100, 200.0), (15, 60.0), (1, 7.0)])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_r_par(grid, bins, span):
    v = GRIDS[grid]
    for own in (v[0], v[len(v) // 2] + 0.25, v[-1], v[0] - 300.0, v[-1] + 150.0, 3850.0):
        for scale in (1.0, 0.9998):
            margin = 1e-12 + 20 * 2.0 ** -53 * (5000.0 * bins / span + bins)
            rps = (own - v) * scale
            row = np.minimum(np.floor(np.abs(rps) / span * bins), bins)
            ref = np.where(rps > 0, -row - 1, row).astype(int)
            keys, edges = H.dmat_band(H.BAND_PAR, v, own, scale, span, bins, margin, -bins, 2 * bins + 1)
            assert np.array_equal(keys, ref)
            assert np.array_equal(edges, np.searchsorted(ref, np.arange(-bins, bins + 1)))


@pytest.mark.parametrize("bins,span", [(50, 200.0), (12, 60.0), (1, 30.0)])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_r_trans(grid, bins, span):
    v = GRIDS[grid]
    for own in (3700.0, 3912.3):
        for scale in (0.001, 0.004, 0.02):
            margin = 1e-12 + 20 * 2.0 ** -53 * (9000.0 * scale * bins / span + bins)
            ref = np.minimum(np.floor((own + v) * scale / span * bins), bins).astype(int)
            keys, edges = H.dmat_band(H.BAND_TRANS, v, own, scale, span, bins, margin, 0, bins + 1)
            assert np.array_equal(keys, ref)
            assert np.array_equal(edges, np.searchsorted(ref, np.arange(bins + 1)))


@pytest.mark.parametrize("bins,lo,hi", [(100, -200.0, 200.0), (30, -60.0, 60.0), (7, -11.0, 3.0)])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_signed_r_par(grid, bins, lo, hi):
    v, span = GRIDS[grid], hi - lo
    for own in (v[0], v[len(v) // 2] + 0.25, v[-1], v[0] - 300.0, v[-1] + 150.0, 3850.0):
        for scale in (1.0, 0.9998):
            margin = 1e-12 + 20 * 2.0 ** -53 * (5000.0 * bins / span + 2 * bins)
            t = np.floor(((v - own) * scale - lo) / span * bins)
            ref = np.minimum(np.maximum(t, -1), bins).astype(int)
            keys, edges = H.dmat_band(H.BAND_SIGNED, v, own, scale, span, bins, margin, 0,
                                      bins + 1, lo)
            assert np.array_equal(np.maximum(keys, -1), ref)
            assert np.array_equal(edges, np.searchsorted(ref, np.arange(bins + 1)))


def test_no_pair_of_an_auto_correlation_rounds_past_the_end():
    """r_trans, and |r_par| from 0, below the range's end have a bin below the number of bins:
    x <= pred(end) gives x / end <= 1 - 2^-53 after rounding, and (1 - 2^-53) n rounds to n minus
    one spacing.  At the end the bin is n.  (A signed r_par counts from r_par_min: there the
    difference to r_par_min may round to the whole range, and the pair is handed back.)"""
    rng = np.random.default_rng(0)
    ends = np.concatenate([2.0 ** np.arange(-2, 10), rng.uniform(0.1, 1000, 4000),
                           np.nextafter(2.0 ** np.arange(-2, 10), 0)])
    for n in (1, 2, 3, 7, 32, 33, 50, 63, 64, 65, 100, 127, 128, 4095, 8192, 100003):
        below = np.nextafter(ends, 0)
        assert np.all(np.floor(below / ends * n) == n - 1)
        assert np.all(np.floor(ends / ends * n) == n)
    for end in ends[:200]:
        for kind in (H.BAND_TRANS, H.BAND_PAR):
            v = np.array([np.nextafter(end, 0), end])   # own coordinate 0, scale 1
            keys, _ = H.dmat_band(kind, v, 0.0, 1.0, end, 50, 1e-9, 0, 1)
            assert list(keys) == [49, 50]
