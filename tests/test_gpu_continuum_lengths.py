"""The continuum fit at the pixel counts where the number of waves of a forest changes (640 pixels
a wave, up to 8 waves, then the kernel that reads its pixels at every evaluation): one batch of
all lengths against the FP64 oracle, masked pixels and variance terms of the general form."""
import numpy as np
import pytest

from oracle import cont_oracle as C
from picca_amd import continuum

pytestmark = pytest.mark.gpu

LENGTHS = (2, 63, 64, 65, 639, 640, 641, 1280, 1281, 2560, 2561, 5120, 5121)


def make_inputs(seed):
    rng = np.random.default_rng(seed)
    parts = []
    for n in LENGTHS:
        ll = np.linspace(3.56, 3.6, n)
        x = np.linspace(0.0, 1.0, n)
        mean = 1.0 + 0.1 * np.sin(7 * x)
        ivar = rng.uniform(1.0, 30.0, n)
        if n > 2:
            ivar[rng.random(n) < 0.1] = 0.0
        flux = (1.5 + 0.4 * x) * mean * rng.uniform(0.5, 1.0, n) + rng.normal(0, 0.2, n)
        parts.append(dict(log_lambda=ll, flux=flux, ivar=ivar, mean_cont=mean, x=x,
                          eta=1.0 + 0.1 * x, var_lss=0.05 + 0.02 * x,
                          fudge=np.full(n, 1e-3), log_lambda_min=ll[0], log_lambda_max=ll[-1]))
    inputs = {k: np.concatenate([p[k] for p in parts]) for k in
              ("flux", "ivar", "mean_cont", "x", "eta", "var_lss", "fudge")}
    inputs["offsets"] = np.concatenate([[0], np.cumsum(LENGTHS)])
    return inputs, parts


@pytest.mark.parametrize("constant", [False, True])
def test_lengths(constant):
    inputs, parts = make_inputs(5)
    res = continuum.fit_arrays(inputs, order=1, use_constant_weight=constant)
    assert np.all(res["status"] == 0)
    for k, spec in enumerate(parts):
        assert res["ndata"][k] == (spec["ivar"] > 0).sum()
        if constant:
            a, b = C.ols(spec, order=1)
            chi = C.chi2(a, b, spec, True)
            # two pixels are fitted exactly: chi2 is the rounding of their fluxes
            assert res["chi2"][k] == pytest.approx(chi, rel=1e-9, abs=1e-28)
        else:
            a, b, chi, _, _ = C.fit(spec, order=1)
            assert res["chi2"][k] == pytest.approx(chi, rel=1e-9)
        # (a, b) are known to the square root of the stopping rule's 1e-12
        assert res["a"][k] == pytest.approx(a, rel=1e-5)
        assert abs(res["b"][k] - b) <= 1e-5 * abs(a)


def test_order_0():
    inputs, parts = make_inputs(6)
    res = continuum.fit_arrays(inputs, order=0)
    assert np.all(res["status"] == 0) and not res["b"].any()
    for k, spec in enumerate(parts):
        a, _, chi, _, _ = C.fit(spec, order=0)
        assert res["ndata"][k] == (spec["ivar"] > 0).sum()
        assert res["chi2"][k] == pytest.approx(chi, rel=1e-9)
        assert res["a"][k] == pytest.approx(a, rel=1e-5)


@pytest.mark.parametrize("constant", [False, True])
def test_validity_of_every_wave(constant):
    """The checks of the final continuum see each pixel, whichever wave holds it, masked ones too:
    negative in the last or the first pixel alone (status 2), zero but for the last or the first
    pixel (valid), zero everywhere (3)."""
    inputs, parts = make_inputs(7)
    specs, want, orders = [], [], []
    for p in parts:
        n = len(p["flux"])
        if n < 63:
            continue
        for kind, status in (("negative_last", 2), ("negative_first", 2), ("last", 0),
                             ("first", 0), ("none", 3)):
            q = {k: p[k].copy() for k in ("flux", "ivar", "mean_cont", "x", "eta", "var_lss",
                                          "fudge")}
            pixel = n - 1 if "last" in kind else 0
            if "negative" in kind:
                q["mean_cont"][pixel] *= -1
                q["ivar"][pixel] = 0.0
            else:
                keep = q["mean_cont"][pixel]
                q["mean_cont"][:] = 0.0
                q["flux"][pixel], q["ivar"][pixel] = 1.5 * keep, 10.0
                if kind != "none":
                    q["mean_cont"][pixel] = keep
            specs.append(q)
            want.append(status)
            orders.append(1 if "negative" in kind else 0)
    many = {k: np.concatenate([q[k] for q in specs]) for k in specs[0]}
    many["offsets"] = np.concatenate([[0], np.cumsum([len(q["flux"]) for q in specs])])
    res = continuum.fit_arrays(many, order=np.array(orders), use_constant_weight=constant)
    assert list(res["status"]) == want
    assert list(res["ndata"]) == [(q["ivar"] > 0).sum() for q in specs]
