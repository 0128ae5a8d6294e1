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
