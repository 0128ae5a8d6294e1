"""What other programs hold on to: the package builds without the tests, and the run walk
compiles against memory types that have only its first interface (tests/native/
xi_walk_records_host.hip), with the planes of the kernel holding the same prefix sums."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import walk_cases as W
import walk_harness as H
from picca_amd.engine import params_from_globals

ROOT = os.path.dirname(H.HERE)


def test_build_leaves_the_tests_alone(monkeypatch):
    """__graft_entry__.build() compiles the package and the oracle, and nothing of tests/."""
    import __graft_entry__ as entry
    from picca_amd import build as engine_build

    made = []
    monkeypatch.setattr(engine_build, "build", lambda verbose=False: made.append("engine"))
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: made.append(" ".join(cmd)))
    monkeypatch.setattr(H, "build", lambda: made.append("harness"))
    monkeypatch.setattr(sys, "path", list(sys.path))
    entry.build()
    assert made[0] == "engine" and len(made) == 2 and "oracle" in made[1]


@pytest.fixture(scope="module")
def records(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("walk") / "libxi_walk_records.so")
    source = os.path.join(H.HERE, "native", "xi_walk_records_host.hip")
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    subprocess.run([hipcc if os.path.exists(hipcc) else "hipcc", "--offload-arch=gfx950", "-O2",
                    "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-o", out, source],
                   check=True)
    lib = ctypes.CDLL(out)
    lib.xi_walk_records.restype = ctypes.c_int64
    return lib


def test_records_against_pixel_pairs(records):
    """One pixel of a 0.8 A survey with another forest, against the sums pixel pair by pixel
    pair (prefix differences: 1e-9 of the summed magnitudes), and the planes' entries."""
    case = W.survey_case("survey_100k", 0.001)
    p, s, g = case.pairs, case.store, case.g
    lengths = np.diff(s.offsets)
    k = int(np.argmax(np.minimum(lengths[p.pair_a], lengths[p.pair_b])))
    a, b, ang = p.pair_a[k], p.pair_b[k], float(p.pair_ang[k])
    lo, hi = s.offsets[b], s.offsets[b + 1]
    n = int(hi - lo)
    r, d, z, w, delta = (np.ascontiguousarray(getattr(s, name)[lo:hi], dtype=np.float64)
                         for name in ("r_comov", "dist_m", "z", "weights", "delta"))
    i = s.offsets[a] + np.searchsorted(s.r_comov[s.offsets[a]:s.offsets[a + 1] - 1], r[n // 2])
    one = np.array([s.r_comov[i], s.dist_m[i], s.z[i], s.weights[i], s.delta[i]])
    out = np.zeros(((g.num_bins_r_par + 1) * (g.num_bins_r_trans + 1), 5))
    entries, planes = np.zeros((n + 1, 6)), np.zeros((3, n + 1, 2))
    params = params_from_globals(g)
    runs = records.xi_walk_records(ctypes.byref(params), ctypes.c_double(ang), H._p(one),
                                   ctypes.c_int(n), H._p(r), H._p(d), H._p(z), H._p(w),
                                   H._p(delta), H._p(out), H._p(entries))
    assert runs > 10
    r_par = np.abs((one[0] - r) * np.cos(ang / 2))
    r_trans = (one[1] + d) * np.sin(ang / 2)
    keep = (r_par < g.r_par_max) & (r_trans < g.r_trans_max) & (w != 0)
    bins = ((r_trans / g.r_trans_max * g.num_bins_r_trans).astype(int)
            + (g.num_bins_r_trans + 1) * (r_par / g.r_par_max * g.num_bins_r_par).astype(int))
    w12 = one[3] * w
    terms = np.stack([w12, one[4] * one[3] * delta * w, r_par * w12, r_trans * w12,
                      0.5 * (one[2] + z) * w12], axis=1)
    want, size = np.zeros_like(out), np.zeros_like(out)
    np.add.at(want, bins[keep], terms[keep])
    np.add.at(size, bins[keep], np.abs(terms[keep]))
    inside = size[:, 0] > 0
    assert inside.sum() > 10 and keep.sum() > 100
    assert np.all(np.abs(out - want)[inside] <= 1e-9 * size[inside].max(axis=0))
    assert not out[:, 0][~inside].any()
    records.xi_walk_planes(ctypes.c_int(n), H._p(r), H._p(d), H._p(z), H._p(w), H._p(delta),
                           H._p(planes))
    assert np.array_equal(planes.transpose(1, 0, 2).reshape(n + 1, 6), entries)
