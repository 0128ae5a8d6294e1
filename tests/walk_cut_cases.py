"""Inputs of the tests of the pair kernel's specialised path for the cross-correlation and the
cuts, shared by the CPU harness tests and the GPU tests."""
import numpy as np

import walk_cases as W

LAYOUTS = ("lattice", "irregular", "random")


def cut_case(layout, option, seed=0):
    """A walk case (exact bin edges; zero weights, short and non-monotone forests; random
    geometry) with signed r_par and / or the cuts, and about half of its pairs on one half
    plate.  Returns (case, r_par rows of one launch of the cross-correlation)."""
    case = {"lattice": W.lattice_case, "irregular": W.irregular_case,
            "random": lambda: W.random_case(seed)}[layout]()
    g, rng = case.g, np.random.default_rng(seed)
    if "cross" in option:
        g.x_correlation = True
        g.num_bins_r_par = 2 * g.num_bins_r_par
        # a range that need not be symmetric, nor put a bin edge at r_par = 0
        g.r_par_min = -g.r_par_max if layout == "lattice" else -0.7 * g.r_par_max
    g.remove_same_half_plate_close_pairs = "plate" in option
    if "z" in option:
        # forests whose pixels sit on the cut, and the cut inside the others
        z = case.store.z
        g.z_min_pairs = float(np.quantile(z, 0.3))
        g.z_max_pairs = float(np.quantile(z, 0.8)) if seed % 2 == 0 else None
    if "err" in option:
        g.zerr_cut_deg, g.zerr_cut_kms = 0.5, 20000.0
        case.store.z_qso[:] = case.store.z[case.store.offsets[:-1]] + 0.01
    case.pairs.pair_flags[:] = rng.random(case.pairs.num_pairs) < 0.5
    return case, max(1, (g.num_bins_r_par + 2) // 3)
