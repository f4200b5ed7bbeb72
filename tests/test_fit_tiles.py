"""Fit kernels at the edges of their lane tiles: boxes the lanes divide with
and without a remainder (padding columns, lanes that hold only padding, the
split last column), on both likelihood paths, against the oracle under the
tolerances of tests/parity.py."""
from __future__ import annotations

import numpy as np
import pytest

import gaussmle_amd as g
from gaussmle_amd import synth
from gaussmle_amd.models import GaussianXYNB, GaussianXYNBS, GaussianXYNBSXSY
from parity import assert_parity, compare, llr_rounding_scale, perturbed_workload
from test_gpu_parity import gpu_fit_host, lanes_for

pytestmark = pytest.mark.gpu

N = 321   # a ragged last wave at every lane count

CASES = {
    "xynb_ideal_10": lambda: synth.generic(GaussianXYNB(1.3), N, 10, seed=901),
    # backgrounds near the 0.01 threshold: the masked likelihood path
    "xynb_ideal_10_low_bg": lambda: synth.generic(GaussianXYNB(1.3), N, 10, seed=902, bg_range=(0.3, 0.6)),
    "xynbs_ideal_9": lambda: synth.generic(GaussianXYNBS(), N, 9, seed=903),
    "xynbsxsy_scmos_10": lambda: synth.generic(GaussianXYNBSXSY(), N, 10, seed=904, scmos=True, sigma_range=(1.0, 1.8)),
    "astig_ideal_14": lambda: synth.generic(synth.ASTIG_CONFIG_PSF, N, 14, seed=905, n_range=(1000, 10000)),
    "xynbs_scmos_17": lambda: synth.generic(GaussianXYNBS(), N, 17, seed=906, scmos=True,
                                            constraints=g.default_constraints(GaussianXYNBS(), 17)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_lane_tiles_match_oracle(name):
    from oracle import refcpu
    w = CASES[name]()
    r32, r64 = refcpu.fit_workload(w, refcpu.FP32), refcpu.fit_workload(w, refcpu.FP64)
    r64p = refcpu.fit_workload(perturbed_workload(w), refcpu.FP64)
    r32fp = refcpu.final_pass(perturbed_workload(w), r32["params"], refcpu.FP32)
    for lanes in lanes_for(w.box):
        print(f"[case] tiles {name} lanes={lanes}", flush=True)
        res = gpu_fit_host(w, "fp32", lanes)
        r32g = refcpu.final_pass(w, np.asarray(res["params"], np.float64), refcpu.FP32)
        rep = compare(w.psf_pixels.model_id, res, r32, r64, "fp32", r64p, None, llr_rounding_scale(w), r32fp, r32g)
        assert_parity(rep, f"{name} L={lanes}")
