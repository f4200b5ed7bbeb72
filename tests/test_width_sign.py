"""Fitted widths with bounds below 0: the pixel integrals depend on sigma^2 alone,
so a spot with a negative width stays a spot; against the oracle under the
tolerances of tests/parity.py.

Two iterations: the first ends at the bound, the second and the final pass run
at a negative width.  More would test the rounding instead: the reference's
position gradient carries the sign of sigma (-N / (sqrt(2 pi) sigma)), so that
below 0 every iteration moves away from the maximum, and a difference grows about
1.5 times in each (Float32 against Float64 oracle: 6.7e-7 px after 2, 8e-4 after 20)."""
from __future__ import annotations

import numpy as np
import pytest

from gaussmle_amd import synth
from gaussmle_amd.models import GaussianXYNBS, GaussianXYNBSXSY, ParameterConstraints, default_constraints
from parity import assert_parity, compare, llr_rounding_scale, perturbed_workload
from test_gpu_parity import gpu_fit_host, lanes_for

N = 193   # a ragged last wave at every lane count


def workload(psf, k, scmos):
    """Parameter k, a width, bounded to [-3, -0.9]."""
    c = default_constraints(psf, 11)
    lo, up = c.lower.copy(), c.upper.copy()
    lo[k], up[k] = -3.0, -0.9
    return synth.generic(psf, N, 11, seed=950 + k, iterations=2, scmos=scmos,
                         constraints=ParameterConstraints(lo, up, c.max_step))


CASES = {"xynbs_ideal": (GaussianXYNBS(), 4, False), "xynbsxsy_ideal": (GaussianXYNBSXSY(), 5, False),
         "xynbsxsy_scmos": (GaussianXYNBSXSY(), 4, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision", ["fp32", "mixed"])
def test_negative_width_matches_oracle(name, precision):
    from oracle import refcpu
    psf, k, scmos = CASES[name]
    w = workload(psf, k, scmos)
    r32, r64 = refcpu.fit_workload(w, refcpu.FP32), refcpu.fit_workload(w, refcpu.FP64)
    r64p = refcpu.fit_workload(perturbed_workload(w), refcpu.FP64)
    rmix = refcpu.fit_workload(w, refcpu.MIXED) if precision == "mixed" else None
    for lanes in lanes_for(w.box):
        print(f"[case] width below 0 {name} {precision} lanes={lanes}", flush=True)
        res = gpu_fit_host(w, precision, lanes)
        assert np.all(res["params"][:, k] < -0.89)
        rep = compare(psf.model_id, res, r32, r64, precision, r64p, rmix, llr_rounding_scale(w))
        assert rep["n"] - rep["n_ill"] > 0.9 * rep["n"]
        assert_parity(rep, f"{name} {precision} L={lanes}")
