"""Fit kernels where the rows' way through LDS and the split of the columns
change form: fewer columns than lanes, one column per lane (with and without a
split last column), and the last column's rows from registers and from LDS;
against the oracle under the tolerances of tests/parity.py."""
from __future__ import annotations

import numpy as np
import pytest

import gaussmle_amd as g
from gaussmle_amd import synth
from gaussmle_amd.models import GaussianXYNB, GaussianXYNBSXSY
from parity import assert_parity, compare, llr_rounding_scale, perturbed_workload
from test_gpu_parity import gpu_fit_host, lanes_for

pytestmark = pytest.mark.gpu

N = 193   # a ragged last wave at every lane count


# (six parameters on the 25 pixels of a 5 px box are beyond Float32: their CRLB is off by 3e-3 in every build)
@pytest.mark.parametrize("scmos", [False, True])
@pytest.mark.parametrize("model,box", [("xynb", b) for b in (5, 8, 9, 13, 16, 17)] +
                         [("xynbsxsy", b) for b in (8, 9, 13, 16, 17)])
def test_row_and_column_forms_match_oracle(model, box, scmos):
    from oracle import refcpu
    psf = GaussianXYNB(1.3) if model == "xynb" else GaussianXYNBSXSY()
    w = synth.generic(psf, N, box, seed=970 + box, scmos=scmos,
                      constraints=g.default_constraints(psf, max(11, box)))
    r32, r64 = refcpu.fit_workload(w, refcpu.FP32), refcpu.fit_workload(w, refcpu.FP64)
    r64p = refcpu.fit_workload(perturbed_workload(w), refcpu.FP64)
    r32fp = refcpu.final_pass(perturbed_workload(w), r32["params"], refcpu.FP32)
    for lanes in lanes_for(box):
        print(f"[case] rows {model} box={box} scmos={scmos} lanes={lanes}", flush=True)
        res = gpu_fit_host(w, "fp32", lanes)
        r32g = refcpu.final_pass(w, np.asarray(res["params"], np.float64), refcpu.FP32)
        rep = compare(psf.model_id, res, r32, r64, "fp32", r64p, None, llr_rounding_scale(w), r32fp, r32g)
        assert_parity(rep, f"{model} box={box} scmos={scmos} L={lanes}")
