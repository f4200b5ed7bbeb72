"""The sCMOS LLR where a pixel's model plus variance is a denormal number: its
term (d - mu)^2 / v is 0 / v there, not a number without one."""
from __future__ import annotations

import numpy as np
import pytest

from gaussmle_amd import synth
from gaussmle_amd.models import GaussianXYNB, ParameterConstraints, default_constraints
from test_gpu_parity import gpu_fit_host, lanes_for

N, BOX, CAM = 67, 13, 32


def workload():
    """Dark ROIs of one bright centre pixel, no read noise, a narrow PSF: at the initial estimate (zero iterations) the
    background is 0 and the corners, ten widths away on both axes, hold about 1e-44 photons."""
    rng = np.random.default_rng(77)
    psf = GaussianXYNB(0.55)
    c = default_constraints(psf, 11)
    lo = c.lower.copy()
    lo[3] = 0.0
    data = np.zeros((BOX, BOX, N), np.float32, order="F")
    data[BOX // 2, BOX // 2] = rng.integers(200, 5000, N)
    xc, yc = (rng.integers(1, CAM - BOX + 2, N).astype(np.int32) for _ in range(2))
    return synth.Workload("dark", psf, BOX, data, np.full((4, N), np.nan), ParameterConstraints(lo, c.upper, c.max_step),
                          0, np.zeros((CAM, CAM), np.float32), xc, yc)


@pytest.mark.gpu
def test_llr_of_denormal_variances_matches_oracle():
    from oracle import refcpu
    w = workload()
    r32 = refcpu.fit_workload(w, refcpu.FP32)
    assert np.all(np.isfinite(r32["llr"]))
    for lanes in lanes_for(BOX):
        print(f"[case] denormal variance lanes={lanes}", flush=True)
        res = gpu_fit_host(w, "fp32", lanes)
        np.testing.assert_array_equal(res["params"], r32["params"])
        assert np.all(np.isfinite(res["llr"])), lanes
        assert np.all(np.abs(res["llr"] - r32["llr"]) <= 1e-4 * np.abs(r32["llr"]))
