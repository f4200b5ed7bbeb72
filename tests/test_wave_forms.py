"""The two forms of the Poisson pixel loop: a wave takes the masked one when any
of its ROIs needs the 0.01 threshold or the caps, and an ROI that needs neither
has to come out the same, bit for bit, whatever its neighbours are."""
from __future__ import annotations

import numpy as np
import pytest

from gaussmle_amd import synth
from gaussmle_amd.models import GaussianXYNB, GaussianXYNBSXSY, GaussianXYNBS
from test_gpu_parity import gpu_fit_host, lanes_for

N = 256   # whole waves at every lane count


def workloads(psf, box):
    """Ordinary ROIs, and the same ones each followed by one of near-zero background."""
    low = synth.low_background(psf, N, box, seed=981, bg_range=(0.002, 0.04))
    plain = synth.generic(psf, N, box, seed=980, constraints=low.constraints)
    both = np.empty((box, box, 2 * N), np.float32, order="F")
    both[:, :, 0::2], both[:, :, 1::2] = plain.data, low.data
    mixed = synth.Workload("mixed", psf, box, both, np.full((len(psf), 2 * N), np.nan), low.constraints, 20)
    return plain, mixed


@pytest.mark.gpu
@pytest.mark.parametrize("psf,box", [(GaussianXYNB(1.3), 11), (GaussianXYNB(1.3), 13), (GaussianXYNBS(), 9),
                                     (GaussianXYNBSXSY(), 11)])
def test_neighbours_do_not_change_an_roi(psf, box):
    plain, mixed = workloads(psf, box)
    for lanes in lanes_for(box):
        print(f"[case] wave forms {type(psf).__name__} {box} px lanes={lanes}", flush=True)
        a, b = gpu_fit_host(plain, "fp32", lanes), gpu_fit_host(mixed, "fp32", lanes)
        for k in ("params", "crlb", "llr"):
            np.testing.assert_array_equal(a[k], b[k][0::2], err_msg=f"{k} lanes={lanes}")
