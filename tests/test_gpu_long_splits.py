"""Splits of more than 2^20 points, whose twiddles are products of two table
entries, and a Bluestein convolution of that length, against 64 bits. Bounds:
the suite's 2e-6 (f32) and 1e-12 (f64) relative L2."""
import numpy as np
import pytest
import torch

import pencil_fft_hip as pf
from util import complex_of, rel_l2, tol, uniform_complex

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1 << 21, 3 << 19, 1500000, 700001])
def test_splits_above_two_to_the_twenty(gpu, n, dt):
    x = uniform_complex(np.random.default_rng(n), (2, n), complex_of(dt))
    plan = pf.LocalC2cPlan(n, dtype=torch.from_numpy(x).dtype)
    y = plan.forward(torch.from_numpy(x).cuda())
    assert rel_l2(y.cpu().numpy(), np.fft.fft(x.astype(np.complex128))) <= tol(dt)
    assert rel_l2(plan.inverse(y).cpu().numpy(), x) <= 2 * tol(dt)
