"""Rounding error of lengths with a factor 11 or 13 against that of the next
7-smooth length with as many radix passes: direct butterflies of 11 and 13
points round about as often as those of 12 and 14, so the relative L2 errors
agree but for the longer sum of the prime butterfly; 25% covers it (a chirp
convolution of twice the length, 60% and more, does not)."""
import numpy as np
import pytest
import torch

import pencil_fft_hip as pf

pytestmark = pytest.mark.gpu


def _error(n, real, dt):
    wide = np.float64 if dt == np.float32 else np.longdouble
    rng = np.random.default_rng(n)
    lines = 24000 // n
    x = rng.standard_normal((lines, n)).astype(dt)
    if not real:
        x = (x + 1j * rng.standard_normal((lines, n))).astype(np.complex64 if dt == np.float32 else np.complex128)
    td = torch.from_numpy(x[:1].copy()).dtype
    plan = pf.LocalR2cPlan(n, dtype=td) if real else pf.LocalC2cPlan(n, dtype=td)
    got = plan.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = np.fft.rfft(x.astype(wide)) if real else np.fft.fft(x.astype(np.result_type(x.dtype, wide)))
    err = got.reshape(ref.shape) - ref
    return float(np.sqrt((np.abs(err) ** 2).sum() / (np.abs(ref) ** 2).sum()))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n, smooth", [(44, 48), (52, 56), (88, 96), (104, 112), (176, 192), (208, 224)])
def test_factors_of_11_and_13_round_like_their_neighbours(gpu, n, smooth, dt):
    assert _error(n, False, dt) <= 1.25 * _error(smooth, False, dt)
    assert _error(2 * n, True, dt) <= 1.25 * _error(2 * smooth, True, dt)
