"""Every planned length on every kind of the line plans that a single stage
reaches, with a full tile of lines and a part of a second one: C2C and even and
odd half-complex lines up to 1024 points, one real-to-real mode after the other
up to 512, and the folded pointwise steps against the separate calls. Bounds:
the suite's 2e-6 (f32) and 1e-12 (f64) relative L2, of a transform of few
passes; folded steps are equal bit for bit."""
import numpy as np
import pytest
import scipy.fft
import torch

import pencil_fft_hip as pf
from test_line_plan_table import _best, _smooth
from util import complex_of, rel_l2, tol, uniform_complex, uniform_real

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64]
PLANNED = [m for m in range(8, 1025) if _smooth(m) and _best(m)] + [385]


def _lines(m):
    """A full tile of row lines (256 threads over the threads of a line) and
    some of a second one."""
    return 256 // _best(m)[2] + 3


def _dev(x):
    return torch.from_numpy(x).cuda()


def _close(got, ref, dt, factor, what):
    assert rel_l2(got.cpu().numpy(), ref) <= factor * tol(dt), what


@pytest.mark.parametrize("dt", DTYPES)
def test_complex_and_half_complex_lengths(gpu, dt):
    rng = np.random.default_rng(61)
    for m in PLANNED:
        lines = _lines(m)
        x = uniform_complex(rng, (lines, m), complex_of(dt))
        plan = pf.LocalC2cPlan(m, dtype=torch.from_numpy(x).dtype)
        _close(plan.forward(_dev(x)), np.fft.fft(x.astype(np.complex128)), dt, 1, m)
        _close(plan.inverse(_dev(x)), np.fft.ifft(x.astype(np.complex128)), dt, 1, m)
        for n in (2 * m,) if m % 2 == 0 else (m, 2 * m):
            r = uniform_real(rng, (lines, n), dt)
            plan = pf.LocalR2cPlan(n, dtype=torch.from_numpy(r).dtype)
            spec = plan.forward(_dev(r))
            _close(spec, np.fft.rfft(r.astype(np.float64)), dt, 1, n)
            _close(plan.inverse(spec), r, dt, 2, n)


@pytest.mark.parametrize("dt", DTYPES)
def test_real_to_real_lengths(gpu, dt):
    """Line lengths whose FFT length is m: DCT-I m + 1, DST-I m - 1, the other
    kinds 2 m, and m where m is odd; the kinds in turn, two per length."""
    rng = np.random.default_rng(67)
    turn = 0
    for m in [m for m in PLANNED if m <= 512]:
        forms = [(1, m + 1), (5, m - 1)] + [(k, 2 * m) for k in (2, 3, 4, 6, 7, 8, 9)]
        if m % 2:
            forms += [(k, m) for k in (2, 3, 6, 7, 9)]
        for kind, n in (forms[turn % len(forms)], forms[(turn + 4) % len(forms)]):
            x = uniform_real(rng, (_lines(m), n), dt)
            td = torch.from_numpy(x).dtype
            wide = x.astype(np.float64)
            if kind == 9:
                plan, f = pf.LocalDhtPlan(n, dtype=td), np.fft.fft(wide)
                ref = f.real - f.imag
            else:
                plan = pf.LocalR2rPlan(n, kind, dtype=td)
                ref = scipy.fft.dct(wide, type=kind) if kind <= 4 else scipy.fft.dst(wide, type=kind - 4)
            _close(plan.forward(_dev(x)), ref, dt, 1, (kind, n))
        turn += 1


@pytest.mark.parametrize("dt", DTYPES)
def test_folded_steps_at_every_length(gpu, dt):
    rng = np.random.default_rng(71)
    td = torch.from_numpy(np.zeros(1, dt)).dtype
    for m in PLANNED:
        plan = pf.C2cPlan((m, 3, 7), dtype=torch.from_numpy(np.zeros(1, complex_of(dt))).dtype)
        x = _dev(uniform_complex(rng, 21 * m, complex_of(dt)))
        f = _dev(uniform_real(rng, m + 10, dt) + dt(2))
        ref = pf.scale_axes(plan, 1, plan.forward(x), f)
        got = plan.execute_scaled(pf.FORWARD, x, torch.empty_like(x), f)
        assert torch.equal(torch.view_as_real(got), torch.view_as_real(ref)), m
        for n in (2 * m,) if m % 2 == 0 else (m, 2 * m):
            plan = pf.R2cPlan((3, 7, n), dtype=td)
            spec = plan.forward(_dev(uniform_real(rng, 21 * n, dt)))
            ref = pf.quadratic(plan.inverse(spec), 0.25)
            assert torch.equal(plan.execute_quadratic(pf.INVERSE, spec, torch.empty_like(ref), 0.25), ref), n
