"""execute_scaled and execute_quadratic give the bits of the operation followed
by scale_axes / quadratic: C2C, R2C and mixed plans, every axis order, extras,
axes of extent 1 (not folded), last axes on line plans (folded), on Bluestein
and on the generic kernel (two steps). Tolerance zero: both compute the same
products in the same order and the same fused multiply-add."""
import pytest
import torch

import pencil_fft_hip as pf

pytestmark = pytest.mark.gpu

SHAPES = [(16, 12, 20), (45, 20, 24), (64, 1, 48), (16, 20, 1), (1, 16, 24), (79, 12, 20), (17, 12, 20), (11, 9, 16), (8, 6, 5, 10)]
COMPLEX = {torch.float32: torch.complex64, torch.float64: torch.complex128}


def _plan(kind, shape, extra, permute, dt):
    if kind == "c2c":
        return pf.C2cPlan(shape, dtype=COMPLEX[dt], extra_shape=extra, permute_dims=permute)
    if kind == "r2c":
        return pf.R2cPlan(shape, dtype=dt, extra_shape=extra, permute_dims=permute)
    axes = [pf.AxisTransform.FFT] * (len(shape) - 2) + [pf.AxisTransform.RFFT, pf.R2rKind.DctII]
    return pf.MixedR2cPlan(shape, axes, dtype=dt, extra_shape=extra, permute_dims=permute)


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("permute", [True, False])
@pytest.mark.parametrize("extra", [(), (3,)])
@pytest.mark.parametrize("kind", ["c2c", "r2c", "mixed"])
def test_folded_steps_give_the_bits_of_two_calls(gpu, kind, extra, permute, dt):
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    for shape in SHAPES:
        if shape[{"c2c": 0, "r2c": -1, "mixed": -2}[kind]] == 1 and kind != "c2c":
            continue
        plan = _plan(kind, shape, extra, permute, dt)
        x = torch.randn(plan.input_elements(), generator=g, device="cuda", dtype=COMPLEX[dt] if kind == "c2c" else dt)
        f = torch.rand(sum(plan.layout(1)[1]), generator=g, device="cuda", dtype=dt) + 0.5
        for op in (pf.FORWARD, pf.ADJOINT_INVERSE, pf.ADJOINT_BACKWARD):
            ref = pf.scale_axes(plan, 1, plan.execute(op, x), f)
            got = plan.execute_scaled(op, x, torch.empty_like(ref), f)
            assert torch.equal(torch.view_as_real(got), torch.view_as_real(ref)), (shape, op)
        if kind == "c2c":
            continue
        spec = plan.forward(x)
        for op in (pf.INVERSE, pf.BACKWARD, pf.ADJOINT_FORWARD):
            ref = pf.quadratic(plan.execute(op, spec), 0.25)
            got = plan.execute_quadratic(op, spec, torch.empty_like(ref), 0.25)
            assert torch.equal(got, ref), (shape, op)


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
def test_factors_the_plan_cannot_take(gpu, dt):
    """Refused before any launch: another precision, too few or too many
    factors. Complex factors are the two calls."""
    other = torch.float64 if dt == torch.float32 else torch.float32
    plan = pf.C2cPlan((16, 12, 20), dtype=COMPLEX[dt])
    x = torch.randn(plan.input_elements(), device="cuda", dtype=COMPLEX[dt])
    dst = torch.zeros_like(x)
    for bad, error in ((torch.ones(48, device="cuda", dtype=other), TypeError),
                       (torch.ones(48, device="cuda", dtype=COMPLEX[other]), TypeError),
                       (torch.ones(47, device="cuda", dtype=dt), ValueError),
                       (torch.ones(49, device="cuda", dtype=dt), ValueError),
                       (torch.ones(47, device="cuda", dtype=COMPLEX[dt]), ValueError)):
        with pytest.raises(error):
            plan.execute_scaled(pf.FORWARD, x, dst, bad)
    with pytest.raises(ValueError):
        plan.execute_scaled(pf.INVERSE, x, dst, torch.ones(48, device="cuda", dtype=COMPLEX[dt]))
    assert not dst.any()
    f = torch.randn(48, device="cuda", dtype=COMPLEX[dt])
    got = plan.execute_scaled(pf.FORWARD, x, dst, f)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(pf.scale_axes(plan, 1, plan.forward(x), f)))
