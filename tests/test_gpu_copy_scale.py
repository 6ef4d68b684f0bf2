"""GPU parity of the layout copies and of the per-axis scaling at the edges of
their tiles: extents around 64 and 32 elements, rows shorter and longer than a
workgroup, odd lengths, extras; copies are bit-exact, scaling is within the
rounding of its few products."""
import itertools

import numpy as np
import pytest
import torch

import pencil_fft_hip as pf
from util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("element", [1, 2, 3, 4, 8, 16, 24])
@pytest.mark.parametrize("shape,extra", [((65, 33, 130), ()), ((1, 127, 64), (2,)), ((300, 2, 31), (3,)), ((70, 1, 1), ())])
def test_copies_are_bit_exact(gpu, shape, extra, element):
    rng = np.random.default_rng(element)
    n = int(np.prod(shape)) * int(np.prod(extra, dtype=int))
    raw = rng.integers(0, 256, size=(n, element), dtype=np.uint8)
    for src, dst in itertools.product(itertools.permutations(range(3)), repeat=2):
        plan = pf.LocalTransposePlan(shape, src, dst, element, extra_shape=extra)
        x = torch.from_numpy(raw.reshape(-1).copy()).cuda()
        y = torch.zeros_like(x)
        plan.execute(x, y)
        a = raw.reshape(-1, *[shape[p] for p in src], element)
        ref = a.transpose(0, *[1 + src.index(d) for d in dst], 4)
        assert np.array_equal(y.cpu().numpy(), np.ascontiguousarray(ref).reshape(-1)), (src, dst)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(7, 300, 33), (513, 3, 2), (4, 5, 256), (3, 1, 700)])
def test_scale_axes_rows(gpu, shape, dt):
    rng = np.random.default_rng(shape[0])
    td = torch.float32 if dt == np.float32 else torch.float64
    plan = pf.R2cPlan(shape, dtype=td, extra_shape=(2,))
    for side, cf in ((0, False), (1, False), (1, True)):
        perm, lshape, count, _ = plan.layout(side)
        f = [rng.uniform(0.5, 1.5, size=m) + (1j * rng.uniform(-1, 1, size=m) if cf else 0) for m in lshape]
        ft = np.concatenate(f).astype((np.complex64 if dt == np.float32 else np.complex128) if cf else dt)
        x = rng.standard_normal(count) + (1j * rng.standard_normal(count) if side else 0)
        x = x.astype((np.complex64 if dt == np.float32 else np.complex128) if side else dt)
        got = pf.scale_axes(plan, side, torch.from_numpy(x.copy()).cuda(), torch.from_numpy(ft).cuda()).cpu().numpy()
        ref = x.astype(np.complex128).reshape(2, *[lshape[p] for p in perm])
        for pos, p in enumerate(perm):
            off = sum(lshape[:p])
            v = ft[off:off + lshape[p]].astype(np.complex128)
            ref = ref * v.reshape([1] + [-1 if q == pos else 1 for q in range(3)])
        # three products, each within one rounding per component (complex: three)
        assert rel_l2(got, ref) <= 16 * np.finfo(dt).eps, (side, cf)


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("permute", [True, False])
@pytest.mark.parametrize("shape,extra", [((45, 20, 24), ()), ((30, 35, 50), (2,)), ((17, 12, 21), ()), ((11, 9, 16), (3,))])
def test_steps_folded_into_the_last_stage(gpu, shape, extra, permute, dt):
    """execute_scaled / execute_quadratic against the two separate calls:
    last axes with a line plan (folded), on Bluestein and on the generic
    kernel (two steps). The factors are multiplied in the same order with
    permuted output and to within a rounding or two otherwise."""
    plan = pf.R2cPlan(shape, dtype=dt, extra_shape=extra, permute_dims=permute)
    g = torch.Generator(device="cuda")
    g.manual_seed(shape[0])
    x = torch.randn(plan.input_elements(), generator=g, device="cuda", dtype=dt)
    f = torch.rand(shape[0] + shape[1] + shape[2] // 2 + 1, generator=g, device="cuda", dtype=dt) + 0.5
    eps = torch.finfo(dt).eps
    for op in (pf.FORWARD, pf.ADJOINT_INVERSE, pf.ADJOINT_BACKWARD):
        ref = pf.scale_axes(plan, 1, plan.execute(op, x), f)
        got = plan.execute_scaled(op, x, torch.empty_like(ref), f)
        assert torch.linalg.norm(got - ref) <= (0 if permute else 4 * eps) * torch.linalg.norm(ref), op
    spec = plan.forward(x)
    for op in (pf.INVERSE, pf.BACKWARD, pf.ADJOINT_FORWARD):
        ref = pf.quadratic(plan.execute(op, spec), 0.25)
        got = plan.execute_quadratic(op, spec, torch.empty_like(ref), 0.25)
        # a y y as one fused multiply-add or as two roundings
        assert torch.linalg.norm(got - ref) <= 2 * eps * torch.linalg.norm(ref), op
