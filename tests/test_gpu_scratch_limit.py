"""A route whose long real lines would take a second region as a split (219 MB)
keeps the pieces that the allocation-free entry point's 128 MiB hold (132 MB), and
gives the transform. Bound: the suite's 1e-12 relative L2 of a 3D f64 transform, 4x
for the three stages."""
import numpy as np
import pytest
import torch

import pencil_fft_hip as pf
from util import rel_l2, tol

pytestmark = pytest.mark.gpu


def test_long_lines_within_the_scratch(gpu):
    shape = (36, 36, 4235)
    plan = pf.R2cPlan(shape, dtype=torch.float64)
    assert plan.workspace_bytes(pf.FORWARD) <= 128 << 20
    x = np.random.default_rng(4235).standard_normal(shape)
    xd = torch.from_numpy(x.reshape(-1)).cuda()
    spec = torch.zeros(plan.output_elements(), dtype=torch.complex128, device="cuda")
    back = torch.zeros_like(xd)
    lib = pf.load_library()
    for op, src, dst in ((pf.FORWARD, xd, spec), (pf.INVERSE, spec, back)):
        pf._check(lib.pfh_execute_noalloc(plan._h, op, pf._ptr(src), src.numel(), pf._ptr(dst), dst.numel(),
                                          pf._stream(), 0))
    ref = np.fft.rfftn(x).transpose(2, 1, 0)
    assert rel_l2(spec.cpu().numpy(), np.ascontiguousarray(ref)) <= 4 * tol(np.float64)
    assert rel_l2(back.cpu().numpy(), x) <= 8 * tol(np.float64)
