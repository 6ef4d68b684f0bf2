"""Batches of local lines that need more threads than one launch may have run
in parts: with the bound lowered, the same bits as in one launch, out of place
and in place, and the same report of a rejected half-complex endpoint."""
import pytest
import torch

import pencil_fft_hip as pf

pytestmark = pytest.mark.gpu


def _plans(monkeypatch, make):
    whole = make()
    monkeypatch.setenv("PFH_LAUNCH_THREADS", "9000")
    parts = make()
    monkeypatch.delenv("PFH_LAUNCH_THREADS")
    return whole, parts


@pytest.mark.parametrize("n", [8, 11, 60, 79, 512])
def test_parts_give_the_bits_of_one_launch(gpu, monkeypatch, n):
    lines = 20011
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(lines * n, dtype=torch.complex64, generator=g, device="cuda")
    whole, parts = _plans(monkeypatch, lambda: pf.LocalC2cPlan(n, dtype=torch.complex64))
    ref = whole.forward(x)
    assert torch.equal(torch.view_as_real(parts.forward(x)), torch.view_as_real(ref))
    y = x.clone()
    parts.forward_in_place(y)
    assert torch.equal(torch.view_as_real(y), torch.view_as_real(ref))
    r = torch.randn(lines * n, dtype=torch.float64, generator=g, device="cuda")
    whole, parts = _plans(monkeypatch, lambda: pf.LocalR2cPlan(n, dtype=torch.float64))
    spec = whole.forward(r)
    assert torch.equal(torch.view_as_real(parts.forward(r)), torch.view_as_real(spec))
    assert torch.equal(parts.inverse(spec), whole.inverse(spec))
    spec = spec.view(lines, n // 2 + 1)
    spec[lines - 2, 0] += 1j
    seen = []
    for plan in (whole, parts):
        out = torch.zeros_like(r)
        with pytest.raises(pf.PfhError) as e:
            plan.inverse(spec.view(-1), out)
        assert not out.any()
        seen.append((e.value.variant, e.value.batch, e.value.index))
    assert seen[0] == seen[1] == ("InvalidSpectrumEndpoint", lines - 2, 0)
