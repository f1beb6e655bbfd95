"""A row's statistics are a function of the row alone: the same bits in calls of
any number of rows, however the call splits a row over threads (MI355X)."""

import pytest
import torch

from rl_project_amd import row_stats

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [33, 4099, 9000, 16384, 32771, 50257, 70001, 128256])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kl", [False, True])
def test_a_row_alone_and_among_others(V, dt, kl):
    print(f"[rowstats rows V={V} {dt} kl={kl}]", flush=True)
    R = 1100
    g = torch.Generator(device="cuda").manual_seed(V)
    x = (2.5 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    y = (x + 0.3 * torch.randn(R, V, generator=g, device="cuda").to(dt)) if kl else None
    lab = torch.randint(0, V, (R,), generator=g, device="cuda")
    whole = row_stats(x, lab, y, entropy=True, lse=True)
    for n in (1, 64, 255, 256, 257, 512, 513, 600):
        part = row_stats(x[:n], lab[:n], None if y is None else y[:n], entropy=True, lse=True)
        for name in ("logprob", "entropy", "lse") + (("kl",) if kl else ()):
            assert torch.equal(getattr(part, name), getattr(whole, name)[:n]), (n, name)
