"""Row statistics of rows masked with a finite value (the type's lowest, as
masked_fill with finfo.min leaves it): every statistic is finite where the
reference's expression is (MI355X), against float64."""

import pytest
import torch

from rl_project_amd import row_stats

pytestmark = pytest.mark.gpu


def _want(x, y):
    a, b = torch.log_softmax(x.double(), -1), torch.log_softmax(y.double(), -1)
    return -(a.exp() * a).sum(-1), (a.exp() * (a - b)).sum(-1)


def _close(got, want, rtol, scale):
    return torch.allclose(got.double(), want, rtol=rtol, atol=rtol * scale)


# (the shortest row whose threads reach whole iterations, a ragged one, several
# iterations; rows of one CU and more)
@pytest.mark.parametrize("where", ["third", "head", "tail", "one"])
@pytest.mark.parametrize("V", [7, 4100, 40000, 70001])
@pytest.mark.parametrize("R", [3, 300])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
def test_finite_masks(dt, R, V, where):
    print(f"[rowstats masks {dt} R={R} V={V} {where}]", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R + V)
    x = (2.0 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    y = (2.0 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    at = {"third": slice(0, V, 3), "head": slice(0, V // 2), "tail": slice(V // 2, V), "one": slice(V // 2, V // 2 + 1)}[where]
    x[:, at] = torch.finfo(dt).min
    y[:, at] = torch.finfo(dt).min
    out = row_stats(x, None, y, entropy=True)
    h, kl = _want(x, y)
    # (float sums of at most 16 terms in float64 partials: a few 2^-24 of the
    # result; a KL term is a difference of exponents up to 2 * 11 * log2 e,
    # each rounded to 2^-24 of that)
    assert _close(out.entropy, h, 2e-6, 1.0), float((out.entropy.double() - h).abs().max())
    assert _close(out.kl, kl, 2e-6, 2.0), float((out.kl.double() - kl).abs().max())
    # a mask of the reference row alone: p times the lowest value, large and finite
    z = (2.0 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    _, kl = _want(z, y)
    out = row_stats(z, None, y, entropy=True)
    assert bool(torch.isfinite(kl).all()) and _close(out.kl, kl, 2e-6, float(kl.abs().min()))
    # of the row alone
    _, kl = _want(x, z)
    assert _close(row_stats(x, None, z).kl, kl, 2e-6, 2.0)


@pytest.mark.parametrize("R", [3, 300])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_infinite_masks_beside_finite_ones(dt, R):
    """-inf logits keep the reference's 0 * -inf = NaN, whether a finite mask
    comes before or after them; a -inf of the reference row alone keeps +inf."""
    print(f"[rowstats masks -inf {dt} R={R}]", flush=True)
    V, low, inf = 40000, torch.finfo(dt).min, float("-inf")
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, V, generator=g, device="cuda").to(dt)
    y = torch.randn(R, V, generator=g, device="cuda").to(dt)
    x[0, :20000:3], x[0, 30000] = low, inf
    x[1, 5], x[1, 20000::3] = inf, low
    y[2, 100], y[2, 200::7], x[2, 200::7] = inf, low, low
    out = row_stats(x, None, y, entropy=True)
    h, kl = _want(x, y)
    assert bool(torch.isnan(out.entropy[:2]).all()) and bool(torch.isnan(out.kl[:2]).all())
    assert bool(torch.isnan(h[:2]).all()) and float(kl[2]) == float("inf") == float(out.kl[2])
    assert _close(out.entropy[2:], h[2:], 2e-6, 1.0) and _close(out.kl[3:], kl[3:], 2e-6, 2.0)


@pytest.mark.parametrize("low", [-3.0e38, -1.7e38, -1.0e38, -6.0e37, -1.0e15, -1.7e9, -1.3e9, -1.0e9])
@pytest.mark.parametrize("V", [5, 2050, 40003])
def test_masks_of_any_depth(low, V):
    """Rows of a mask value alone but for their last, with the row's end inside
    an iteration: the mask is some lanes' reference."""
    print(f"[rowstats masks low={low} V={V}]", flush=True)
    R = 3
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.full((R, V), low, device="cuda")
    y = torch.full((R, V), low, device="cuda")
    x[1:, V - 3:], y[2:, V - 4:] = torch.randn(R - 1, 3, generator=g, device="cuda"), torch.randn(R - 2, 4, generator=g, device="cuda")
    lab = torch.full((R,), V - 2, device="cuda")
    out = row_stats(x, lab, y, entropy=True, lse=True)
    h, kl = _want(x, y)
    assert _close(out.entropy, h, 2e-6, 1.0) and _close(out.logprob, torch.log_softmax(x.double(), -1)[:, V - 2], 2e-6, 1.0)
    assert _close(out.lse, torch.logsumexp(x.double(), -1), 2e-6, 1.0)
    assert _close(out.kl, kl, 2e-6, 2.0), (out.kl, kl)
