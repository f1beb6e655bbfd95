"""Row statistics at the edges of the work-group split and of the reference
that a thread's sums are relative to (MI355X), against float64."""

import pytest
import torch

from rl_project_amd import row_stats

pytestmark = pytest.mark.gpu


def _check(x, y, lab, tol, per_row=None):
    """Within rtol = tol and an absolute bound: tol of the batch's largest
    value, or ``per_row`` of each row's own."""
    out = row_stats(x, lab, y, entropy=True, lse=True)
    a = torch.log_softmax(x.double(), -1)
    want = {"logprob": a.gather(-1, lab[:, None])[:, 0], "entropy": -(a.exp() * a).sum(-1),
            "kl": (a.exp() * (a - torch.log_softmax(y.double(), -1))).sum(-1), "lse": torch.logsumexp(x.double(), -1)}
    for name, w in want.items():
        got = getattr(out, name).double()
        if per_row is not None:
            over = ((got - w).abs() / (tol * w.abs() + per_row)).max()
            assert float(over) <= 1.0, (name, float(over))
            continue
        assert torch.allclose(got, w, rtol=tol, atol=tol * (1.0 + float(w.abs().max()))), (name, float((got - w).abs().max()))


# one row per CU and more (256 / 257 rows: a KL's runs go side by side in fours or
# twos); rows shorter than an iteration, its edges, and several iterations
@pytest.mark.parametrize("R", [1, 256, 257])
@pytest.mark.parametrize("V", [1, 7, 2047, 2048, 2049, 4096, 8193, 16385])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_rows_and_lengths(R, V, dt):
    print(f"[rowstats shapes R={R} V={V} {dt}]", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R + V)
    x = (3.0 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    y = (3.0 * torch.randn(R, V, generator=g, device="cuda")).to(dt)
    # (float sums of at most 16 terms in float64 partials: a few 2^-24)
    _check(x, y, torch.randint(0, V, (R,), generator=g, device="cuda"), 1e-6)


@pytest.mark.parametrize("order", ["rising", "falling", "late peak", "far apart"])
@pytest.mark.parametrize("R", [3, 300])
def test_references_that_move(order, R):
    """Values that pass a thread's reference again and again, once, or by less
    than it takes to move it; and rows whose threads hold references far apart."""
    print(f"[rowstats references {order} R={R}]", flush=True)
    V = 40000
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, V, generator=g, device="cuda")
    y = torch.randn(R, V, generator=g, device="cuda")
    ramp = torch.linspace(-60.0, 60.0, V, device="cuda")
    if order == "rising":
        x, y = x + ramp, y + 0.5 * ramp
    elif order == "falling":
        x, y = x - ramp, y + ramp
    elif order == "late peak":
        x[:, -1] = 7.5     # (within the slack of most references)
        x[:, -2000] = 30.0
        y[:, 5] = 50.0
    else:
        x[:, ::7] -= 300.0
        y[:, 1::3] -= 80.0
    # A float term's exponent is rounded to 2^-24 of itself, at most the row's
    # range of scores (times log2 e, and once more for its own weight in the
    # entropy and the KL); the result to 2^-24 of itself.
    span = (x.amax(-1) - x.amin(-1)).double() + (y.amax(-1) - y.amin(-1)).double()
    _check(x, y, torch.randint(0, V, (R,), generator=g, device="cuda"), 2.0 ** -23, per_row=4.0 * 2.0 ** -24 * span)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("R", [3, 300])
@pytest.mark.parametrize("masked", [5000, 20000])
def test_rows_that_begin_with_the_lowest_value(dt, R, masked):
    """A mask of the type's lowest value (its base-2 exponent overflows) over a
    row's head, so that threads begin with it, and over the whole row."""
    print(f"[rowstats lowest {dt} R={R} masked={masked}]", flush=True)
    V = 20000
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, V, generator=g, device="cuda").to(dt)
    x[:, :masked] = torch.finfo(dt).min
    lab = torch.randint(min(masked, V - 100), V, (R,), generator=g, device="cuda")
    out = row_stats(x, lab, entropy=False, lse=True)
    a = torch.log_softmax(x.double(), -1).gather(-1, lab[:, None])[:, 0]
    assert torch.allclose(out.logprob.double(), a, rtol=1e-6, atol=1e-6)
    assert torch.allclose(out.lse.double(), torch.logsumexp(x.double(), -1), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("R", [255, 600])
@pytest.mark.parametrize("V", [512, 4099, 50257])
def test_entropy_is_as_good_as_its_own_rounding(R, V):
    """Scores around 12: the rounding of a reference's base-2 form, up to 3e-7,
    would be in every term of its thread.  Bound: a float32 result's own
    rounding, 2^-24 of it."""
    print(f"[rowstats entropy R={R} V={V}]", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R + V)
    x = 2.5 * torch.randn(R, V, generator=g, device="cuda") + 12.0
    out = row_stats(x, torch.zeros(R, dtype=torch.int64, device="cuda"), entropy=True)
    a = torch.log_softmax(x.double(), -1)
    want = -(a.exp() * a).sum(-1)
    assert float((out.entropy.double() - want).norm() / want.norm()) < 2.0 ** -24
