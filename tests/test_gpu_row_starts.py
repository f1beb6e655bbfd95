"""Rows that start at any multiple of their element size (odd vocabularies,
slices of padded buffers) take the same 16-byte loads as aligned ones and give
the same results, bit for bit (MI355X)."""

import pytest
import torch

from rl_project_amd import SpecPlan, row_stats, sample_tokens, workloads
from tests.helpers import classify_workload

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _placed(x, offset, pad):
    """x [B, V] on the GPU as a view that starts `offset` elements into rows of V + pad."""
    B, V = x.shape
    base = torch.full((B, V + pad), 99.0, dtype=x.dtype, device="cuda")  # (read past a row: the largest value)
    base[:, offset:offset + V] = x.cuda()
    return base[:, offset:offset + V]


# one chunk and less, the edges of a chunk and of a slot of 1024 chunks, the
# register tiles' edges (32768 float32, 131072 16-bit values) and past them
@pytest.mark.parametrize("dt,V", [("bf16", 7), ("bf16", 8193), ("bf16", 50257), ("bf16", 131071), ("bf16", 131077),
                                  ("f16", 8191), ("f32", 5), ("f32", 4097), ("f32", 32767), ("f32", 50257)])
def test_sampler_same_at_every_start(dt, V):
    print(f"[row starts {dt} V={V}]", flush=True)
    B = 6
    w = workloads.make("hetero_bf16_256x128256", seed=3, batch=B, vocab=V)
    x = w.logits.to(DT[dt])
    x[0, V - 1] = 60.0   # the last value: greedy and certain
    w.temperature[0] = 0.0
    x[1, V - 1] = 60.0
    w.repetition_penalty[1] = 1.0
    hist = w.history[:, :64].contiguous()
    kw = dict(w.to("cuda").kwargs(), history=hist.cuda())
    ref = sample_tokens(x.cuda().contiguous(), return_logprobs=True, return_desc=True, **kw)
    for offset in (0, 1, 3, 6):
        for pad in (7, 8):
            out = sample_tokens(_placed(x, offset, pad), return_logprobs=True, return_desc=True, **kw)
            for name in ("tokens", "status", "logprobs", "desc"):
                assert torch.equal(getattr(out, name).cpu(), getattr(ref, name).cpu()), (offset, pad, name)
    assert int(ref.tokens[1]) == V - 1
    import dataclasses
    summ, verdicts = classify_workload(dataclasses.replace(w, logits=x, history=hist), ref.tokens)
    assert all(v.ok for v in verdicts), summ


@pytest.mark.parametrize("dt,V", [("bf16", 1021), ("f16", 50257), ("f32", 4099), ("f32", 50257)])
def test_row_stats_same_at_every_start(dt, V):
    print(f"[row starts, stats {dt} V={V}]", flush=True)
    g = torch.Generator().manual_seed(1)
    x = (2.0 * torch.randn(3, V, generator=g)).to(DT[dt])
    y = (2.0 * torch.randn(3, V, generator=g)).to(DT[dt])
    lab = torch.tensor([0, V - 1, V // 2]).cuda()
    ref = row_stats(x.cuda(), lab, y.cuda(), entropy=True, lse=True)
    for ox, oy in ((1, 0), (3, 2), (0, 5)):
        out = row_stats(_placed(x, ox, 7), lab, _placed(y, oy, 7), entropy=True, lse=True)
        for name in ("logprob", "entropy", "kl", "lse"):
            assert torch.equal(getattr(out, name).cpu(), getattr(ref, name).cpu()), (ox, oy, name)


@pytest.mark.parametrize("dt,V", [("bf16", 4099), ("bf16", 50257), ("f32", 50257)])
@pytest.mark.parametrize("sliced", [True, False])
def test_spec_odd_rows_equal_padded_rows(dt, V, sliced):
    """An odd vocabulary's rows against the same rows with -inf appended to a
    multiple of 16 values (never kept, no weight): the same walk and tokens."""
    print(f"[row starts, spec {dt} V={V} sliced={sliced}]", flush=True)
    w = workloads.make_spec(seed=2, batch=9, vocab=V, k=3)
    ids = torch.randint(0, V, (9, 3), generator=torch.Generator().manual_seed(4))
    t, d = w.target.to(DT[dt]), w.draft.to(DT[dt])
    ids[:6] = d[:6].argmax(-1)  # (some drafts the target may accept)
    padded = [torch.nn.functional.pad(v, (0, 16 - V % 16), value=float("-inf")) for v in (t, d)]
    res = []
    for tt, dd in ((t, d), padded):
        p = SpecPlan(tt.cuda(), dd.cuda(), ids.cuda(), temperature=0.8, top_k=50, u_accept=w.u_accept.cuda(),
                     u_resample=w.u_resample.cuda(), sliced=sliced)
        p.launch()
        assert bool(p.status_ok().all())
        res.append((p.output.n_accepted.cpu(), p.output.tokens.cpu(), p.output.ratio.cpu().nan_to_num(-1.0)))
    for a, b in zip(*res):
        assert torch.equal(a, b)
