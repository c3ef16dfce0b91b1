"""The gate's two arrangements of a workgroup (four heads of 64 tokens, or 256 tokens of a head): picks and counts at the
edges of both, against the oracle (GPU only)."""

import numpy as np
import pytest
import torch

from oracle import moba_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,heads,B,topk", [
    ([255], 1, 64, 3), ([256, 256], 2, 64, 3), ([257, 700], 4, 64, 3),      # around a workgroup's 256 tokens
    ([1023, 1, 513], 3, 256, 4), ([300, 40, 2000], 1, 128, 4),               # sequences that end inside them
    ([4200], 2, 64, 3), ([4200], 1, 32, 36),                                 # more than 64 candidates; lists too long to be staged
    ([13107], 5, 512, 3), ([13200], 5, 512, 3),                              # either side of the line for more than 4 heads
    ([13200, 300], 6, 64, 36)])
def test_picks_and_counts(lens, heads, B, topk):
    from moba_amd import moba_efficient as E
    print("gate", lens, heads, B, topk, flush=True)
    cu = [0, *np.cumsum(lens).tolist()]
    g = torch.Generator().manual_seed(sum(lens) + heads)
    q, k = (torch.randn((cu[-1], heads, 128), generator=g).to(torch.bfloat16) for _ in range(2))
    plan = E.make_plan(cu, B, topk, device="cuda")
    buffers = E.list_buffers(plan, heads, torch.device("cuda"))
    kbar = E.chunk_mean(k.cuda(), plan, clear=buffers[0])
    sel, scores = E.gate_topk(q.cuda(), kbar, plan, return_scores=True)
    assert torch.equal(E.gate_topk(q.cuda(), kbar, plan, cnt=buffers[0]), sel)
    lists = E.build_lists(sel, plan, buffers=buffers, counted=True)
    sel, scores = sel.cpu(), scores.cpu()
    assert (scores - O.gate_scores(q, kbar.cpu(), cu, B)).abs().nan_to_num(0).max() < 1e-4
    picks = torch.sort(torch.where(sel < 0, 1 << 30, sel), dim=-1).values
    assert torch.equal(torch.where(picks == 1 << 30, -1, picks), O.select_topk(scores, plan.K))
    counts, offs, rows, slots = O.gather_lists(sel, plan.F)
    assert np.array_equal(lists[0].cpu().numpy(), offs)
    dest = (rows * heads + np.repeat(np.arange(plan.F * heads) % heads, counts)) * (plan.K + 1) + 1 + slots
    assert np.array_equal(lists[2].cpu().numpy()[:offs[-1]], dest)
