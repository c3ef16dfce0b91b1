"""The gate's two arrangements of a workgroup (four heads of 64 tokens, or 256 tokens of a head): picks and counts at the
edges of both, against the oracle (GPU only)."""

import numpy as np
import pytest
import torch

from oracle import moba_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,heads,B,topk,dim,kv_heads", [(*case, 128, 0)[:6] for case in [
    # by heads: three heads in four waves and more, around a wave's 64 tokens
    ([255], 1, 64, 3), ([256, 256], 2, 64, 3), ([257, 700], 4, 64, 3), ([1023, 1, 513], 3, 256, 4), ([300, 40, 2000], 1, 128, 4),
    # more than 64 candidates; lists too long to be staged
    ([4200], 2, 64, 3), ([4200], 1, 32, 36), ([13107], 5, 512, 3), ([13200], 5, 512, 3), ([13200, 300], 6, 64, 36),
    # by tokens, for the additions: around a workgroup's 256 tokens, sequences that end inside them
    ([767], 1, 512, 3), ([1024], 2, 512, 3), ([1025], 4, 512, 3), ([1300, 700, 2049], 3, 512, 4), ([600, 1100], 7, 512, 3),
    # a workgroup's joint histogram: 63 and 64 earlier chunks, and beyond them each wave's own
    ([33900], 1, 512, 3), ([17000, 16700], 1, 256, 3),
    # by tokens, for waves without a head: either side of the 1024 waves, more than 64 candidates, lists too long to be staged
    ([16384], 1, 128, 3), ([16385], 1, 128, 3), ([16700], 1, 256, 3), ([16800], 3, 64, 36), ([5462], 9, 128, 3),
    # four heads: either side of the line for their longer kernels
    ([32768], 4, 512, 3), ([32769], 4, 512, 3),
    # 64-element heads, grouped-query heads: both arrangements
    ([1100, 130], 8, 128, 4, 64, 2), ([1300, 700], 8, 512, 4, 64, 2), ([2500], 6, 128, 3, 128, 3), ([2500], 6, 512, 3, 128, 2),
    ([16500], 2, 128, 3, 64, 1)]])
def test_picks_and_counts(lens, heads, B, topk, dim, kv_heads):
    from moba_amd import moba_efficient as E
    print("gate", lens, heads, B, topk, dim, kv_heads, flush=True)
    cu = [0, *np.cumsum(lens).tolist()]
    g = torch.Generator().manual_seed(sum(lens) + heads)
    q, k = (torch.randn((cu[-1], h, dim), generator=g).to(torch.bfloat16) for h in (heads, kv_heads or heads))
    plan = E.make_plan(cu, B, topk, device="cuda")
    buffers = E.list_buffers(plan, heads, torch.device("cuda"))
    kbar = E.chunk_mean(k.cuda(), plan, clear=buffers[0])
    sel, scores = E.gate_topk(q.cuda(), kbar, plan, return_scores=True)
    assert torch.equal(E.gate_topk(q.cuda(), kbar, plan, cnt=buffers[0]), sel)
    lists = E.build_lists(sel, plan, buffers=buffers, counted=True)
    sel, scores = sel.cpu(), scores.cpu()
    of_heads = kbar.cpu().repeat_interleave(heads // kbar.shape[1], dim=1)
    assert (scores - O.gate_scores(q, of_heads, cu, B)).abs().nan_to_num(0).max() < 1e-4
    picks = torch.sort(torch.where(sel < 0, 1 << 30, sel), dim=-1).values
    assert torch.equal(torch.where(picks == 1 << 30, -1, picks), O.select_topk(scores, plan.K))
    counts, offs, rows, slots = O.gather_lists(sel, plan.F)
    assert np.array_equal(lists[0].cpu().numpy(), offs)
    dest = (rows * heads + np.repeat(np.arange(plan.F * heads) % heads, counts)) * (plan.K + 1) + 1 + slots
    assert np.array_equal(lists[2].cpu().numpy()[:offs[-1]], dest)
