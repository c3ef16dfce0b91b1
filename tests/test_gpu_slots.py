"""Rows put together from their slots, by the forms for a constant number of slots and by the general one: the merge of the
forward's partial results and the sum of the partial dQ (GPU only)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,dim", [(torch.bfloat16, 128), (torch.float16, 64)])
@pytest.mark.parametrize("H", [1, 3])
@pytest.mark.parametrize("slots,parts", [(1, 1), *((n, 1) for n in (*range(2, 14), 36, 38, 40, 42, 44, 65)), (2, 2), (3, 2), (4, 2), (5, 2), (6, 2), (7, 2),
                                         (2, 4), (3, 4), (4, 4), (2, 8)])
def test_merge_of_token_ranges(slots, parts, H, dtype, dim):
    """Random partial results and statistics, a third of the history slots absent (and poisoned), merged for the tokens of
    ranges that end within a wave's four rows; the rows of other tokens stay as they are."""
    from moba_amd import _lib
    print("merge", slots, parts, H, dtype, dim, flush=True)
    lib, S, K = _lib.load(), 203, slots - 1
    g = torch.Generator().manual_seed(100 * slots + 10 * parts + H)
    po = torch.randn((parts, S * H, slots, dim), generator=g).to(dtype)
    lse = torch.randn((parts, S * H, slots), generator=g) * 6
    sel = torch.randint(0, 50, (S, H, max(K, 1)), generator=g, dtype=torch.int32)
    sel[torch.rand(sel.shape, generator=g) < 0.33] = -1
    absent = torch.cat([torch.zeros((S * H, 1), dtype=torch.bool), (sel < 0).view(S * H, -1)[:, :K]], dim=1).repeat(parts, 1, 1)
    absent[1:, :, 0] = True
    x, l = po.double().masked_fill(absent[..., None], 0), lse.double().masked_fill(absent, -math.inf)
    w = l - torch.logsumexp(l, dim=(0, 2), keepdim=True)
    want, want_lse = (w.exp()[..., None] * x).sum(dim=(0, 2)), torch.logsumexp(l, dim=(0, 2))
    po[absent] = math.nan
    log2 = (lse / math.log(2)).masked_fill(absent, math.nan).float()
    start, lens = torch.tensor([3, 10, 60, 101], dtype=torch.int32), [2, 1, 37, 102]
    prefix = torch.tensor([0, 2, 3, 40, 142], dtype=torch.int32)
    out = torch.full((S * H, dim), 7.0, dtype=dtype, device="cuda")
    out_lse = torch.full((S * H,), 7.0, device="cuda")
    bufs = [t.cuda() for t in (po, log2, sel[..., :K].contiguous() if K else sel, start, prefix)]
    p = [t.data_ptr() for t in bufs]
    _lib.check(lib.moba_fwd_merge(p[0], p[1], p[2] if K else None, out.data_ptr(), out_lse.data_ptr(), S, H, dim, K, parts, p[3],
                                  p[4], 4, 142, _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16,
                                  torch.cuda.current_stream().cuda_stream), "moba_fwd_merge")
    walked = torch.zeros((S, H), dtype=torch.bool)
    for a, n in zip(start.tolist(), lens):
        walked[a:a + n] = True
    walked = walked.view(-1)
    out, out_lse = out.cpu().double(), out_lse.cpu().double()
    assert bool((out[~walked] == 7).all()) and bool((out_lse[~walked] == 7).all())
    # the result's rounding (to 8 and 11 significant bits: half a unit of the last is up to 2^-8 and 2^-11 of the value), and
    # fp32 sums of values up to about 5 by weights that are off by up to 2^-19 (exponentials of differences up to 60, 2^-24 of that)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert bool(((out - want)[walked].abs() <= unit * want[walked].abs() + 5 * 2.0 ** -18).all())
    assert (out_lse - want_lse)[walked].abs().max() < 2e-5


@pytest.mark.parametrize("topk,heads,dense", [(t, 1 + t % 3, bool(t & 1)) for t in range(2, 15)])
def test_results_and_gradients_by_slots(topk, heads, dense):
    """Forward and backward with every number of slots, five sequences, against the oracle."""
    from test_gpu_operator import run_case
    print("slots", topk, heads, dense, flush=True)
    run_case(5, 2400, heads, 30, topk, seed=topk, ref_bounds=False, dense=dense)


@pytest.mark.parametrize("dtype,dim", [(torch.bfloat16, 128), (torch.float16, 64)])
@pytest.mark.parametrize("slots,parts", [(2, 1), (3, 1), (8, 1), (9, 1), (12, 1), (3, 2), (6, 2), (2, 4), (3, 4)])
def test_slots_without_weight(slots, parts, dtype, dim):
    """A slot whose weight is 0 (its statistic lies 300 below another's) takes no part in its row, whatever its partial result
    holds: an infinite value of one key stays with the rows that see it."""
    from moba_amd import _lib
    print("no weight", slots, parts, dtype, dim, flush=True)
    lib, S, K = _lib.load(), 37, slots - 1
    g = torch.Generator().manual_seed(slots + parts)
    po = torch.randn((parts, S, slots, dim), generator=g).to(dtype)
    log2 = torch.randn((parts, S, slots), generator=g)
    none = torch.zeros((parts, S, slots), dtype=torch.bool)
    none[parts - 1, 0::3, slots - 1] = True    # a history slot, the last part of it,
    none[0, 1::3, 0] = True                    # the self slot, or none
    log2[none] -= 300
    weights = log2.double().exp2()
    weights[1:, :, 0] = 0                      # (the self slot has part 0 only)
    weights[none] = 0
    want = (weights[..., None] * po.double()).sum(dim=(0, 2)) / weights.sum(dim=(0, 2))[:, None]
    want_lse = weights.sum(dim=(0, 2)).log()
    values = torch.tensor([math.inf, -math.inf, math.nan], dtype=dtype)
    po[none] = values[torch.arange(dim) % 3]
    sel = torch.zeros((S, K), dtype=torch.int32)
    bufs = [t.cuda() for t in (po, log2.float(), sel)]
    out, lse = torch.empty((S, dim), dtype=dtype, device="cuda"), torch.empty((S,), device="cuda")
    p = [t.data_ptr() for t in bufs]
    _lib.check(lib.moba_fwd_merge(p[0], p[1], p[2], out.data_ptr(), lse.data_ptr(), S, 1, dim, K, parts, None, None, 0, S,
                                  _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16,
                                  torch.cuda.current_stream().cuda_stream), "moba_fwd_merge")
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)   # (as above)
    assert bool(((out.cpu().double() - want).abs() <= unit * want.abs() + 5 * 2.0 ** -18).all())
    assert (lse.cpu().double() - want_lse).abs().max() < 2e-5
