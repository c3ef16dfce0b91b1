"""Tile tables that cut the lists of a key/value head's heads together: which rows share a tile changes no row's result."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,heads,kv_heads,B,topk,dtype", [
    ([1500], 6, 2, 100, 4, torch.bfloat16),               # 3 heads together, 24 list numbers a token: no power of two
    ([700, 65, 1, 1313], 7, 1, 64, 7, torch.float16),     # all of 7 heads, 49 a token
    ([2100, 900], 8, 4, 128, 2, torch.bfloat16),          # 16: a power of two
    ([1111], 5, 1, 37, 13, torch.float16),                # chunks of less than a key tile, 65 a token
])
def test_rows_of_several_heads(lens, heads, kv_heads, B, topk, dtype):
    """The token and the head of every list entry come from multiplications: outputs and dQ are bit for bit those of the
    same call with the key/value heads repeated, whose tiles are of one head each."""
    from moba_amd import moba_attn_varlen, moba_attn_varlen_gqa
    print("rows of several heads", lens, heads, kv_heads, B, topk, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads)
    S, rep = sum(lens), heads // kv_heads
    q, k, v, do = (torch.randn((S, n, 128), generator=g, device="cuda").to(dtype) for n in (heads, kv_heads, kv_heads, heads))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")

    def run(op, k, v):
        x = q.clone().requires_grad_(True)
        out = op(x, k, v, cu, max(lens), B, topk)
        out.backward(do)
        return out.detach(), x.grad

    got = run(moba_attn_varlen_gqa, k, v)
    want = run(moba_attn_varlen, k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1))
    for a, b in zip(got, want):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("lens,heads,kv_heads,B,topk,dtype", [
    ([4242], 8, 1, 512, 3, torch.bfloat16),               # tiles of 128 rows: forward and backward share their tables
    ([3000, 1200], 6, 3, 256, 4, torch.float16),
    ([20000], 4, 2, 1024, 3, torch.bfloat16),             # (with tall tiles below: the backward's tables only)
])
@pytest.mark.parametrize("tall", [False, True])
def test_either_side_of_the_rule(lens, heads, kv_heads, B, topk, dtype, tall, monkeypatch):
    """Lists cut head by head or together: the same outputs and gradients, bit for bit."""
    from moba_amd import moba_attn_varlen_gqa
    from moba_amd import moba_efficient as E
    from moba_amd import plan as P
    print("single heads or together", lens, heads, kv_heads, B, topk, dtype, tall, flush=True)
    if tall:
        monkeypatch.setattr(E, "forward_tile_rows", lambda *a: E.FWD_TILE_ROWS)
    g = torch.Generator(device="cuda").manual_seed(heads)
    S = sum(lens)
    x = [torch.randn((S, n, 128), generator=g, device="cuda").to(dtype) for n in (heads, kv_heads, kv_heads)]
    do = torch.randn((S, heads, 128), generator=g, device="cuda").to(dtype)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")

    def run(below):
        P._BY_VALUE.clear()   # (a plan keeps what was chosen for it)
        P._BY_TENSOR.clear()
        monkeypatch.setattr(E, "SHARED_LISTS_CHUNK", below)
        chosen, real = [], E._Geometry
        monkeypatch.setattr(E, "_Geometry", lambda *a: chosen.append(real(*a)) or chosen[-1])
        leaves = [t.clone().requires_grad_(True) for t in x]
        out = moba_attn_varlen_gqa(*leaves, cu, max(lens), B, topk)
        out.backward(do)
        monkeypatch.setattr(E, "_Geometry", real)
        assert {c.bwd_list_heads for c in chosen} == {heads // kv_heads if below else 1}
        return [out.detach()] + [t.grad for t in leaves]

    for a, b in zip(run(0), run(1 << 40)):
        assert torch.isfinite(a).all() and torch.equal(a, b)
