"""The dK/dV kernel's shares: with few key tiles the stages of all tiles of a key/value head are walked in equal shares, whose
sums a second kernel adds up."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,heads,kv_heads,B,topk,dtype", [
    ([1024], 1, 1, 128, 2, torch.bfloat16),              # the fewest tokens
    ([1023, 1], 1, 1, 1024, 3, torch.float16),           # no history; a tile of one key; shares fewer than units
    ([700, 65, 1, 513], 3, 1, 64, 4, torch.bfloat16),    # tiles of half a width, ragged ones, lists of three heads
    ([1111, 2222], 8, 1, 129, 2, torch.float16),         # a key tile of one key in every chunk
    ([5000], 14, 7, 1000, 3, torch.bfloat16),            # shares that do not divide the units, ragged stages
    ([1024], 126, 63, 256, 2, torch.bfloat16),           # as many heads as there can be: more than one tile per unit and head
])
def test_shares_of_key_tiles(lens, heads, kv_heads, B, topk, dtype, monkeypatch):
    """Whatever the layout of q (packed rows, a slice of a wider tensor) the same sums bit for bit, and those of whole tiles
    up to the order of fp32 additions: rounded once either way, so values only move across a rounding boundary (in norm far
    below half a step of the type, 2^-9 or 2^-12; no element by more than a step of the largest)."""
    from moba_amd import _lib, moba_attn_varlen_gqa
    from moba_amd import plan as P
    lib = _lib.load()
    print("shares", lens, heads, kv_heads, B, topk, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads)
    S = sum(lens)
    q, k, v, do = (torch.randn((S, n, 128), generator=g, device="cuda").to(dtype) for n in (heads, kv_heads, kv_heads, heads))
    slice_of = torch.zeros((S, heads + 1, 128), device="cuda", dtype=dtype)[:, 1:]
    slice_of.copy_(q)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")

    def run(qq):   # (a new plan each time: a plan keeps the sizes of its scratch)
        P._BY_VALUE.clear()
        P._BY_TENSOR.clear()
        kg, vg = (x.clone().requires_grad_(True) for x in (k, v))
        moba_attn_varlen_gqa(qq, kg, vg, cu_t, max(lens), B, topk).backward(do)
        return kg.grad, vg.grad

    real, asked = lib.moba_bwd_dkv_shares, []
    monkeypatch.setattr(lib, "moba_bwd_dkv_shares", lambda *a: asked.append(real(*a)) or asked[-1])
    shares, again, strided = run(q), run(q), run(slice_of)
    assert asked[0] > 0
    for a, b, c in zip(shares, again, strided):
        assert torch.equal(a, b) and torch.equal(a, c)
    monkeypatch.setattr(lib, "moba_bwd_dkv_shares", lambda *a: 0)
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for a, b in zip(shares, run(q)):
        a, b = a.float(), b.float()
        assert torch.isfinite(a).all()
        assert (a - b).norm() < step / 2 * b.norm() and (a - b).abs().max() <= 2 * step * b.abs().max()


def test_no_shares_beyond_32_bits():
    """What moba_bwd would refuse for its number of stages gets no shares in the first place."""
    from moba_amd import _lib
    lib = _lib.load()
    assert lib.moba_bwd_dkv_shares(65280, 8, 1, 510) > 0
    assert lib.moba_bwd_dkv_shares(65280, 4200, 1, 510) == 0
    assert lib.moba_bwd_dkv_shares(65280, 4200, 4200, 510) == 0 and lib.moba_bwd_dkv_shares(65280, 7, 2, 100) == 0
