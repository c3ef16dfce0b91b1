"""Where a forward's scratch lies."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("lens,heads,kv_heads,B,topk", [
    ([4096], 4, 4, 512, 3),
    ([12704], 4, 1, 4096, 2),
    ([1001, 777], 6, 2, 100, 4),
])
def test_rows_start_on_lines(lens, heads, kv_heads, B, topk, train, monkeypatch):
    """The chunk representatives, the chunk mean's sums and the picks share allocations with other scratch; each starts at a
    multiple of 256 bytes, so that a representative of 128 elements is two whole lines."""
    from moba_amd import _lib, moba_attn_varlen_gqa
    lib, at = _lib.load(), {}
    mean, gate = lib.moba_chunk_mean, lib.moba_gate_topk
    monkeypatch.setattr(lib, "moba_chunk_mean", lambda *a: at.update(kbar=a[2], sums=a[3]) or mean(*a))
    monkeypatch.setattr(lib, "moba_gate_topk", lambda *a: at.update(picks=a[4]) or gate(*a))
    g = torch.Generator(device="cuda").manual_seed(0)
    S = sum(lens)
    q, k, v = (torch.randn((S, n, 128), generator=g, device="cuda").to(torch.bfloat16).requires_grad_(train)
               for n in (heads, kv_heads, kv_heads))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    print("scratch", lens, heads, kv_heads, B, topk, train, flush=True)
    moba_attn_varlen_gqa(q, k, v, cu, max(lens), B, topk)
    assert set(at) == {"kbar", "sums", "picks"} and all(a % 256 == 0 for a in at.values()), at
