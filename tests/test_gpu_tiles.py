"""The two tile heights of the forward attention kernel against each other and against the dense oracle: 128 rows, one
workgroup per tile (short chunks and short calls), and 256 rows, by resident workgroups or one workgroup each."""

import numpy as np
import pytest
import torch

from oracle import moba_oracle as O
from test_gpu_queued import test_queued_kernels_against_the_dense_oracle as queued_case

pytestmark = pytest.mark.gpu


@pytest.fixture
def tile_rows(monkeypatch):
    """Sets the tile height; plans keep what was derived from it, so their caches start and end empty."""
    from moba_amd import moba_efficient as E
    from moba_amd import plan as P

    def forget():
        P._BY_VALUE.clear()
        P._BY_TENSOR.clear()

    def choose(rows):
        monkeypatch.setattr(E, "forward_tile_rows", lambda plan, H, D=128: rows)
        forget()

    yield choose
    forget()


@pytest.mark.parametrize("dense,dtype,spread", [(True, torch.bfloat16, 1.0), (False, torch.bfloat16, 8.0),
                                                (True, torch.float16, 8.0)])
def test_resident_workgroups_against_the_dense_oracle(dense, dtype, spread, tile_rows, monkeypatch):
    """The shape of the queued kernels' test, whose chunks are short, on the resident workgroups all the same."""
    tile_rows(256)
    queued_case(dense, dtype, spread, monkeypatch)


@pytest.mark.parametrize("lens,heads,kv_heads,B,topk,dtype", [
    ([128], 1, 1, 64, 2, torch.bfloat16),
    ([129, 127, 1, 257], 2, 1, 65, 3, torch.float16),      # one-row tiles, a key tile of one key
    ([640, 63], 3, 3, 128, 2, torch.bfloat16),
    ([2048], 4, 2, 512, 1, torch.float16),                 # full causal attention
    ([4096], 1, 1, 2048, 3, torch.bfloat16),               # history tiles cut along their keys
    ([3000], 2, 2, 192, 3, torch.bfloat16),
])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_tile_heights_agree(lens, heads, kv_heads, B, topk, dtype, spread, tile_rows):
    """A row's result does not depend on the tile it lies in (bit for bit) unless some row of a tile leaves the range of
    the fixed-reference softmax (spread 8): the two softmax forms then differ by their roundings, at most a few of the
    element type's steps at values of up to about 4."""
    from moba_amd import moba_efficient as E
    cu = [0] + np.cumsum(lens).tolist()
    S = cu[-1]
    print("tile case", lens, heads, B, topk, dtype, spread, flush=True)
    g = torch.Generator().manual_seed(S + heads)
    q = (torch.randn((S, heads, 128), generator=g) * spread).to(dtype).cuda()
    k = (torch.randn((S, kv_heads, 128), generator=g) * spread).to(dtype).cuda()
    v = torch.randn((S, kv_heads, 128), generator=g).to(dtype).cuda()
    got = []
    for rows in (128, 256):
        tile_rows(rows)
        cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")
        got.append(E.moba_attn_varlen_with_lse(q, k, v, cu_t, max(lens), B, topk, gqa=True))
    (out_a, lse_a), (out_b, lse_b) = got
    assert torch.isfinite(out_a.float()).all() and torch.isfinite(lse_a).all()
    if spread == 1.0 and not (len(lens) == 1 and B == 2048):   # (parts: their number follows from the number of tiles)
        assert torch.equal(out_a, out_b) and torch.equal(lse_a, lse_b)
    else:
        step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        assert (out_a.float() - out_b.float()).abs().max() < 4 * 4 * step
        assert (lse_a - lse_b).abs().max() < 1e-3 * max(1.0, spread * spread)


@pytest.mark.parametrize("lens,heads,kv_heads,B,topk,dtype", [
    ([128], 1, 1, 64, 2, torch.bfloat16),
    ([129, 127, 1, 257], 2, 1, 65, 3, torch.float16),
    ([2048], 4, 2, 512, 1, torch.float16),
    ([4096], 1, 1, 2048, 3, torch.bfloat16),
    ([3000], 5, 1, 192, 13, torch.bfloat16),
])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_heads_of_64_are_those_of_128_padded(lens, heads, kv_heads, B, topk, dtype, spread, tile_rows):
    """The forward's kernels for 64-element heads form the same sums as those for 128 on zero-padded heads (zeros add
    nothing): selection, output and log-sum-exp bit for bit, on the packed and on the batched layout."""
    from moba_amd import moba_efficient as E
    cu = [0] + np.cumsum(lens).tolist()
    S = cu[-1]
    print("narrow case", lens, heads, B, topk, dtype, spread, flush=True)
    g = torch.Generator().manual_seed(S + heads)
    q = (torch.randn((S, heads, 64), generator=g) * spread).to(dtype).cuda()
    k = (torch.randn((S, kv_heads, 64), generator=g) * spread).to(dtype).cuda()
    v = torch.randn((S, kv_heads, 64), generator=g).to(dtype).cuda()
    tile_rows(128)
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = E.moba_attn_varlen_with_lse(q, k, v, cu_t, max(lens), B, topk, gqa=True)
    wide = [torch.nn.functional.pad(x, (0, 64)) for x in (q, k, v)]
    want, want_lse = E._attend(*wide, E.make_plan(cu_t, B, topk), None, 64 ** -0.5)
    assert out.shape == q.shape and torch.isfinite(out.float()).all()
    assert torch.equal(out, want[..., :64]) and torch.equal(lse, want_lse)
    if len(lens) == 1:
        one = E.moba_attn_batched(*(x.transpose(0, 1)[None] for x in (q, k, v)), B, topk)
        assert torch.equal(one, out)


@pytest.mark.parametrize("rows", [128, 256])
def test_overflow_in_any_dimension_is_found(rows, tile_rows):
    """Probabilities of 2^68 to 2^96 (relative to the fixed reference) times values of 2^60 leave fp32 in the accumulators of
    some dimensions only: v is zero in dimensions 0 and 4 of every 32, those of the first accumulator registers.  Such
    tiles have to be computed again with a running maximum all the same; scaling v by a power of two scales the result."""
    from moba_amd import moba_efficient as E
    S, H, B, topk = 32768, 8, 1024, 3
    print("overflow case", rows, flush=True)
    g = torch.Generator(device="cuda").manual_seed(17)
    q, k, v = (torch.randn((S, H, 128), generator=g, device="cuda") for _ in range(3))
    q, k, v = (q * 4.5).to(torch.bfloat16), (k * 4.5).to(torch.bfloat16), v.to(torch.bfloat16)
    v[..., 0::32] = 0
    v[..., 4::32] = 0
    tile_rows(rows)
    cu_t = torch.tensor([0, S], dtype=torch.int32, device="cuda")
    small = E.moba_attn_varlen(q, k, v, cu_t, S, B, topk)
    large = E.moba_attn_varlen(q, k, (v.float() * 2.0 ** 60).to(torch.bfloat16), cu_t, S, B, topk)
    assert torch.isfinite(large.float()).all()
    err = (large.float() * 2.0 ** -60 - small.float()).abs()
    # Near one-hot rows: values of up to about 4.5 on both sides, each rounded to 8 bits three times (probabilities,
    # partial result, result): 2 * 3 * 2^-9 * 4.5 = 5.3e-2 at most; in the mean (values of about 0.8, roundings of either
    # sign, half a rounding on average) below 2 * 3 * 2^-10 * 0.8 = 4.7e-3.
    assert err.max() < 5.3e-2 and err.mean() < 4.7e-3, (err.max().item(), err.mean().item())


@pytest.mark.parametrize("S,H,B,D", [
    (20, 3, 1, 128), (50, 1, 7, 64), (900, 2, 127, 128), (1100, 2, 300, 128), (2400, 1, 777, 64),   # fewer and more than
    (9000, 1, 4096, 128), (5000, 4, 1024, 128),          # eight tokens per lane; one workgroup of 1024, a chunk that needs two stages
    (3000, 37, 100, 128), (33000, 2, 8, 128), (8200, 9, 8, 64),   # many workgroups; very many short chunks (two stages)
])
def test_chunk_mean_forms(S, H, B, D):
    """Every form of the chunk mean gives the rounded exact mean, whatever its number of threads and token lanes."""
    from moba_amd import moba_efficient as E
    print("mean case", S, H, B, D, flush=True)
    g = torch.Generator().manual_seed(S)
    k = torch.randn((S, H, D), generator=g).to(torch.bfloat16)
    plan = E.make_plan([0, S], B, 3, device="cuda")
    want = O.chunk_mean(k, [0, S], B)
    clear = torch.full((1000,), 7, dtype=torch.int32, device="cuda")
    got = E.chunk_mean(k.cuda(), plan, clear=clear)
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16)) and int(clear.abs().max()) == 0
    strided = k.transpose(0, 1).contiguous().cuda().transpose(0, 1)      # [heads, tokens, dim] seen token-first
    assert torch.equal(E.chunk_mean(strided, plan), got)


def test_list_of_tiles_computed_again_is_bounded(tile_rows, monkeypatch):
    """With history tiles cut along their keys more parts than tiles can leave the fixed reference's range: they are all
    counted, and nothing is written behind the list (here, and in every call, the end of the scratch allocation)."""
    from moba_amd import moba_efficient as E
    S, H, B, topk = 8192, 1, 4096, 2
    tile_rows(128)
    cu_t = torch.tensor([0, S], dtype=torch.int32, device="cuda")
    plan = E.make_plan(cu_t, B, topk)
    g = E._geometry(plan, E._lib.load(), H, 128, 2)
    entries = g.scratch_ints - 9
    guard = g.split * (g.bound + g.self_tiles) * 4
    assert g.split * (S - B) // 128 > entries     # (every token of the second chunk attends the first: full tiles)
    monkeypatch.setattr(g, "ws_bytes", g.ws_bytes + guard)
    monkeypatch.setattr(E, "KEEP_SCRATCH", True)
    # scores that rise along the keys: every part's first 32 keys are far below its last ones
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn((S, H, 128), generator=gen, device="cuda") for _ in range(3))
    q = q.abs() + 1
    k = k * 0.1 + torch.arange(S, device="cuda")[:, None, None] % 512 * (8.0 / 512)
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    torch.use_deterministic_algorithms(True)
    try:
        E._run_forward(q, k, v, plan)
    finally:
        torch.use_deterministic_algorithms(False)
    redo = E.last_scratch["redo"]
    whole = torch.empty(0, dtype=torch.uint8, device="cuda").set_(redo.untyped_storage())
    torch.cuda.synchronize()
    assert redo[0] > entries, (redo[0].item(), entries)
    assert redo[1:].min() >= 0 and redo[1:].max() < g.bound + g.self_tiles * H
    assert (whole[g.ws_bytes - guard:g.ws_bytes] == 255).all()


@pytest.mark.parametrize("lens,heads,D,B,topk,rows", [
    ([3000], 2, 128, 192, 3, 128), ([3000], 2, 128, 192, 3, 256), ([700, 2333], 3, 64, 256, 4, 128),
    ([4096], 1, 128, 2048, 3, 128),                  # history tiles cut along their keys
    ([8155, 7777, 8192, 6013, 8000, 8492], 4, 128, 512, 4, 256),    # resident workgroups
])
def test_running_maximum_from_the_start(lens, heads, D, B, topk, rows, tile_rows, monkeypatch):
    """The switch for the running maximum reaches every form of the forward.  Scores rise by up to 2^40 above a row's first
    32 keys: inside the fixed reference's range, so that no tile is computed again, but beyond the 2^8 by which the running
    maximum may lag, so that its probabilities are rounded elsewhere: the two agree as far as roundings go (probabilities, partial
    result and result, to half a step at values of up to about 4.5 each), and not bit for bit."""
    from moba_amd import moba_efficient as E
    cu = [0] + np.cumsum(lens).tolist()
    print("switch case", lens, heads, D, B, topk, rows, flush=True)
    tile_rows(rows)
    g = torch.Generator().manual_seed(cu[-1])
    q, k, v = (torch.randn((cu[-1], heads, D), generator=g) * s for s in (3.0, 2.0, 1.0))
    q, k, v = (x.to(torch.bfloat16).cuda() for x in (q, k, v))
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")
    outs = []
    for fixed in (True, False):
        monkeypatch.setattr(E, "FIXED_REFERENCE", fixed)
        outs.append(E.moba_attn_varlen_with_lse(q, k, v, cu_t, max(lens), B, topk))
    (out_f, lse_f), (out_r, lse_r) = outs
    err = (out_f.float() - out_r.float()).abs()
    assert not torch.equal(out_f, out_r) and err.max() < 2 * 3 * 4.5 * 2.0 ** -9 and err.mean() < 2 * 3 * 0.8 * 2.0 ** -10
    assert (lse_f - lse_r).abs().max() < 1e-3


@pytest.mark.parametrize("q_len,resident", [(600, 1 << 30), (600, 0), (300, 1 << 30)])
def test_running_maximum_of_new_tokens(q_len, resident, monkeypatch):
    """The same for new tokens against a cache, on both routes of the causal tiles."""
    from moba_amd import moba_efficient as E
    import moba_amd.decode as D
    g = torch.Generator().manual_seed(q_len)
    q, k, v = (torch.randn((1, 16, n, 128), generator=g) * s for n, s in ((q_len, 3.0), (1000, 2.0), (1000, 1.0)))
    q, k, v = (x.to(torch.bfloat16).cuda() for x in (q, k, v))
    monkeypatch.setattr(D, "RESIDENT_TILES", resident)
    monkeypatch.setattr(D, "_takes_tiles", lambda *a: True)
    outs = []
    for fixed in (True, False):
        monkeypatch.setattr(E, "FIXED_REFERENCE", fixed)
        outs.append(D.chunk_decode_attention(q, k, v).float())
    err = (outs[0] - outs[1]).abs()
    assert err.max() > 0 and err.max() < 2 * 3 * 4.5 * 2.0 ** -9 and err.mean() < 2 * 3 * 0.8 * 2.0 ** -10


def test_short_tiles_need_no_queues(tile_rows, monkeypatch):
    """The tiles with a workgroup each draw nothing from queues: the C entry takes none."""
    from moba_amd import _lib
    from moba_amd import moba_efficient as E
    lib = _lib.load()

    class WithoutQueues:
        def __getattr__(self, name):
            if name != "moba_fwd_partials_rows":
                return getattr(lib, name)
            return lambda *a: lib.moba_fwd_partials_rows(*a[:28], None, *a[29:])

    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn((900, 2, 128), generator=g).to(torch.bfloat16).cuda() for _ in range(3))
    cu_t = torch.tensor([0, 900], dtype=torch.int32, device="cuda")
    tile_rows(128)
    want = E.moba_attn_varlen(q, k, v, cu_t, 900, 128, 3)
    monkeypatch.setattr(_lib, "load", lambda: WithoutQueues())
    assert torch.equal(E.moba_attn_varlen(q, k, v, cu_t, 900, 128, 3), want)


@pytest.mark.parametrize("S,H,B,D", [
    (6200, 1, 2048, 128), (6200, 4, 2048, 128), (6200, 5, 2048, 128), (3200, 1, 1025, 128), (3200, 1, 1024, 128),
    (9000, 1, 2049, 64), (9000, 3, 2900, 64), (134000, 1, 2050, 128)])
def test_chunk_mean_at_the_line_between_its_forms(S, H, B, D):
    """Few chunks on either side of the line between one workgroup each and two stages: the rounded exact mean."""
    from moba_amd import moba_efficient as E
    print("mean line", S, H, B, D, flush=True)
    k = torch.randn((S, H, D), generator=torch.Generator().manual_seed(S + H)).to(torch.bfloat16)
    want = O.chunk_mean(k, [0, S], B)
    got = E.chunk_mean(k.cuda(), E.make_plan([0, S], B, 3, device="cuda"))
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16))
