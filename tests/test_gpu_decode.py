"""Decode attention kernel (one query token against the key/value cache) against an fp32
softmax on the same inputs; through the C ABI, and through the adapter's decode branch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(q, k, v, scale):
    rep = q.shape[1] // k.shape[1]
    kk = k.float().repeat_interleave(rep, dim=1)
    vv = v.float().repeat_interleave(rep, dim=1)
    p = torch.softmax((q.float() @ kk.transpose(-1, -2)) * scale, dim=-1)
    return (p @ vv).transpose(1, 2)            # [B, 1, H, D]


@pytest.mark.parametrize("B,H,Hkv,Skv,dtype", [
    (1, 32, 8, 131072, torch.bfloat16),
    (2, 8, 8, 1000, torch.bfloat16),
    (3, 16, 2, 4097, torch.float16),
    (1, 4, 2, 1, torch.bfloat16),
    (5, 2, 1, 37, torch.float16),
    (4, 32, 8, 777, torch.bfloat16),
])
def test_decode_matches_softmax(B, H, Hkv, Skv, dtype):
    from moba_amd.decode import decode_attention
    print("decode case", B, H, Hkv, Skv, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q = torch.randn((B, H, 1, 128), generator=g, device="cuda").to(dtype)
    k = torch.randn((B, Hkv, Skv, 128), generator=g, device="cuda").to(dtype)
    v = torch.randn((B, Hkv, Skv, 128), generator=g, device="cuda").to(dtype)
    for scale in (None, 0.2):
        out = decode_attention(q, k, v, scale)
        want = _ref(q, k, v, 128 ** -0.5 if scale is None else scale)
        assert out.shape == (B, 1, H, 128)
        err = (out.float() - want).abs()
        assert err.max() < 1e-2 and err.mean() < 1e-3, (err.max().item(), err.mean().item())


def test_decode_reads_a_cache_view_in_place():
    """A preallocated cache [B, Hkv, Smax, D] sliced to the filled length: strided, not copied."""
    from moba_amd.decode import decode_attention
    g = torch.Generator(device="cuda").manual_seed(1)
    cache_k = torch.randn((2, 4, 512, 128), generator=g, device="cuda").to(torch.bfloat16)
    cache_v = torch.randn((2, 4, 512, 128), generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn((2, 8, 1, 128), generator=g, device="cuda").to(torch.bfloat16)
    k, v = cache_k[:, :, :300], cache_v[:, :, :300]
    assert not k.is_contiguous()
    out = decode_attention(q, k, v)
    err = (out.float() - _ref(q, k, v, 128 ** -0.5)).abs()
    assert err.max() < 1e-2


def test_adapter_decode_branch_uses_the_kernel_and_agrees_with_sdpa():
    from moba_amd import MoBAConfig, moba_attn_varlen
    from moba_amd.moba_naive import moba_attn_varlen_naive
    from moba_amd.wrapper import moba_layer

    class Mod(torch.nn.Module):
        is_causal = True

    g = torch.Generator(device="cuda").manual_seed(2)
    q = torch.randn((2, 8, 1, 128), generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn((2, 2, 333, 128), generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn((2, 2, 333, 128), generator=g, device="cuda").to(torch.bfloat16)
    cfg = MoBAConfig(64, 3)
    a, _ = moba_layer(moba_attn_varlen, cfg, Mod(), q, k, v, None)          # HIP decode kernel
    b, _ = moba_layer(moba_attn_varlen_naive, cfg, Mod(), q, k, v, None)    # SDPA
    assert a.shape == b.shape == (2, 1, 8, 128)
    assert (a.float() - b.float()).abs().max() < 2e-2


def _ref_tail(q, k, v, scale):
    """fp32 attention of the last q_len tokens: token j sees the keys up to position Skv - q_len + j."""
    rep = q.shape[1] // k.shape[1]
    kk = k.float().repeat_interleave(rep, dim=1)
    vv = v.float().repeat_interleave(rep, dim=1)
    q_len, skv = q.shape[2], k.shape[2]
    logits = (q.float() @ kk.transpose(-1, -2)) * scale                          # [B, H, q_len, Skv]
    pos = torch.arange(q_len, device=q.device)[:, None] + (skv - q_len)
    logits = logits.masked_fill(torch.arange(skv, device=q.device)[None, :] > pos, float("-inf"))
    return (torch.softmax(logits, dim=-1) @ vv).transpose(1, 2)                  # [B, q_len, H, D]


@pytest.mark.parametrize("B,H,Hkv,Skv,q_len,dtype", [
    (2, 8, 2, 1000, 2, torch.bfloat16),       # a few tokens: the decode kernel per token
    (1, 32, 8, 20000, 16, torch.bfloat16),
    (3, 4, 4, 333, 7, torch.float16),
    (2, 6, 2, 1000, 5, torch.bfloat16),       # three query heads per key/value head: the causal tiles
    (2, 8, 2, 1000, 17, torch.bfloat16),      # more tokens: the forward kernel's causal tiles on the tail
    (1, 8, 8, 5000, 300, torch.float16),
    (2, 16, 4, 4097, 1025, torch.bfloat16),
    (1, 4, 2, 700, 699, torch.bfloat16),
    (1, 32, 8, 40000, 4096, torch.bfloat16),  # enough tiles for the resident-workgroup kernel
])
def test_several_new_tokens_against_the_cache(B, H, Hkv, Skv, q_len, dtype):
    from moba_amd.decode import chunk_decode_attention
    print("tail case", B, H, Hkv, Skv, q_len, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(Skv + q_len)
    q = torch.randn((B, H, q_len, 128), generator=g, device="cuda").to(dtype)
    cache_k = torch.randn((B, Hkv, Skv + 50, 128), generator=g, device="cuda").to(dtype)
    cache_v = torch.randn((B, Hkv, Skv + 50, 128), generator=g, device="cuda").to(dtype)
    k, v = cache_k[:, :, :Skv], cache_v[:, :, :Skv]       # a preallocated cache sliced to its filled length
    for scale in (None, 0.15):
        out = chunk_decode_attention(q, k, v, scale)
        want = _ref_tail(q, k, v, 128 ** -0.5 if scale is None else scale)
        assert out.shape == (B, q_len, H, 128) and torch.isfinite(out.float()).all()
        err = (out.float() - want).abs()
        assert err.max() < 2e-2 and err.mean() < 1e-3, (err.max().item(), err.mean().item())


def test_adapter_decodes_several_tokens_with_the_kernels():
    from moba_amd import MoBAConfig, moba_attn_varlen
    from moba_amd.moba_naive import moba_attn_varlen_naive
    from moba_amd.wrapper import moba_layer
    import moba_amd.decode as D

    class Mod(torch.nn.Module):
        is_causal = True

    g = torch.Generator(device="cuda").manual_seed(4)
    cfg = MoBAConfig(64, 3)
    for q_len in (3, 40):
        q = torch.randn((2, 8, q_len, 128), generator=g, device="cuda").to(torch.bfloat16)
        k = torch.randn((2, 2, 333, 128), generator=g, device="cuda").to(torch.bfloat16)
        v = torch.randn((2, 2, 333, 128), generator=g, device="cuda").to(torch.bfloat16)
        calls, real = [], D.chunk_decode_attention
        D.chunk_decode_attention = lambda *a, **kw: (calls.append(1), real(*a, **kw))[1]
        try:
            a, _ = moba_layer(moba_attn_varlen, cfg, Mod(), q, k, v, None)          # HIP kernels
        finally:
            D.chunk_decode_attention = real
        b, _ = moba_layer(moba_attn_varlen_naive, cfg, Mod(), q, k, v, None)    # SDPA with the bottom-right mask
        assert calls == [1] and a.shape == b.shape == (2, q_len, 8, 128)
        assert (a.float() - b.float()).abs().max() < 2e-2


@pytest.mark.parametrize("B,H,Hkv,dtype", [(1, 8, 2, torch.bfloat16), (2, 3, 1, torch.float16), (1, 2, 2, torch.bfloat16)])
@pytest.mark.parametrize("Skv,q_len", [(1, 1), (31, 5), (32, 32), (33, 8), (129, 9), (300, 16), (1025, 17), (700, 33), (2113, 129)])
def test_decode_kernel_at_the_edges_of_its_blocks(B, H, Hkv, dtype, Skv, q_len):
    """Key counts around the 32-key steps and the splits, row counts around 32, 64 and 128 rows per key/value head (one,
    two and four row blocks per workgroup, several workgroups), a group of three heads, q as a slice of a fused
    projection.  Errors: the result is rounded once to the element type (2^-9 / 2^-12 of values up to about 4)."""
    from moba_amd.decode import chunk_decode_attention
    print("block case", B, H, Hkv, Skv, q_len, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(Skv * 131 + q_len)
    q = torch.randn((B, q_len, H + 2 * Hkv, 128), generator=g, device="cuda").to(dtype)[:, :, :H].transpose(1, 2)
    k = torch.randn((B, Hkv, Skv + 7, 128), generator=g, device="cuda").to(dtype)[:, :, :Skv]
    v = torch.randn((B, Hkv, Skv + 7, 128), generator=g, device="cuda").to(dtype)[:, :, :Skv]
    out = chunk_decode_attention(q, k, v)
    want = _ref_tail(q, k, v, 128 ** -0.5)
    err = (out.float() - want).abs()
    bound = (4.0 if dtype == torch.bfloat16 else 0.5) * 2.0 ** -8
    assert torch.isfinite(out.float()).all() and err.max() < bound, err.max().item()


def test_decode_kernel_keeps_small_probabilities():
    """One key far above 100000 others whose probabilities are 2^-22 to 2^-16 of its own and together weigh a quarter of it:
    they must not fall below the element type (fp16's smallest number is 2^-24) or be rounded away."""
    from moba_amd.decode import chunk_decode_attention
    for dtype in (torch.float16, torch.bfloat16):
        q = torch.zeros((1, 1, 1, 128), device="cuda", dtype=dtype)
        q[..., 0] = 1.0
        k = torch.zeros((1, 1, 100001, 128), device="cuda", dtype=dtype)
        k[0, 0, 1:, 0] = -torch.linspace(16, 22, 100000, device="cuda").to(dtype)
        v = torch.ones((1, 1, 100001, 128), device="cuda", dtype=dtype)
        v[0, 0, 0] = 0
        out = chunk_decode_attention(q, k, v, 0.6931471805599453)     # (a score of -x is a probability of 2^-x)
        p = torch.exp2(k[0, 0, :, 0].double())
        want = (p[1:].sum() / p.sum()).item()
        assert abs(out.float().mean().item() - want) < 2.0 ** -7 * want, (dtype, out.float().mean().item(), want)


@pytest.mark.parametrize("B,H,Hkv,Skv,q_len,dtype,spread", [
    (1, 2, 1, 129, 129, torch.bfloat16, 1.0),       # one row in the last tile, no key before the first token
    (3, 1, 1, 700, 127, torch.float16, 1.0),
    (2, 6, 2, 1000, 300, torch.bfloat16, 8.0),      # tiles computed again with a running maximum
    (1, 5, 5, 65, 64, torch.float16, 8.0),
    (2, 32, 4, 777, 760, torch.bfloat16, 1.0),      # tiles of 256 rows, the last of 248
    (2, 32, 4, 1100, 1024, torch.float16, 8.0),
])
@pytest.mark.parametrize("layout", ["cache", "fused", "expanded"])
def test_causal_tiles_of_new_tokens(B, H, Hkv, Skv, q_len, dtype, spread, layout):
    """The causal tiles read q, k and v in place, whatever their strides, and all sequences in one launch.  Errors: values of up
    to about 4.5, the probabilities and the result each rounded to the element type, to half a step of a significand of 8
    (bf16) or 11 bits: relative to the value at most u = 2^-8 or 2^-11 (just above a power of two), so at most 2 * 4.5 * u
    together, and on average (half of that, over values of about 0.8) below 0.8 * u."""
    import moba_amd.decode as D
    print("new-token tiles", B, H, Hkv, Skv, q_len, dtype, spread, layout, flush=True)
    g = torch.Generator(device="cuda").manual_seed(Skv + q_len)
    randn = lambda *s: torch.randn(s, generator=g, device="cuda")
    q = (randn(B, q_len, H, 128) * spread).to(dtype).transpose(1, 2)
    if layout == "cache":        # preallocated for more tokens
        k = (randn(B, Hkv, Skv + 9, 128) * spread).to(dtype)[:, :, :Skv]
        v = randn(B, Hkv, Skv + 9, 128).to(dtype)[:, :, :Skv]
    elif layout == "fused":      # slices of one projection, heads beside heads
        kv = randn(B, Skv, 2 * Hkv, 128).to(dtype)
        kv[:, :, :Hkv] *= spread
        k, v = kv[:, :, :Hkv].transpose(1, 2), kv[:, :, Hkv:].transpose(1, 2)
    else:                        # one prompt under every sequence; values in another layout than keys
        k = (randn(1, Hkv, Skv, 128) * spread).to(dtype).expand(B, -1, -1, -1)
        v = randn(1, Skv, Hkv, 128).to(dtype).transpose(1, 2).expand(B, -1, -1, -1)
    out = D._tail_tiles(q, k, v, None)
    err = (out.float() - _ref_tail(q, k, v, 128 ** -0.5)).abs()
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert out.shape == (B, q_len, H, 128) and torch.isfinite(out.float()).all()
    assert err.max() < 2 * 4.5 * u and err.mean() < 0.8 * u, (err.max().item(), err.mean().item())


def test_routes_of_new_tokens(monkeypatch):
    """Few tokens always take the decode kernel; the kernel for very many gives the tiles' result bit for bit."""
    import moba_amd.decode as D
    for b, h, hkv in ((1, 1, 1), (64, 32, 32), (8, 64, 4), (3, 45, 5), (1, 128, 1)):
        assert not any(D._takes_tiles(b, h, hkv, n) for n in range(1, 17))
    # more sequences than the decode kernel's grid takes
    assert D._takes_tiles(70000, 1, 1, 17) and D._takes_tiles(70000, 3, 1, 5) and not D._takes_tiles(65535, 1, 1, 17)
    q, k, v = (torch.randn((66000, 1, n, 128), device="cuda").to(torch.bfloat16) for n in (17, 18, 18))
    out = D.chunk_decode_attention(q, k, v)
    some = [0, 1, 32767, 65535, 65536, 65999]
    assert (out[some].float() - _ref_tail(q[some], k[some], v[some], 128 ** -0.5)).abs().max() < 2e-2
    del q, k, v, out
    g = torch.Generator(device="cuda").manual_seed(8)
    q = torch.randn((2, 32, 1500, 128), generator=g, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn((2, 8, 1777, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    assert D._takes_tiles(2, 32, 8, 1500)
    tiles = D.chunk_decode_attention(q, k, v)
    assert torch.equal(tiles, D._tail_tiles(q, k, v, None))
    monkeypatch.setattr(D, "RESIDENT_TILES", 0)
    assert torch.equal(tiles, D.chunk_decode_attention(q, k, v))


def test_long_pieces_of_a_prompt_take_the_tiles(monkeypatch):
    """Very many new tokens of one sequence: the causal tiles, read in place (the other route copies q and the result)."""
    import moba_amd.decode as D
    calls, real = [], D._tail_tiles
    monkeypatch.setattr(D, "_tail_tiles", lambda *a: (calls.append(1), real(*a))[1])
    g = torch.Generator(device="cuda").manual_seed(6)
    q = torch.randn((1, 128, 8200, 128), generator=g, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn((1, 2, 8300, 128), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    out = D.chunk_decode_attention(q, k, v)
    assert calls == [1]
    rows = [0, 1, 127, 128, 4097, 8199]
    for j in rows:
        want = _ref(q[:, :, j:j + 1], k[:, :, :101 + j], v[:, :, :101 + j], 128 ** -0.5)
        assert (out[:, j:j + 1].float() - want).abs().max() < 2e-2


def test_a_call_lets_other_python_threads_run():
    """The native call holds no interpreter lock while it allocates and launches: in the place of moba_tail stands CPython's own
    PyGILState_Check, whose answer -- 1 with the lock -- would be taken for an error code."""
    import ctypes
    from moba_amd import _lib
    host, lib = _lib.host(), _lib.load()
    q, k = torch.zeros((1, 8, 1, 128), device="cuda", dtype=torch.bfloat16), torch.zeros((1, 2, 64, 128), device="cuda", dtype=torch.bfloat16)
    try:
        _lib.bind(host, ctypes.pythonapi.PyGILState_Check)
        assert host.tail(q, k, k, None).shape == (1, 1, 8, 128)
    finally:
        _lib.bind(host, lib.moba_tail)
    assert host.tail(q, k, k, None).abs().max() == 0
