"""New tokens against a key/value cache: what the kernels make of values at the edge of their types, of unusual strides
and addresses, and of batches beyond one launch."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _note(*case):
    print(*case, flush=True)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _exact(q, k, v, scale):
    """float64 attention of the last q_len tokens, every token on its own slice of the cache: [B, q_len, H, D]."""
    rep = q.shape[1] // k.shape[1]
    q_len, skv = q.shape[2], k.shape[2]
    kk, vv = (x.double().repeat_interleave(rep, dim=1) for x in (k, v))
    rows = []
    for j in range(q_len):
        n = skv - q_len + j + 1
        p = torch.softmax((q[:, :, j:j + 1].double() @ kk[:, :, :n].transpose(-1, -2).contiguous()) * scale, dim=-1)
        rows.append((p @ vv[:, :, :n])[:, :, 0])
    return torch.stack(rows, dim=1)


def _close(out, want, dtype, largest=5.0):
    """Rounded once to the element type: half a step of a significand of 8 or 11 bits at values below `largest`."""
    bound = 1.05 * largest * 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    return (out.double() - want).abs().max().item() < bound


def _partials(q, k, v, scale):
    """moba_tail's result before it is rounded: its splits' partial outputs, put together in float64."""
    from moba_amd import _lib
    lib = _lib.load()
    b, h, n, d = q.shape
    hkv, skv = k.shape[1], k.shape[2]
    splits = lib.moba_tail_splits(b, hkv, h // hkv, n, skv)
    assert splits > 1
    out = torch.empty((b, n, h, d), dtype=q.dtype, device="cuda")
    part_o = torch.empty((b, n, h, splits, d), dtype=torch.float32, device="cuda")
    part_lse = torch.empty((b, n, h, splits), dtype=torch.float32, device="cuda")
    strides = (ctypes.c_int64 * 5)(*q.stride()[:3], *k.stride()[:2])
    _lib.check(lib.moba_tail(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), part_o.data_ptr(),
                             part_lse.data_ptr(), b, h, hkv, n, skv, d, strides, scale,
                             _lib.DTYPE_F16 if q.dtype == torch.float16 else _lib.DTYPE_BF16,
                             torch.cuda.current_stream().cuda_stream), "moba_tail")
    weight = torch.softmax(part_lse.double() * 0.6931471805599453, dim=-1)
    return (weight[..., None] * part_o.double()).sum(-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_len", [1, 5, 16])
def test_probabilities_keep_their_32_bits(dtype, q_len):
    """Key i < 128 has its whole value in dimension i, so that an output is one probability over their sum, before any
    rounding to the element type.  Bound: the scores are exact; their factor, the product and the difference from the
    maximum (numbers below 4) are rounded to 2^-23 each, times ln 2; the exponential, the sums and the quotient to a few
    times 2^-24: together below 2^-20.  A probability of 16 bits would be off by up to 2^-18."""
    _note("probability bits", dtype, q_len)
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.zeros((1, 8, q_len, 128), device="cuda", dtype=dtype)
    q[..., 0] = 1
    k = torch.zeros((1, 2, 400, 128), device="cuda", dtype=dtype)
    k[..., 0] = -2 * torch.rand((1, 2, 400), generator=g, device="cuda").to(dtype)
    v = torch.zeros((1, 2, 400, 128), device="cuda", dtype=dtype)
    v[:, :, :128] = torch.eye(128, device="cuda", dtype=dtype)
    got, want = _partials(q, k, v, 1.0), _exact(q, k, v, 1.0)
    assert ((got - want).abs() / want).max().item() < 2.0 ** -20


@pytest.mark.parametrize("B,H,Hkv,Skv,q_len", [
    (2, 8, 2, 1000, 3), (1, 4, 4, 40, 16), (1, 32, 8, 1025, 8), (1, 6, 2, 9000, 5), (2, 16, 4, 300, 13),
    (1, 32, 4, 700, 9)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_a_later_tokens_values_do_not_reach_an_earlier_one(B, H, Hkv, Skv, q_len, dtype, bad):
    from moba_amd.decode import chunk_decode_attention
    _note("hidden values", B, H, Hkv, Skv, q_len, dtype, bad)
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q, k, v = (_randn(g, B, h, n, 128).to(dtype) for h, n in ((H, q_len), (Hkv, Skv), (Hkv, Skv)))
    want = _exact(q, k, v, 128 ** -0.5)
    v[:, :, -1, 5] = bad
    v[:, :, -2, 7] = bad
    out = chunk_decode_attention(q, k, v)
    others = [d for d in range(128) if d not in (5, 7)]
    assert _close(out[..., others], want[..., others], dtype)
    assert _close(out[:, :-1, :, 5], want[:, :-1, :, 5], dtype) and _close(out[:, :-2, :, 7], want[:, :-2, :, 7], dtype)
    for hit in (out[:, -1, :, 5], out[:, -2:, :, 7]):
        assert torch.isnan(hit).all() if bad != bad else (hit == bad).all()
    # a key that is not a number: only the tokens that see it
    v[:, :, -2:] = 1
    k[:, :, -1] = bad
    out = chunk_decode_attention(q, k, v)
    assert torch.isfinite(out[:, :-1].float()).all() and torch.isnan(out[:, -1].float()).any()


@pytest.mark.parametrize("B,H,Hkv,Skv,q_len", [(1, 32, 8, 4097, 1), (2, 2, 2, 50, 1), (3, 16, 2, 1000, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_visible_infinity_stays_one(B, H, Hkv, Skv, q_len, dtype):
    """As in fp32 arithmetic: its dimension becomes that infinity, two of opposite signs are not a number, and the other
    dimensions are what they were."""
    from moba_amd.decode import chunk_decode_attention
    _note("visible infinity", B, H, Hkv, Skv, q_len, dtype)
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q, k, v = (_randn(g, B, h, n, 128).to(dtype) for h, n in ((H, q_len), (Hkv, Skv), (Hkv, Skv)))
    want = _exact(q, k, v, 128 ** -0.5)
    v[:, :, 5, 3], v[:, :, 40, 9] = float("inf"), float("-inf")
    v[:, :, 2, 100], v[:, :, 33, 100] = float("inf"), float("-inf")
    out = chunk_decode_attention(q, k, v)
    assert (out[..., 3] == float("inf")).all() and (out[..., 9] == float("-inf")).all()
    assert torch.isnan(out[..., 100]).all()
    others = [d for d in range(128) if d not in (3, 9, 100)]
    assert _close(out[..., others], want[..., others], dtype)


def test_large_values_stay_finite():
    """Scores that rise by 2^7 after a wave's first keys: sums of 64 products of at most 2^119 fit fp32 with the maximum
    taken out, and would not with a maximum that lags behind by that factor."""
    from moba_amd.decode import decode_attention
    q = torch.zeros((256, 1, 1, 128), device="cuda", dtype=torch.bfloat16)
    q[..., 0] = 1
    k = torch.zeros((256, 1, 256, 128), device="cuda", dtype=torch.bfloat16)
    k[:, :, 128:, 0] = 7.0
    v = torch.full((256, 1, 256, 128), 2.0 ** 119, device="cuda", dtype=torch.bfloat16)
    out = decode_attention(q, k, v, 0.6931471805599453)
    assert (out.double() / 2.0 ** 119 - 1).abs().max().item() < 2.0 ** -8


def test_scores_far_below_zero():
    """Every score below -1e30: the maximum is still found."""
    from moba_amd.decode import decode_attention
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.zeros((1, 4, 1, 128), device="cuda", dtype=torch.bfloat16)
    q[..., 0] = 1e20
    k = torch.zeros((1, 4, 100, 128), device="cuda", dtype=torch.bfloat16)
    k[..., 0] = -1e14
    v = _randn(g, 1, 4, 100, 128).to(torch.bfloat16)
    out = decode_attention(q, k, v, 1.0)
    assert _close(out, v.double().mean(2)[:, None], torch.bfloat16)


def _odd(t, where):
    """The same values at other places: strides of one-entry dimensions that are no multiple of 8, or an address that is
    no multiple of 16."""
    b, h, n, d = t.shape
    if where == "address":
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
        return flat.view(t.shape).copy_(t)
    strides = list(t.contiguous().stride())
    for i in range(3):
        if t.shape[i] == 1:
            strides[i] = 3
    return torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device).as_strided(t.shape, strides).copy_(t)


@pytest.mark.parametrize("B,H,Hkv,Skv,q_len", [
    (2, 8, 4, 300, 1), (1, 8, 2, 300, 1), (1, 1, 1, 300, 1), (1, 4, 1, 50, 3), (1, 2, 2, 77, 20), (1, 1, 1, 1, 1)])
@pytest.mark.parametrize("where", ["strides", "address"])
def test_strides_that_say_nothing_and_odd_addresses(B, H, Hkv, Skv, q_len, where):
    import moba_amd.decode as D
    _note("odd layout", B, H, Hkv, Skv, q_len, where)
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q, k, v = (_randn(g, B, h, n, 128).to(torch.bfloat16) for h, n in ((H, q_len), (Hkv, Skv), (Hkv, Skv)))
    for change in ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)):
        args = [_odd(t, where) if c else t for t, c in zip((q, k, v), change)]
        for f in (D.chunk_decode_attention, D._tail_tiles) + ((D.decode_attention,) if q_len == 1 else ()):
            got = f(*args, None) if f is D._tail_tiles else f(*args)
            want = f(q, k, v, None) if f is D._tail_tiles else f(q, k, v)
            assert torch.equal(got, want), (f.__name__, change)
    # [B, H, D, 1] transposed: the token dimension of one entry has a stride of one element
    if q_len == 1:
        assert torch.equal(D.decode_attention(q.transpose(2, 3).contiguous().transpose(2, 3), k, v),
                           D.decode_attention(q, k, v))


def test_a_cache_is_not_copied_for_strides_that_say_nothing():
    from moba_amd.decode import decode_attention
    q = torch.zeros((1, 4, 1, 128), device="cuda", dtype=torch.bfloat16)
    cache = torch.zeros((1, 4, 16384, 128), device="cuda", dtype=torch.bfloat16)
    k = cache[:, :, :16000]
    v = torch.zeros_like(cache).as_strided(k.shape, (8, *k.stride()[1:]))
    decode_attention(q, k, k)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    decode_attention(q, k, v)
    assert torch.cuda.max_memory_allocated() - before < k.numel()      # (half of one tensor's bytes)


@pytest.mark.parametrize("q_len", [40, 2000])
def test_no_sequences_at_all(q_len):
    from moba_amd.decode import chunk_decode_attention
    q, k = (torch.empty((0, 4, n, 128), device="cuda", dtype=torch.bfloat16) for n in (q_len, 3000))
    assert chunk_decode_attention(q, k, k).shape == (0, q_len, 4, 128)


@pytest.mark.parametrize("q_len,scale", [(1, None), (5, None), (17, -0.1), (3, 0.0)])
def test_more_sequences_than_one_grid(q_len, scale):
    """66000 sequences, whatever the number of tokens and the scale."""
    import moba_amd.decode as D
    _note("many sequences", q_len, scale)
    g = torch.Generator(device="cuda").manual_seed(q_len)
    q, k, v = (_randn(g, 66000, 1, n, 128).to(torch.bfloat16) for n in (q_len, 18, 18))
    out = D.chunk_decode_attention(q, k, v, scale)
    some = [0, 1, 32767, 65534, 65535, 65536, 65999]
    assert _close(out[some], _exact(q[some], k[some], v[some], 128 ** -0.5 if scale is None else scale), torch.bfloat16)
    if q_len == 1:
        assert torch.equal(out, D.decode_attention(q, k, v, scale))


@pytest.mark.parametrize("B,H,Hkv,q_len", [
    (163, 8, 8, 1), (75, 8, 4, 1), (321, 1, 1, 7), (90, 32, 8, 8), (257, 5, 1, 4), (130, 16, 8, 3), (1300, 33, 1, 1)])
@pytest.mark.parametrize("Skv", [8, 31, 33, 64, 129, 300, 777, 1500, 4096, 4097])
def test_many_sequences_of_short_caches(B, H, Hkv, q_len, Skv):
    """More key/value heads than compute units: workgroups of one, two and four waves, with and without splits, on caches
    that end within, at and behind a wave's and a workgroup's step; the last case has a row more than they take.  The
    same sequences alone (four waves, more splits) agree to a rounding each."""
    import moba_amd.decode as D
    _note("short caches", B, H, Hkv, q_len, Skv)
    dtype = torch.float16 if Skv % 2 else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q, k, v = (torch.randn((B, h, n, 128), generator=g, device="cuda", dtype=dtype)
               for h, n in ((H, q_len), (Hkv, Skv), (Hkv, Skv)))
    out = D._tail(q, k, v, None)
    some = sorted({0, 1, B // 2, B - 2, B - 1})
    assert _close(out[some], _exact(q[some], k[some], v[some], 128 ** -0.5), dtype)
    few = torch.cat([D._tail(q[i:i + 1], k[i:i + 1], v[i:i + 1], None) for i in range(B)])
    assert (out.float() - few.float()).abs().max() < 2 * 5.0 * 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    # a value that is not finite stays with the tokens that see it, in these forms too
    v[:, :, -1, 3] = float("inf")
    hit = D._tail(q, k, v, None)
    assert (hit[:, -1, :, 3] == float("inf")).all() and torch.isfinite(hit[..., 4:].float()).all()
    if q_len > 1:
        assert _close(hit[some][:, :-1], _exact(q[some][:, :, :-1], k[some][:, :, :-1], v[some][:, :, :-1], 128 ** -0.5), dtype)


def test_the_c_entry_takes_results_at_any_address():
    """moba_decode writes out and its scratch wherever their elements can lie."""
    from moba_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(9)
    for skv in (60, 3000):                                             # one split, several
        q, k, v = (_randn(g, 2, h, n, 128).to(torch.bfloat16) for h, n in ((8, 1), (4, skv), (4, skv)))
        splits = lib.moba_decode_splits(2, 4, skv)
        got = []
        for shift in (0, 1):
            out = torch.zeros(2 * 8 * 128 + 1, dtype=torch.bfloat16, device="cuda")[shift:][:2 * 8 * 128]
            part_o = torch.zeros(2 * 8 * splits * 128 + 1, dtype=torch.float32, device="cuda")[shift:]
            part_lse = torch.zeros(2 * 8 * splits + 1, dtype=torch.float32, device="cuda")[shift:]
            _lib.check(lib.moba_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), part_o.data_ptr(),
                                       part_lse.data_ptr(), 2, 8, 4, skv, 128, 1024, 128, 4 * skv * 128, skv * 128,
                                       128 ** -0.5, _lib.DTYPE_BF16, torch.cuda.current_stream().cuda_stream),
                       "moba_decode")
            got.append(out.clone())
        assert torch.equal(*got)
