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
