"""Decode attention on MI355X: new query tokens against the key/value cache (the adapter's decode
branch, moba/wrapper.py:76-82, which calls flash_attn_func in the reference: every cached key is
visible to a new token up to its own position).  One token or a few: the HIP decode kernel reads K and V of
the cache in place, once for up to 32 query rows of a key/value head.  Many tokens (chunked prefill against a
cache): the forward attention kernel's causal tiles on the tail of the sequences."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _lib
from . import moba_efficient as E
from .moba_efficient import _aligned

SUPPORTED_GROUP_SIZES = (1, 2, 4, 8)


def supported(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor) -> bool:
    """True when decode_attention can take these tensors ([B,H,1,D] and [B,Hkv,Skv,D])."""
    return query.is_cuda and _lib.host().supported(query, key, value, False)


def chunk_supported(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor) -> bool:
    """True when chunk_decode_attention can take these tensors ([B,H,q_len,D] and [B,Hkv,Skv,D], q_len <= Skv)."""
    return query.is_cuda and _lib.host().supported(query, key, value, True)


def _packed(t: torch.Tensor):
    t = _aligned(t)
    b, h, n, d = t.shape
    return t, (h * n * d if b > 1 else 0, n * d if h > 1 else 0, d if n > 1 else 0)


def _placed(t: torch.Tensor, row_step: int = 0):
    """A [B,heads,tokens,D] tensor as the kernels will read it, and its strides of batch, head and token: untouched where
    its rows are contiguous (and row_step apart, if given) and everything 16-byte friendly, a packed copy otherwise.
    The stride of a dimension of one entry says nothing and is 0 here."""
    b, h, n, _ = t.shape
    sb, sh, sn, sd = t.stride()
    steps = (sb if b > 1 else 0, sh if h > 1 else 0, sn if n > 1 else 0)
    if (sd == 1 and not (steps[0] | steps[1] | steps[2]) & 7 and steps[2] <= 1 << 23 and t.data_ptr() % 16 == 0
            and (sn == row_step or not row_step or n == 1)):
        return t, steps
    return _packed(t)


def _placed_three(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, row_step: int = 0):
    """query, key and value by _placed, and the strides of the first and of the other two, which share theirs."""
    q, qs = _placed(query)
    k, ks = _placed(key, row_step)
    v, vs = _placed(value, row_step)
    if ks != vs:
        (k, ks), (v, vs) = _packed(k), _packed(v)
    return q, k, v, qs, ks


MOST_SEQUENCES = 65535  # that a launch of the decode kernel takes: its grid's third dimension


def _tail(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, scaling: Optional[float]) -> torch.Tensor:
    """[B,H,q_len,D] against [B,Hkv,Skv,D] -> [B,q_len,H,D] on the decode kernel: the cache is read once for up to 32
    query rows of a key/value head."""
    out = _lib.host().tail(query, key, value, scaling)
    if out is not None:
        return out
    # tensors that have to be copied first, very many sequences, none at all
    lib = _lib.load()
    b, h, q_len, d = query.shape
    hkv, skv = key.shape[1], key.shape[2]
    q, k, v, qs, ks = _placed_three(query, key, value, d)
    dev = query.device
    out = torch.empty((b, q_len, h, d), dtype=query.dtype, device=dev)
    most = min(b, MOST_SEQUENCES)
    rows = q_len * h * most * lib.moba_tail_splits(most, hkv, h // hkv, q_len, skv)
    if b > most and b % most:    # (the last piece: fewer sequences, perhaps more splits)
        rest = b % most
        rows = max(rows, q_len * h * rest * lib.moba_tail_splits(rest, hkv, h // hkv, q_len, skv))
    part = torch.empty(rows * (d + 1), dtype=torch.float32, device=dev)   # partial outputs, then their log-sum-exps
    part_o = part.data_ptr()
    scale = float(scaling) if scaling is not None else d ** -0.5
    dtype = _lib.DTYPE_F16 if query.dtype == torch.float16 else _lib.DTYPE_BF16
    strides = (ctypes.c_int64 * 5)(*qs, ks[0], ks[1])
    stream = E._stream(dev)
    qp, kp, vp, op = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    for i in range(0, b or 1, MOST_SEQUENCES):   # (one piece, but for very many sequences)
        if i:
            qp, kp, vp = (x + 2 * MOST_SEQUENCES * step for x, step in ((qp, qs[0]), (kp, ks[0]), (vp, ks[0])))
            op += 2 * MOST_SEQUENCES * q_len * h * d
        _lib.check(lib.moba_tail(qp, kp, vp, op, part_o, part_o + rows * d * 4, min(b - i, MOST_SEQUENCES), h, hkv, q_len,
                                 skv, d, strides, scale, dtype, stream), "moba_tail")
    return out


def decode_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                     scaling: Optional[float] = None) -> torch.Tensor:
    """query [B,H,1,D], key/value [B,Hkv,Skv,D] -> [B,1,H,D] (the layout the adapter returns).
    Softmax scale ``scaling`` (default D**-0.5); every cached key is visible."""
    if not supported(query, key, value):
        raise ValueError("decode_attention needs bf16/fp16 GPU tensors, one query token, head_dim 128 and "
                         "1, 2, 4 or 8 query heads per key/value head")
    return _tail(query, key, value, scaling)


def _tail_tiles(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, scaling: Optional[float]) -> torch.Tensor:
    """As _tail, on the forward kernel's causal tiles, all sequences in one launch."""
    lib = _lib.load()
    b, h, q_len, d = query.shape
    hkv, skv = key.shape[1], key.shape[2]
    q, k, v, qs, ks = _placed_three(query, key, value)
    out = torch.empty((b, q_len, h, d), dtype=query.dtype, device=query.device)
    scale = float(scaling) if scaling is not None else d ** -0.5
    dtype = _lib.DTYPE_F16 if query.dtype == torch.float16 else _lib.DTYPE_BF16
    _lib.check(lib.moba_tail_tiles(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), b, h, hkv, q_len, skv, d,
                                   (ctypes.c_int64 * 6)(*qs, *ks), scale, dtype, 0 if E.FIXED_REFERENCE else 1,
                                   E._stream(query.device)), "moba_tail_tiles")
    return out


def _takes_tiles(b: int, h: int, hkv: int, q_len: int) -> bool:
    """Whether the causal tiles beat the decode kernel, by the number of 32-row blocks that one walks (rows of a key/value
    head packed together, whole workgroups of 32, 64 or 128 rows) and of 128-row tiles of the other, both times the keys.
    At 40000 keys a block takes 1.5 us; tiles take 540 us up to about one per compute unit (of 256: as long as 288 blocks
    and a margin) and 2.25 us each, as long as one and a half blocks, in the long run.  Decode kernel / tiles in us: 512 tokens, 32 heads on 8: 681 / 542; 256 tokens: 367 / 540; 4 sequences of 40
    tokens: 405 / 584; of 100: 787 / 585; 4 x 4096 tokens, 1 head: 741 / 549; 4 x 2048: 402 / 551.  (Up to 16 tokens it is
    always the decode kernel, whose probabilities are not rounded to the element type.)"""
    rows = h // hkv * q_len
    unit = 32 if rows <= 32 else 64 if rows <= 64 else 128
    groups = -(-rows // unit)
    blocks = b * hkv * groups * (unit // 32)
    tiles = b * h * -(-q_len // 128)
    if b > 65535 or hkv * groups > 65535 or rows > 1 << 20:   # (more than the decode kernel's grid takes)
        return q_len > 16 or h // hkv not in SUPPORTED_GROUP_SIZES
    return q_len > 16 and blocks > max(288, tiles * 3 // 2)


# The causal tiles of all sequences in one launch number their rows in 32 bits.  Calls of more rows (this many tiles of
# 256) go one sequence at a time to the forward kernel with resident workgroups, which reads its tiles' tables and
# wants q, the result and the log-sum-exps as copies.  It is the slower of the two at every size measured, resident
# workgroups / tiles, heads on key/value heads, new tokens, keys: 32 on 8, 32768, 32769: 8.3 / 7.4 ms; 65536: 22.9 / 21.7;
# 131072: 51.3 / 50.1; 64 on 8, 16384, 16385: 4.6 / 3.8; 65536, 262144: 402 / 398; 128 on 16, 65536, 131072: 347 / 341; 8 on
# 1, 262144, 300000: 149 / 146; four sequences of 32768 on 40000: 46.7 / 41.9.
RESIDENT_TILES = (1 << 31) // 256


_TAIL_TABLES = {}  # (kv_len, row tiles skipped, device) -> int32 tables of the causal tiles of a sequence's tail


def _tail_tables(kv_len: int, skip: int, tile_rows: int, device):
    """achunk_tok [2], self_tile_prefix [2], self_tile_chunk [m], chunk_direct [1] for one sequence of kv_len keys
    whose first `skip` row tiles do not exist; one small upload per distinct (length, skip)."""
    key = (kv_len, skip, str(device))
    hit = _TAIL_TABLES.get(key)
    if hit is None:
        if len(_TAIL_TABLES) >= 64:
            _TAIL_TABLES.pop(next(iter(_TAIL_TABLES)))
        m = -(-kv_len // tile_rows) - skip
        t = torch.tensor([0, kv_len, 0, m] + [0] * m + [1], dtype=torch.int32).to(device)
        hit = _TAIL_TABLES[key] = (t, m)
    return hit


def chunk_decode_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                           scaling: Optional[float] = None) -> torch.Tensor:
    """query [B,H,q_len,D]: the last q_len tokens of sequences whose keys and values [B,Hkv,Skv,D] the cache
    holds; token j attends the keys up to its own position Skv - q_len + j.  Returns [B,q_len,H,D]."""
    if not chunk_supported(query, key, value):
        raise ValueError("chunk_decode_attention needs bf16/fp16 GPU tensors, head_dim 128, no more query tokens than "
                         "keys and a whole number of query heads per key/value head")
    b, h, q_len, d = query.shape
    hkv, kv_len = key.shape[1], key.shape[2]
    if b == 0:
        return torch.empty((b, q_len, h, d), dtype=query.dtype, device=query.device)
    if not _takes_tiles(b, h, hkv, q_len) or (scaling is not None and not scaling > 0):
        return _tail(query, key, value, scaling)
    if b * h * q_len // 256 < RESIDENT_TILES:
        return _tail_tiles(query, key, value, scaling)
    lib = _lib.load()
    dev = query.device
    tile_rows = lib.moba_fwd_tile_rows()
    shift = kv_len - q_len
    skip = shift // tile_rows
    q_shift = skip * tile_rows
    pad = shift - q_shift                 # rows of the first tile that lie before the first query token
    tables, m = _tail_tables(kv_len, skip, tile_rows, dev)
    tp = tables.data_ptr()
    at = lambda i: ctypes.c_void_p(tp + 4 * i)
    scale = float(scaling) if scaling is not None else 0.0
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    code = _lib.DTYPE_F16 if query.dtype == torch.float16 else _lib.DTYPE_BF16
    null = ctypes.c_void_p(0)
    out = torch.empty((b, q_len, h, d), dtype=query.dtype, device=dev)
    for i in range(b):
        # q and the outputs hold the rows from token q_shift on: `pad` rows of padding, then the new tokens
        q_rows = torch.zeros((pad + q_len, h, d), dtype=query.dtype, device=dev)
        q_rows[pad:] = query[i].transpose(0, 1)
        out_rows = torch.empty((pad + q_len, h, d), dtype=query.dtype, device=dev)
        lse_rows = torch.empty((pad + q_len, h), dtype=torch.float32, device=dev)
        q_rows, k_rows, v_rows = E._in_place(q_rows, key[i].transpose(0, 1), value[i].transpose(0, 1))
        scratch = torch.empty(8 + 1 + m * h, dtype=torch.int32, device=dev)   # tile counters, then the redo list
        _lib.check(lib.moba_fwd_partials(
            E._ptr(q_rows), E._ptr(k_rows), E._ptr(v_rows), E._ptr(out_rows), E._ptr(lse_rows), null, null, null, null,
            at(0), at(2), null, at(4), at(4 + m), E._ptr(out_rows), E._ptr(lse_rows), kv_len, h, hkv, d, 0, 0, 1, kv_len,
            0, m, 1, E._strides(q_rows, k_rows), ctypes.c_void_p(scratch.data_ptr()),
            ctypes.c_void_p(scratch.data_ptr() + 32) if E.FIXED_REFERENCE else null, scale, code, skip, q_shift, stream),
            "moba_fwd_partials")
        out[i] = out_rows[pad:]
    return out
