"""The work a user of this package has it do, as cases whose time and results can be compared between two builds.

Five kinds of call, each through the public entry point a program uses:

  prefill   the attention of one decoder layer over whole prompts, as the transformers plugin calls it (``moba_layer``
            on [batch, heads, tokens, head_dim] tensors), or the packed operator ``moba_attn_varlen`` itself
  train     forward and backward of the packed operator over a batch of sequences of different lengths
  decode    one new token per sequence against its key/value cache (the plugin's decode branch)
  extend    several new tokens against the cache: a few (checking drafted tokens, a short user turn) or thousands
            (a long prompt taken in pieces)

Values are N(0, 1), the distribution of this repository's tests and benchmark; the queries, keys and values of the
128K prefill are brought to unit root mean square first, as its benchmark does.
"""

import random

import torch

from moba_amd import MoBAConfig, moba_attn_varlen
from moba_amd.moba_efficient import moba_attn_varlen_gqa
from moba_amd.wrapper import moba_layer

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, kind, **kw):
    base = dict(name=name, kind=kind, dtype="bf16", heads=32, kv_heads=8, head_dim=128)
    base.update(kw)
    return base


def listed():
    return [
        # the smallest call: a short prompt through the packed operator, where launches and latency count
        _case("prefill_4k", "prefill", entry="packed", lens="4096", heads=4, kv_heads=4, chunk=512, topk=3),
        # a batch of three short prompts, one layer of a grouped-query model, fp16 (the example's default type); the
        # last chunk of every sequence is ragged
        _case("prefill_batch", "prefill", entry="layer", lens="2001,2001,2001", chunk=256, topk=3, dtype="fp16"),
        # a middling prompt of odd length on a model with 64-element heads
        _case("prefill_narrow", "prefill", entry="layer", lens="8191", head_dim=64, chunk=512, topk=4),
        # the headline configuration: one layer of a 32-head model with 8 key/value heads over 128K tokens
        _case("prefill_128k", "prefill", entry="layer", lens="131072", chunk=4096, topk=12),
        # the reference's own speed-test shape, forward and backward: one head, too few tiles to fill the chip
        _case("train_32k", "train", lens="32768", heads=1, kv_heads=1, chunk=2048, topk=3),
        # an ordinary training batch: five documents packed to 20K tokens, grouped-query heads
        _case("train_packed", "train", lens="1023,7001,400,3579,8477", heads=8, kv_heads=2, chunk=512, topk=3),
        # the large one: eight sequences of 4K to 64K tokens, 302060 in all, none a multiple of the chunk
        _case("train_varlen8", "train", lens="59436,29343,53769,62439,31658,6749,21064,37602", kv_heads=32, chunk=2048,
              topk=3),
        # generation: a short conversation, ...
        _case("decode_4k", "decode", batch=1, kv_len=4097, spare=0),
        # ... a long document in the cache, ...
        _case("decode_128k", "decode", batch=1, kv_len=131072, spare=0),
        # ... and a batch of sixteen users, fp16, in a cache preallocated for more tokens than it holds
        _case("decode_batch", "decode", batch=16, kv_len=8191, dtype="fp16", spare=1025),
        # five drafted tokens per sequence to be checked in one pass
        _case("extend_few", "extend", batch=4, kv_len=20000, new=5, spare=480),
        # a long prompt taken in pieces of 2048 tokens: the seventeenth piece
        _case("extend_2k", "extend", batch=1, kv_len=34816, new=2048, spare=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _heads(rng):
    kv = rng.choice((1, 2, 4, 8))
    return dict(kv_heads=kv, heads=kv * rng.choice((1, 2, 4, 4, 8)) if kv < 8 else rng.choice((8, 16, 32, 32)))


def _draw_once(rng):
    kind = rng.choice(("prefill", "train", "decode", "extend"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "decode":
        return _case("", kind, dtype=dtype, batch=_log_int(rng, 1, 32), kv_len=_log_int(rng, 500, 131072),
                     spare=rng.choice((0, rng.randint(1, 2000))), **_heads(rng))
    if kind == "extend":
        kv_len = _log_int(rng, 1000, 131072)
        new = _log_int(rng, 2, 16) if rng.random() < 0.5 else _log_int(rng, 17, min(4096, kv_len // 2))
        return _case("", kind, dtype=dtype, batch=_log_int(rng, 1, 8), kv_len=kv_len, new=new,
                     spare=rng.choice((0, rng.randint(1, 2000))), **_heads(rng))
    chunk = rng.choice((128, 256, 512, 1024, 2048, 4096))
    topk = rng.randint(2, 12)
    total = _log_int(rng, 2000, 262144)
    if kind == "prefill":
        entry = rng.choice(("layer", "layer", "packed"))
        if entry == "layer":
            batch = rng.randint(1, 4)
            lens = [max(total // batch, 200)] * batch
        else:
            lens = _cut(rng, total, rng.randint(1, 6))
        head_dim = 64 if entry == "layer" and rng.random() < 0.25 else 128
        return _case("", kind, dtype=dtype, entry=entry, lens=",".join(map(str, lens)), head_dim=head_dim, chunk=chunk,
                     topk=topk, **_heads(rng))
    return _case("", kind, dtype=dtype, lens=",".join(map(str, _cut(rng, total, rng.randint(1, 8)))), chunk=chunk,
                 topk=topk, **_heads(rng))


def _cut(rng, total, parts):
    marks = sorted(rng.sample(range(1, total), parts - 1))
    return [b - a for a, b in zip([0] + marks, marks + [total])]


def draw(rng):
    """One more case of the same ranges: no dearer than the dearest listed one, in operations and in bytes."""
    most = [work(c) for c in listed()]
    flops, nbytes = (max(w[x] for w in most) for x in ("flops", "bytes"))
    while True:
        case = _draw_once(rng)
        need = work(case)
        if need["flops"] <= flops and need["bytes"] <= nbytes:
            del case["name"]
            return case


class _Attention(torch.nn.Module):
    """Stands for the decoder layer's attention module: all the plugin asks of it."""
    is_causal = True


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["head_dim"]

    def randn(*shape):
        return torch.randn(shape, generator=g, device=dev).to(dtype)

    if case["kind"] in ("decode", "extend"):
        batch, kv_len, new = case["batch"], case["kv_len"], case.get("new", 1)
        q = randn(batch, heads, new, dim)
        cache_k = randn(batch, kv_heads, kv_len + case["spare"], dim)
        cache_v = randn(batch, kv_heads, kv_len + case["spare"], dim)
        return dict(case=case, q=q, k=cache_k[:, :, :kv_len], v=cache_v[:, :, :kv_len], module=_Attention(),
                    config=MoBAConfig(4096, 12))
    lens = _lens(case)
    if case.get("entry") == "layer":
        shapes = [(len(lens), h, lens[0], dim) for h in (heads, kv_heads, kv_heads)]
        q, k, v = (randn(*s) for s in shapes)
        if lens[0] >= 131072:
            q, k, v = (x * x.float().pow(2).mean(-1, keepdim=True).rsqrt().to(dtype) for x in (q, k, v))
        return dict(case=case, q=q, k=k, v=v, module=_Attention(), config=MoBAConfig(case["chunk"], case["topk"]))
    bounds = [0]
    for n in lens:
        bounds.append(bounds[-1] + n)
    state = dict(case=case, q=randn(bounds[-1], heads, dim), k=randn(bounds[-1], kv_heads, dim),
                 v=randn(bounds[-1], kv_heads, dim), max_seqlen=max(lens),
                 cu_seqlens=torch.tensor(bounds, dtype=torch.int32, device=dev))
    if case["kind"] == "train":
        state["dout"] = randn(bounds[-1], heads, dim)
        for x in "qkv":
            state[x].requires_grad_(True)
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if "module" in state:
        with torch.no_grad():
            return moba_layer(moba_attn_varlen, state["config"], state["module"], q, k, v, None)[0]
    op = moba_attn_varlen if case["heads"] == case["kv_heads"] else moba_attn_varlen_gqa
    rest = (state["cu_seqlens"], state["max_seqlen"], case["chunk"], case["topk"])
    if case["kind"] == "prefill":
        return op(q, k, v, *rest)
    q.grad = k.grad = v.grad = None
    out = op(q, k, v, *rest)
    out.backward(state["dout"])
    return {"out": out.detach(), "dq": q.grad, "dk": k.grad, "dv": v.grad}


def _pairs(lens, chunk, topk):
    """(query, key) pairs attended and (query, chunk) pairs scored by the gate, per head."""
    attended = scored = 0
    for n in lens:
        for c in range(-(-n // chunk)):
            rows = min(chunk, n - c * chunk)
            attended += rows * (rows + 1) // 2 + rows * min(topk - 1, c) * chunk
            scored += rows * c
    return attended, scored


def work(case):
    """Every input read once and every output written once; 4 * head_dim operations per attended pair forward (two
    products), 10 * head_dim backward (five), and the gate's scores."""
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] in ("decode", "extend"):
        batch, kv_len, new = case["batch"], case["kv_len"], case.get("new", 1)
        attended = new * kv_len - new * (new - 1) // 2
        return {"bytes": 4 * batch * dim * (kv_heads * kv_len + heads * new), "flops": 4 * dim * heads * batch * attended}
    lens = _lens(case)
    tokens = sum(lens)
    attended, scored = _pairs(lens, case["chunk"], case["topk"])
    flops = heads * dim * (4 * attended + 2 * scored)
    nbytes = 4 * tokens * dim * (heads + kv_heads)
    if case["kind"] == "train":
        flops += 10 * heads * dim * attended
        nbytes += 4 * tokens * dim * (heads + kv_heads)   # dout in; dq, dk, dv out
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Against the same attention evaluated in 64 bits, outputs and gradients are off by 1.7e-3 (decode) to 2.7e-3 (dq)
    # in bf16 and by 1.9e-4 to 3.3e-4 in fp16: the rounding of the result, of the probabilities and of partial results.
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3}
