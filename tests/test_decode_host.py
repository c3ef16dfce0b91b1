"""How the decode entry points prepare their tensors (no GPU)."""

import torch


def _as_strided(shape, strides, offset=0):
    span = sum((n - 1) * s for n, s in zip(shape, strides)) + 1
    return torch.arange(span + offset, dtype=torch.float32).to(torch.bfloat16).as_strided(shape, strides, offset)


def test_tensors_read_in_place_and_copied():
    from moba_amd.decode import _placed, _placed_three
    cases = [  # shape, strides, offset of the address in elements, key rows next to each other asked for, read in place
        ((2, 4, 10, 128), (5120, 1280, 128, 1), 0, True, True),
        ((2, 4, 10, 128), (8192, 2048, 128, 1), 0, True, True),       # a slice of a longer cache
        ((2, 4, 1, 128), (1024, 128, 1, 1), 0, True, True),           # one token: its stride says nothing
        ((1, 4, 10, 128), (3, 1280, 128, 1), 0, True, True),          # one sequence
        ((2, 1, 10, 128), (1280, 5, 128, 1), 0, True, True),          # one head
        ((2, 4, 10, 128), (5120, 128, 512, 1), 0, False, True),       # heads beside heads
        ((2, 4, 10, 128), (5120, 128, 512, 1), 0, True, False),
        ((2, 4, 10, 128), (0, 1280, 128, 1), 0, True, True),          # one cache under every sequence
        ((2, 4, 10, 128), (512, 128, 0, 1), 0, True, False),          # one row under every token
        ((2, 4, 10, 128), (5120, 1280, 128, 1), 1, True, False),      # an odd address
        ((2, 4, 10, 128), (5124, 1280, 128, 1), 0, True, False),      # an odd batch stride
        ((2, 4, 10, 128), (10240, 2560, 256, 2), 0, False, False),    # elements apart
    ]
    for shape, strides, offset, rows, kept in cases:
        t = _as_strided(shape, strides, offset)
        assert offset or t.data_ptr() % 16 == 0
        got, steps = _placed(t, 128 if rows else 0)
        assert (got.data_ptr() == t.data_ptr()) == kept, (shape, strides, offset)
        assert torch.equal(got, t) and got.data_ptr() % 16 == 0 and got.stride(3) == 1
        for step, s, n in zip(steps, got.stride(), shape):
            assert step == (s if n > 1 else 0) and step % 8 == 0
    # strides that differ only where they say nothing: no copies; others: both packed
    k = _as_strided((1, 4, 10, 128), (8, 2048, 128, 1))
    v = _as_strided((1, 4, 10, 128), (8192, 2048, 128, 1))
    q, k2, v2, qs, ks = _placed_three(k, k, v, 128)
    assert (q.data_ptr(), k2.data_ptr(), v2.data_ptr()) == (k.data_ptr(), k.data_ptr(), v.data_ptr()) and ks == (0, 2048, 128)
    v = _as_strided((1, 4, 10, 128), (8192, 1280, 128, 1))
    q, k2, v2, qs, ks = _placed_three(k, k, v, 128)
    assert ks == (0, 1280, 128) and qs == (0, 2048, 128) and torch.equal(k2, k) and torch.equal(v2, v)


def test_the_extension_reads_in_place_what_the_general_path_does():
    """csrc/host.cpp decides on strides and addresses as _placed does, over layouts of every kind."""
    import random
    from moba_amd import _lib
    from moba_amd.decode import _placed
    host, rng, kept = _lib.host(), random.Random(1), 0
    for _ in range(3000):
        shape = tuple(rng.choice((1, 1, 2, 3)) for _ in range(3)) + (128,)
        strides = tuple(rng.choice((0, 3, 8, 100, 128, 256, 1024, 1 << 23, (1 << 23) + 8)) for _ in range(3)) + (rng.choice((1, 1, 1, 2)),)
        span = sum((n - 1) * s for n, s in zip(shape, strides)) + 1
        if span > 1 << 22:
            continue     # (memory)
        base = torch.empty(span + 8, dtype=torch.bfloat16)
        t = base.as_strided(shape, strides, rng.choice((0, 0, 0, 1, 8)))     # (also odd addresses)
        step = rng.choice((0, 128))
        got, steps = _placed(t, step)
        same = got.data_ptr() == t.data_ptr() and got.stride() == t.stride()
        native = host.in_place(t, step)
        if native is not None:
            kept += 1
            assert same and native == steps, (shape, strides, step)
        else:
            assert not same or t.is_contiguous(), (shape, strides, step)
    assert kept > 200


def test_an_extension_built_for_something_else_is_refused_and_built_again(monkeypatch):
    """Another PyTorch's tensors, another version of the C ABI: neither may meet code compiled for the former one."""
    import ctypes
    import pytest
    from moba_amd import _lib, build
    host, lib = _lib.host(), _lib.load()
    assert host.torch_version == torch.__version__
    with pytest.raises(RuntimeError, match="of the C ABI"):
        other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: _lib.ABI_VERSION + 1)
        host.bind(*(ctypes.cast(f, ctypes.c_void_p).value for f in (other, lib.moba_tail_splits, lib.moba_tail, lib.moba_strerror)))
    build._host_module(force=False)
    ran = []
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **kw: ran.append(cmd) or (_ for _ in ()).throw(InterruptedError))
    build._host_module(force=False)
    assert not ran     # (nothing changed: nothing to build)
    monkeypatch.setattr(torch, "__version__", "2.0.0")
    with pytest.raises(InterruptedError):
        build._host_module(force=False)
    assert '-DMOBA_TORCH_VERSION="2.0.0"' in ran[0]
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.raises(RuntimeError, match="was built for PyTorch"):
        _lib.host()
