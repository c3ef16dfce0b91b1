"""The C-ABI library loads and exports every symbol include/moba_hip.h declares
(no compute calls: this runs without a GPU)."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "moba_amd", "libmoba_hip.so")
HDR = os.path.join(ROOT, "include", "moba_hip.h")


def declared_symbols():
    text = open(HDR).read()
    return sorted(set(re.findall(r"\b(moba_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        import __graft_entry__ as entry
        entry.build()
    return ctypes.CDLL(LIB)


def test_header_symbols_exported(lib):
    names = declared_symbols()
    assert len(names) >= 8
    for n in names:
        assert hasattr(lib, n), f"{n} declared in include/moba_hip.h but not exported"


def test_binding_covers_header():
    from moba_amd import _lib
    assert sorted(_lib.exported_symbols()) == declared_symbols()


def test_version_and_strerror(lib):
    from moba_amd import _lib
    lib.moba_version.restype = ctypes.c_int
    header = open(os.path.join(os.path.dirname(__file__), "..", "include", "moba_hip.h")).read()
    assert f"#define MOBA_ABI_VERSION {_lib.ABI_VERSION} " in header
    assert lib.moba_version() == _lib.ABI_VERSION
    lib.moba_strerror.restype = ctypes.c_char_p
    assert lib.moba_strerror(0) == b"ok"
    assert b"argument" in lib.moba_strerror(-1)


def _header_prototypes():
    """name -> list of parameter type strings, parsed from the header's declarations."""
    text = re.sub(r"/\*.*?\*/", " ", open(HDR).read(), flags=re.S)
    protos = {}
    for m in re.finditer(r"\b(?:int|size_t|const char\s*\*)\s*(moba_[a-z0-9_]+)\s*\(([^;]*?)\)\s*;", text, flags=re.S):
        params = [p.strip() for p in m.group(2).replace("\n", " ").split(",")]
        protos[m.group(1)] = [] if params == ["void"] else params
    return protos


def test_binding_signatures_match_header():
    """Every ctypes signature has the header's number of parameters, pointer for pointer and
    integer width for integer width (a binding out of step with the header would hand the kernels
    garbage pointers)."""
    from moba_amd import _lib
    protos = _header_prototypes()
    assert sorted(protos) == declared_symbols()
    for name, (_, argtypes) in _lib._SIGNATURES.items():
        params = protos[name]
        assert len(params) == len(argtypes), (name, len(params), len(argtypes))
        for p, a in zip(params, argtypes):
            if "*" in p:
                want = (ctypes.c_void_p, ctypes.c_char_p, ctypes.POINTER(ctypes.c_int64))
            elif p.startswith("int64_t"):
                want = (ctypes.c_int64,)
            elif p.startswith("size_t"):
                want = (ctypes.c_size_t,)
            elif p.startswith("float"):
                want = (ctypes.c_float,)
            else:
                assert p.startswith("int "), (name, p)
                want = (ctypes.c_int,)
            assert a in want, (name, p, a)


def test_list_counts_beyond_an_int_are_refused(lib):
    """The scan of the list counts steps through them 4096 at a time in 32 bits: a number of counts whose last step would
    pass 2^31 is refused before anything is launched."""
    from moba_amd import _lib
    bound = _lib.load()
    some = ctypes.c_void_p(256)   # (never read)
    for P, H in ((0x7fffffff - 4095, 1), (0x7ffffffe, 1), ((0x7fffffff - 100) // 2, 2)):
        rc = bound.moba_build_lists(*[some] * 10, 4096, H, 1, 16, 64, P, 10, 128, 1024, 1, 0, None, None, 0, 0, None)
        assert rc == -4, (P, H, rc)


def test_shares_beyond_32_bits_are_refused(lib):
    """moba_bwd with shares of a key/value head's work: more stages than the kernel's numbers hold are refused before anything is
    launched; without the scratch for the shares, which leaves whole tiles, they are no matter."""
    from moba_amd import _lib
    bound = _lib.load()
    some = 256   # (never read: the odd strides end every call that gets that far)
    odd = (ctypes.c_int64 * 7)(*[1] * 7)

    def call(S, H, Hkv, kv_tiles, shares, scratch=some, size=1 << 62):
        return bound.moba_bwd(*[some] * 20, None, None, None, 0, S, *[some] * 5, S, H, Hkv, 128, 0, 0, 1, 64, 0, 1, kv_tiles, 1, odd,
                              some, scratch, size, shares, 1, 0.0, 0, None)

    refused = [(1 << 19, 64 * 2, 2, 4096),        # 8192 causal stages a head, 64 heads: 2^32 exactly, but too many places
               ((1 << 19) + 64, 64, 1, 1),        # one stage a head more than the division takes
               (1 << 16, 1 << 14, 4, 512)]        # 2^31 places
    for sizes in refused:
        assert call(*sizes, 4) == -4, sizes
        assert call(*sizes, 0) != -4 and call(*sizes, 4, None) != -4 and call(*sizes, 4, some, 4096) != -4, sizes
    assert call(1 << 19, 64, 1, 1, 4) != -4


def test_merges_beyond_32_bit_slot_rows_are_refused(lib):
    """moba_fwd_merge numbers slot rows in 32 bits: a call with more of them is refused before anything is launched, whichever
    factor takes it there; one without rows to merge has nothing to number."""
    from moba_amd import _lib
    bound = _lib.load()
    some = 256   # (never read)

    def call(S, H, K, parts, tokens=None, ranges=None):
        return bound.moba_fwd_merge(some, some, some, some, some, S, H, 128, K, parts, ranges, ranges, 1 if ranges else 0,
                                    S if tokens is None else tokens, 0, None)

    for S, H, K, parts in ((1 << 31, 1, 2, 1), (1 << 29, 1, 3, 1), (1 << 28, 1, 3, 2), (1 << 20, 1 << 9, 3, 1), (1 << 62, 64, 3, 1),
                           (1 << 30, 1 << 30, (1 << 30) - 1, 8), ((1 << 31) - 1, 1, 0, 1)):
        assert call(S, H, K, parts) == -4, (S, H, K, parts)
        assert call(S, H, K, parts, 1, some) == -4, (S, H, K, parts)
        assert call(S, H, K, parts, 0, some) == 0, (S, H, K, parts)
