"""The chunk mean with a head's columns in one, two and four workgroups, and in two stages, either side of the lines between them:
the exact mean rounded once, and the caller's array cleared on the way (GPU only)."""

import pytest
import torch

from oracle import moba_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,chunks,B,D", [
    (4, 7, 512, 128), (1, 1, 33, 128), (3, 2, 1000, 128), (1, 65, 100, 128), (3, 21, 1500, 128), (1, 127, 40, 128),   # halves
    (1, 8, 33, 128), (8, 3, 700, 128), (4, 16, 40, 128), (8, 9, 40, 128),                      # quarters; beyond 64: halves
    (1, 128, 40, 128), (1, 191, 40, 128), (1, 192, 40, 128), (3, 64, 77, 128),                 # whole rows
    (1, 3, 500, 64), (5, 12, 130, 64), (1, 65, 129, 64), (13, 5, 64, 64),                      # 64-element heads: whole rows,
    (8, 1, 500, 64), (1, 64, 40, 64), (2, 12, 333, 64),                                        # halves
    (1, 3, 16384, 128), (1, 1, 16385, 128), (1, 2, 40000, 64),                                 # two stages: too many bytes,
    (1, 16, 3100, 128), (1, 15, 3100, 128), (1, 3, 3072, 64), (1, 3, 3073, 64),                # or too many for narrow rows,
    (2, 2, 16384, 128), (2, 2, 16385, 128), (5, 1, 16384, 64), (5, 1, 16385, 64)])            # and the lines of both
def test_chunk_mean_in_column_parts(H, chunks, B, D, dtype):
    from moba_amd import moba_efficient as E
    print("mean", H, chunks, B, D, dtype, flush=True)
    S = chunks * B + 17
    g = torch.Generator().manual_seed(S + H)
    k = torch.randn((S, H, D), generator=g).to(dtype)
    clear = torch.full((70001,), 5, dtype=torch.int32, device="cuda")
    got = E.chunk_mean(k.cuda(), E.make_plan([0, S], B, 3, device="cuda"), clear=clear[:70000])
    assert int(clear[:70000].abs().max()) == 0 and int(clear[70000]) == 5
    assert torch.equal(got.cpu().view(torch.int16), O.chunk_mean(k, [0, S], B).view(torch.int16))
