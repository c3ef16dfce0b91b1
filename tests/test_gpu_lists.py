"""The gather lists' one-launch form (scan, fill and tables) at the edges of its range."""

import pytest

from test_gpu_stages import test_gather_lists as check_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("batch,seqlen,heads,B,topk", [
    (1, 5000, 3, 1024, 3),       # long chunks: 16 waves per query chunk and head
    (1, 12400, 2, 1030, 13),     # ... more than 4 picks
    (1, 128 * 66, 1, 66, 3),     # 8128 counts, 127 candidates: the most but one row
    (1, 129 * 66, 1, 66, 3),     # 8256 counts: separate launches again
    (2, 1000, 16, 100, 6),       # as many workgroups for the tables as heads, segments past a workgroup's lanes
    (1, 130, 33, 64, 2),         # fewer tiles than table workgroups
])
def test_lists_in_one_launch(batch, seqlen, heads, B, topk, counted, dense):
    if dense and seqlen <= topk * B:
        pytest.skip("every token lies in a dense prefix")
    check_lists(batch, seqlen, heads, B, topk, counted, dense)
