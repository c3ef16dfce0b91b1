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


@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("batch,seqlen,heads,B,topk", [
    (1, 16 * 512, 4, 512, 13),   # 64 workgroups of 16 waves for chunks of 512 and 12 picks
    (1, 16 * 512, 5, 512, 13),   # ... one more head: 4 waves
    (1, 4500, 3, 1024, 3),       # chunks of 1024, the last one short: 16 waves
    (1, 6 * 704, 2, 704, 9),     # ... of a length between
    (3, 3000, 3, 300, 6),        # 300 and 5 picks: 16 waves
    (1, 16 * 512, 8, 512, 4),    # 512 and few picks: 4 waves
    (1, 45 * 64, 1, 64, 3),      # 990 counts: one step of 4 waves
    (1, 46 * 64, 1, 64, 3),      # 1035: two
    (1, 91 * 1024, 1, 1024, 3),  # 4095 counts: one step of 16 waves
    (1, 92 * 1024, 1, 1024, 3),  # 4186: two
])
def test_steps_of_the_scan(batch, seqlen, heads, B, topk, counted):
    check_lists(batch, seqlen, heads, B, topk, counted, False)


@pytest.mark.parametrize("seqlen,heads,group,B,topk", [
    (1500, 6, 3, 100, 4),        # one launch
    (5000, 4, 4, 1024, 3),       # ... of 16 waves
    (129 * 66, 2, 2, 66, 3),     # separate launches, one workgroup for the tables
    (60007, 4, 2, 16, 3),        # ... and many
])
def test_tiles_of_several_heads(seqlen, heads, group, B, topk):
    """Tile tables that cut the lists of the heads of a key/value head together: lists as ever, tiles of all their rows."""
    import numpy as np
    import torch
    from moba_amd import _lib
    from moba_amd import moba_efficient as E
    lib = _lib.load()
    print("tiles of heads", seqlen, heads, group, B, topk, flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads)
    plan = E.make_plan(torch.tensor([0, seqlen], dtype=torch.int32, device="cuda"), B, topk)
    q = torch.randn((seqlen, heads, 128), generator=g, device="cuda").to(torch.bfloat16)
    sel = E.gate_topk(q, E.chunk_mean(q, plan), plan)
    want_off, _, want_dest, _ = E.build_lists(sel, plan)
    segments, t = plan.F * heads // group, plan.tables
    bounds = [plan.hist_tile_bound(heads, rows, n) for rows, n in ((256, 1), (128, group))]
    dev = dict(dtype=torch.int32, device="cuda")
    cnt, seg_off = torch.empty(plan.P * heads + 1, **dev), torch.empty(plan.F * heads + 1, **dev)
    seg_dest = torch.empty_like(want_dest)
    off_a, seg_a = torch.empty(plan.F * heads + 1, **dev), torch.full((bounds[0],), -7, **dev)
    off_b, seg_b = torch.empty(segments + 1, **dev), torch.full((bounds[1],), -7, **dev)
    p = lambda x: x.data_ptr()
    _lib.check(lib.moba_build_lists_grouped(
        p(sel), p(t["chunk_tok"]), p(t["chunk_fb"]), p(t["chunk_local"]), p(t["pair_off"]), p(cnt), p(seg_off), p(off_a),
        p(seg_dest), p(seg_a), seqlen, heads, plan.K, plan.N, plan.F, plan.P, plan.cmax, 256, bounds[0], 0, 128, p(off_b),
        p(seg_b), bounds[1], 0, 1, group, torch.cuda.current_stream().cuda_stream), "moba_build_lists_grouped")
    assert torch.equal(seg_off, want_off) and torch.equal(seg_dest, want_dest)
    counts = np.diff(want_off.cpu().numpy())
    for n, rows, off, seg in ((1, 256, off_a, seg_a), (group, 128, off_b, seg_b)):
        tiles = -(-counts.reshape(-1, n).sum(1) // rows)
        assert np.array_equal(off.cpu().numpy(), np.concatenate([[0], np.cumsum(tiles)]))
        names = np.repeat(np.arange(tiles.size), tiles)
        got = seg.cpu().numpy()
        assert names.size <= got.size and np.array_equal(got[:names.size], names) and (got[names.size:] == -1).all()


def test_first_tables_of_several_heads():
    """Both pairs of tile tables for all heads of a key/value head, in arrays of just their size: 511 segments, while the scan of
    the 4.2 million counts works on 1021 sums, more than the tables hold.  What lies behind the arrays stays as it was."""
    import numpy as np
    import torch
    from moba_amd import _lib
    from moba_amd import moba_efficient as E
    lib = _lib.load()
    seqlen, heads, B, topk = 512 * 16, 32, 16, 3
    plan = E.make_plan(torch.tensor([0, seqlen], dtype=torch.int32, device="cuda"), B, topk)
    segments, t = plan.F, plan.tables      # (one segment per chunk: 32 heads on one)
    assert -(-plan.P * heads // 4096) > segments + 1
    print("tables of all heads", plan.P * heads, segments, flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn((seqlen, heads, 128), generator=g, device="cuda").to(torch.bfloat16)
    sel = E.gate_topk(q, E.chunk_mean(q, plan), plan)
    want_off, _, want_dest, _ = E.build_lists(sel, plan)
    dev, guard, p = dict(dtype=torch.int32, device="cuda"), 4096, lambda x: x.data_ptr()
    cnt, seg_off = torch.empty(plan.P * heads + 1, **dev), torch.empty(plan.F * heads + 1, **dev)
    seg_dest = torch.empty_like(want_dest)
    bounds = [plan.hist_tile_bound(heads, rows, heads) for rows in (256, 128)]
    offs = [torch.full((segments + 1 + guard,), -7, **dev) for _ in bounds]
    segs = [torch.full((n + guard,), -7, **dev) for n in bounds]
    _lib.check(lib.moba_build_lists_grouped(
        p(sel), p(t["chunk_tok"]), p(t["chunk_fb"]), p(t["chunk_local"]), p(t["pair_off"]), p(cnt), p(seg_off), p(offs[0]),
        p(seg_dest), p(segs[0]), seqlen, heads, plan.K, plan.N, plan.F, plan.P, plan.cmax, 256, bounds[0], 0, 128, p(offs[1]),
        p(segs[1]), bounds[1], 0, heads, heads, torch.cuda.current_stream().cuda_stream), "moba_build_lists_grouped")
    assert torch.equal(seg_off, want_off) and torch.equal(seg_dest, want_dest)
    counts = np.diff(want_off.cpu().numpy()).reshape(-1, heads).sum(1)
    for rows, off, seg, bound in zip((256, 128), offs, segs, bounds):
        tiles = -(-counts // rows)
        off, seg = off.cpu().numpy(), seg.cpu().numpy()
        assert np.array_equal(off[:segments + 1], np.concatenate([[0], np.cumsum(tiles)])) and (off[segments + 1:] == -7).all()
        names = np.repeat(np.arange(tiles.size), tiles)
        assert np.array_equal(seg[:names.size], names)
        assert (seg[names.size:bound] == -1).all() and (seg[bound:] == -7).all()
