"""Gradients where the delta kernel takes one or four rows to a lane, with rows left over, and where the dQ kernel's workgroups
have a tile each, too few, or some to draw, against 64 bits (GPU only)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sequences,H", [(1, 1), (1, 2), (2, 5), (3, 3), (4095, 1),   # one row: up to 32767
                                         (4096, 1), (4099, 1), (1367, 3), (830, 5),  # four
                                         (511, 1), (512, 1), (513, 1), (257, 2)])    # tiles around the 512 workgroups
def test_dq_of_short_sequences(sequences, H, dtype):
    from moba_amd import moba_efficient as E
    print("delta", sequences, H, dtype, flush=True)
    n, D = 8, 128
    S = sequences * n
    g = torch.Generator().manual_seed(S + H)
    q, k, v, do = (torch.randn((S, H, D), generator=g).to(dtype) for _ in range(4))
    gq = q.cuda().requires_grad_()
    cu = torch.arange(0, S + 1, n, dtype=torch.int32, device="cuda")
    E.moba_attn_varlen(gq, k.cuda(), v.cuda(), cu, n, 64, 3).backward(do.cuda())
    got = gq.grad.cpu().double()

    def by_head(x):  # [sequences, H, n, D]
        return x.double().view(sequences, n, H, D).permute(0, 2, 1, 3).contiguous()

    q4, k4, v4, do4 = map(by_head, (q, k, v, do))
    scale = D ** -0.5
    mask = torch.ones(n, n, dtype=torch.bool).triu(1)
    p = ((q4 @ k4.transpose(2, 3).contiguous()) * scale).masked_fill(mask, float("-inf")).softmax(-1)
    o = p @ v4
    ds = p * (do4 @ v4.transpose(2, 3).contiguous() - (do4 * o).sum(-1, keepdim=True))
    want = scale * ds @ k4
    # The result, dS and O are rounded to the element type, O in each term of delta: `unit` each, twice for what goes on in 32
    # bits (sums of 128 terms, an exponential) besides.
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    of_ds = 2 * unit * (ds.abs() + p * (do4 * o).abs().sum(-1, keepdim=True))
    bound = unit * want.abs() + scale * of_ds @ k4.abs()
    assert bool(((by_head(got) - want).abs() <= bound).all())
