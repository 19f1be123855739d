"""The bf16 attention kernels' output rows at the edges of a wave's 32-row tile."""

import numpy as np
import pytest
import torch

from _helpers import check_bf16, operands, torch_reference
from mfattn.kernels import attention, bidirectional

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 16, 31, 32, 33, 63, 97, 128, 129])
@pytest.mark.parametrize("heads", [(2, 1), (3, 1), (4, 4)])
def test_ragged_row_tiles(t, heads, device):
    """Three rows of t tokens (the last wave's tile cut at every kind of edge; rows past T or a
    neighbour row must stay untouched), one padded in part: out, dq, dk and dv against the fp32
    reference at the bf16 bar, zeros on padding, for one and two heads per workgroup."""
    rng = np.random.default_rng(4100 + 10 * t + heads[0])
    q, k, v, do = operands(rng, 3, t, *heads, 64, torch.bfloat16, 1.0)
    seg = np.ones((3, t), np.int32)
    seg[1, t // 2:] = 2
    seg[2, t - t // 3:] = 0
    mask = (seg != 0).astype(np.int32)
    tm, ts = torch.tensor(mask, device=device), torch.tensor(seg, device=device)
    for mode in (0, 1):
        leaves = [x.detach().clone().requires_grad_(True) for x in (q, k, v)]
        if mode == 0:
            out = attention.packed_causal_attention(*leaves, tm, ts, backend="hip")
        else:
            out = bidirectional.attention(*leaves, tm, ts)
        grads = torch.autograd.grad(out, leaves, do)
        ref = torch_reference(mode, q, k, v, mask, seg, do)
        for name, a, r in zip(("out", "dq", "dk", "dv"), (out.detach(), *grads), ref):
            check_bf16(f"{name} mode {mode} t {t} heads {heads}", a, r)
            assert not a[tm == 0].any(), name
