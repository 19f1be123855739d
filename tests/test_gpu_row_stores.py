"""The bf16 attention kernels' output rows at the edges of a wave's 32-row tile."""

import numpy as np
import pytest
import torch

from _helpers import check_bf16, operands, torch_reference
from mfattn import ops
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


def test_outputs_at_an_eight_byte_offset(device):
    """The 16-byte row stores into caller's buffers that start eight bytes past a 16-byte
    boundary: the bits of the aligned call, and nothing around them touched."""
    rng = np.random.default_rng(77)
    q, k, v, do = operands(rng, 2, 161, 4, 2, 64, torch.bfloat16, 1.0)
    seg = torch.ones((2, 161), dtype=torch.int32, device=device)
    plan = ops.block_map(seg, seg, 0, 161, 161)
    out, lse = ops.attn_fwd(q, k, v, plan, 0, 0.125)
    ws = ops.bwd_workspace(q)
    ops.attn_bwd_delta(out, do, lse, ws)

    def buffers(n):
        whole = torch.full((q.numel() + 16,), 7.0, dtype=torch.bfloat16, device=device)
        return whole, [whole[at:at + n] for at in (8, 4)]

    whole, views = buffers(q.numel())
    results = []
    for x in views:
        whole.fill_(7.0)
        ops.attn_bwd_dq(q, k, v, do, lse, plan, 0, 0.125, ws, x.view_as(q))
        results.append(x.clone())
        at = x.storage_offset()
        assert (whole[:at] == 7).all() and (whole[at + q.numel():] == 7).all()
    assert torch.equal(*results)
    whole, views = buffers(k.numel())
    results = []
    for x in views:
        whole.fill_(7.0)
        dv = torch.empty_like(v)
        ops.attn_bwd_dkdv(q, k, v, do, lse, plan, 0, 0.125, ws, x.view_as(k), dv)
        results.append(x.clone())
        at = x.storage_offset()
        assert (whole[:at] == 7).all() and (whole[at + k.numel():] == 7).all()
    assert torch.equal(*results)
