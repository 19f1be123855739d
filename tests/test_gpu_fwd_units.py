"""The bf16 forward's and dq's workgroup shapes give the same bits."""

import numpy as np
import pytest
import torch

from _helpers import operands
from mfattn import ops
from mfattn.kernels import prologue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("t", [129, 321, 641])
@pytest.mark.parametrize("hq, hkv", [(16, 8), (32, 8), (16, 2), (12, 4)])
def test_rows_of_a_large_batch_equal_rows_alone(hq, hkv, mode, t, device):
    """40 rows of t tokens (14 of 641) fill the chip: even groups take two heads per workgroup (more
    than 1024 tiles x heads), a row alone (at most 192) takes one; the group of three takes ring
    slots of one stage in the batches of 40 (960 and 1440 workgroups), of two alone and at t = 641.
    Out, lse and the gradients of every row are bit-identical, also with the query's norm and
    rotation in the forward: lists of one to eleven stages, odd and even, with segments and padding
    that cut them."""
    rng = np.random.default_rng(900 + 10 * t + mode)
    rows = 40 if t < 600 else 14
    q, k, v, do = operands(rng, rows, t, hq, hkv, 64, torch.bfloat16, 1.0)
    gain = torch.ones(64, device=device, dtype=torch.bfloat16)
    seg = np.ones((rows, t), np.int32)
    for r in range(rows):
        cuts = np.sort(rng.integers(1, t, size=int(rng.integers(0, 4))))
        for c in cuts:
            seg[r, c:] += 1
        seg[r, t - int(rng.integers(0, t // 2)):] = 0
    seg[0] = 1
    mask = torch.tensor((seg != 0).astype(np.int32), device=device)
    ids = None if mode == 2 else torch.tensor(seg, device=device)

    def results(rows):
        x, y, z, g = (a[rows].contiguous() for a in (q, k, v, do))
        plan = ops.block_map(None if ids is None else ids[rows].contiguous(),
                             mask[rows].contiguous(), mode, t, t)
        out, lse = ops.attn_fwd(x, y, z, plan, mode, 0.125)
        fused = ops.attn_fwd_rope_q(x, y, z, gain, None, plan, mode, 0.125, eps=1e-5,
                                    rope_theta=1e4)
        return (out, lse, *ops.attn_bwd(x, y, z, out, g, lse, plan, mode, 0.125), *fused)

    whole = results(slice(0, rows))
    for r in range(0, rows, 9):
        alone = results(slice(r, r + 1))
        for name, a, b in zip(("out", "lse", "dq", "dk", "dv", "fused out", "fused lse"), whole, alone):
            assert torch.equal(a[r:r + 1], b), (name, r)
    # the fused form against the two passes, at the large batch's shapes
    normed, _ = prologue.qk_norm_rope(q, k, gain, gain, None, eps=1e-5, rope_theta=1e4)
    plan = ops.block_map(ids, mask, mode, t, t)
    out, lse = ops.attn_fwd(normed, k, v, plan, mode, 0.125)
    assert torch.equal(out, whole[5]) and torch.equal(lse, whole[6])
