"""The bf16 forward's two workgroup shapes give the same bits."""

import numpy as np
import pytest
import torch

from _helpers import operands
from mfattn import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("t", [129, 321])
def test_rows_of_a_large_batch_equal_rows_alone(mode, t, device):
    """24 rows of t tokens, 16/8 heads, fill the chip (two heads per workgroup: more than 1024
    tiles x heads for t = 321, fewer for t = 129, whose rows take one head per workgroup both
    ways); a row alone never does.  Out and lse of every row are bit-identical: lists of one to
    six stages, odd and even, with segments and padding that cut them."""
    rng = np.random.default_rng(900 + 10 * t + mode)
    rows = 24
    q, k, v, _ = operands(rng, rows, t, 16, 8, 64, torch.bfloat16, 1.0)
    seg = np.ones((rows, t), np.int32)
    for r in range(rows):
        cuts = np.sort(rng.integers(1, t, size=int(rng.integers(0, 4))))
        for c in cuts:
            seg[r, c:] += 1
        seg[r, t - int(rng.integers(0, t // 2)):] = 0
    seg[0] = 1
    mask = torch.tensor((seg != 0).astype(np.int32), device=device)
    ids = None if mode == 2 else torch.tensor(seg, device=device)
    plan = ops.block_map(ids, mask, mode, t, t)
    out, lse = ops.attn_fwd(q, k, v, plan, mode, 0.125)
    for r in range(0, rows, 5):
        one = slice(r, r + 1)
        p = ops.block_map(None if ids is None else ids[one].contiguous(), mask[one].contiguous(),
                          mode, t, t)
        o, l = ops.attn_fwd(q[one].contiguous(), k[one].contiguous(), v[one].contiguous(), p, mode,
                            0.125)
        assert torch.equal(out[one], o) and torch.equal(lse[one], l), r
