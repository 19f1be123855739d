"""fp32 attention where a sequence ends inside a 32-row block."""

import pytest
import torch

from mfattn import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 5, 33, 63, 100, 129, 190])
def test_an_infinite_last_row_stays_infinite(t, device):
    """One segment per row, every key valid.  The last value row is infinite in one dimension: so
    is the output there on every query.  The last output gradient is infinite in one dimension:
    so is dv there on every key.  (Rows past the end that read the last row again weighed it with
    a zero probability: NaN.)  Everything else is finite."""
    gen = torch.Generator(device=device).manual_seed(t)
    q, k, v, do = (torch.randn((2, t, h, 64), generator=gen, device=device) for h in (4, 2, 2, 4))
    seg = torch.ones((2, t), dtype=torch.int32, device=device)
    plan = ops.block_map(seg, seg, 1, t, t)
    out, lse = ops.attn_fwd(q, k, v, plan, 1, 0.125)
    far = do.clone()
    far[1, t - 1, 2, 7] = float("inf")
    _, _, dv = ops.attn_bwd(q, k, v, out, far, lse, plan, 1, 0.125)
    inf = torch.zeros_like(dv, dtype=torch.bool)
    inf[1, :, 1, 7] = True
    assert (dv[inf] == float("inf")).all() and torch.isfinite(dv[~inf]).all()
    v[0, t - 1, 1, 3] = float("inf")
    out, lse = ops.attn_fwd(q, k, v, plan, 1, 0.125)
    inf = torch.zeros_like(out, dtype=torch.bool)
    inf[0, :, 2:, 3] = True
    assert (out[inf] == float("inf")).all() and torch.isfinite(out[~inf]).all()
    assert torch.isfinite(lse).all()
