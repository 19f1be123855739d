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


def test_more_workgroups_than_one_launch_may_have(device):
    """65535 rows of one token, 260/130 heads: the forward, dq and dk/dv each exceed 2**32 threads,
    the limit of one launch.  A row that sees one key copies it: out is the value of each head's
    group, dq and dk are zero and dv sums the group's gradients."""
    rows, hq, hkv = 65535, 260, 130
    gen = torch.Generator(device=device).manual_seed(1)
    q, k, v, do = (torch.randn((rows, 1, h, 64), generator=gen, device=device)
                   for h in (hq, hkv, hkv, hq))
    seg = torch.ones((rows, 1), dtype=torch.int32, device=device)
    plan = ops.block_map(seg, seg, 0, 1, 1)
    out, lse = ops.attn_fwd(q, k, v, plan, 0, 0.125)
    # softmax of one score is 1: exp2 of a rounding error (2**-21 of a score below 16), times 1 / l
    assert torch.allclose(out, v.repeat_interleave(2, dim=2), rtol=1e-5, atol=1e-5)
    dq, dk, dv = ops.attn_bwd(q, k, v, out, do, lse, plan, 0, 0.125)
    assert torch.allclose(dv, do.view(rows, 1, hkv, 2, 64).sum(3), rtol=1e-5, atol=2e-5)
    # dS = P (dP - D): dP and D are the same 64 products in another order
    assert dq.abs().max() < 1e-4 and dk.abs().max() < 1e-4


def test_one_token_segments_have_gradients_of_the_rounding_alone(device):
    """A token that sees only itself has P = 1 and O = V, so dP - D is zero but for the roundings
    of O, two per dimension: their root mean square is at most 2**-24 sqrt(2) times the 2-norm of
    the 64 products of dO and V, as long as the sums of dP and D round alike.  (Sums in different
    orders, or dP started from -D, add sqrt(64) roundings of partial sums: several times that.)"""
    gen = torch.Generator(device=device).manual_seed(5)
    rows, t, h = 4, 100, 8
    q, k, v, do = (torch.randn((rows, t, h, 64), generator=gen, device=device) for _ in range(4))
    seg = torch.arange(1, t + 1, device=device, dtype=torch.int32).repeat(rows, 1)
    plan = ops.block_map(seg, seg, 0, t, t)
    out, lse = ops.attn_fwd(q, k, v, plan, 0, 0.125)
    dq, dk, _ = ops.attn_bwd(q, k, v, out, do, lse, plan, 0, 0.125)
    ws = ops.bwd_workspace(q)
    ops.attn_bwd_delta(out, do, lse, ws)
    dq2 = torch.empty_like(q)
    ops.attn_bwd_dq(q, k, v, do, lse, plan, 0, 0.125, ws, dq2)
    assert torch.equal(dq, dq2)  # the separate pass adds D in the same order
    rms = lambda x: x.double().square().mean().sqrt().item()  # noqa: E731
    products = (do.double() * v.double()).square().sum(-1).mean().sqrt().item()
    bound = 2.0 ** -24 * 2 ** 0.5 * products * 0.125
    assert rms(dq) <= bound * rms(k) and rms(dk) <= bound * rms(q)
