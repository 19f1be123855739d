"""fp32 attention at the edges of its work units: 32-row blocks of one head, the other side's
32-row blocks dealt to four waves (eight in dk/dv) in turn."""

import numpy as np
import pytest
import torch

from _helpers import operands
from mfattn.kernels import attention, bidirectional
from oracle import attention as oatt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [31, 32, 33, 96, 97, 160, 257, 289, 545])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_block_counts_around_the_wave_split(t, mode, device):
    """One to eighteen blocks of the other side (fewer, as many and more than the waves), three
    heads per KV head, one row of one segment and one of two; forward and backward against the
    FP64 oracle at the fp32 bar (rtol = atol = 1e-5)."""
    rng = np.random.default_rng(7000 + 3 * t + mode)
    q, k, v, do = operands(rng, 2, t, 6, 2, 64, torch.float32, 0.7)
    seg = np.ones((2, t), np.int32)
    seg[1, t // 3:] = 2
    seg[1, t - t // 8:] = 0
    mask = (seg != 0).astype(np.int32)
    tm, ts = torch.tensor(mask, device=device), torch.tensor(seg, device=device)
    leaves = [x.detach().clone().requires_grad_(True) for x in (q, k, v)]
    if mode == 0:
        out = attention.dense_packed_causal_attention(*leaves, tm, ts)
    else:
        out = bidirectional.attention(*leaves, tm, ts if mode == 1 else None)
    out.backward(do)
    ref = oatt.grouped_fp64(mode, *(x.cpu().numpy() for x in (q, k, v)), mask,
                            None if mode == 2 else seg, d_out=do.cpu().numpy())
    for name, a, r in zip(("out", "dq", "dk", "dv"), (out.detach(), *(x.grad for x in leaves)), ref):
        np.testing.assert_allclose(a.cpu().numpy(), r, rtol=1e-5, atol=1e-5, err_msg=name)
