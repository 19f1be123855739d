"""The row decode's splits of an item (one wave, four, the most) at the lines between them."""

import numpy as np
import pytest
import torch

from _helpers import check_bf16
from mfattn.kernels import attention
from oracle import attention as oatt

pytestmark = pytest.mark.gpu


# rows x ceil(capacity / 128) items: up to 256 the most waves an item, up to 512 four, then one;
# caches above 256 MiB stream V
@pytest.mark.parametrize("rows, cap", [(3, 127), (3, 128), (3, 129), (128, 200), (129, 200),
                                       (256, 130), (257, 130)])
@pytest.mark.parametrize("hq, hkv", [(8, 8), (16, 8), (40, 8), (64, 8), (12, 4), (10, 2), (7, 1),
                                     (8, 1)])
def test_splits_against_fp64(rows, cap, hq, hkv, device):
    """Lengths 0 (the uniform average), 1, around a wave's tokens and the item's 128, and past the
    capacity; then one step with an append (out of the step equals the plain decode of the written
    cache bit for bit, slots at both ends of the cache among them)."""
    rng = np.random.default_rng(rows * 1000 + cap + hq)
    q = torch.tensor(rng.standard_normal((rows, 1, hq, 64)), device=device).to(torch.bfloat16)
    k, v = (torch.tensor(rng.standard_normal((rows, cap, hkv, 64)), device=device).to(torch.bfloat16)
            for _ in range(2))
    edge = np.array([1, cap, 0, 8, 9, 63, 65, 127, 128, 129, cap + 5, -2], np.int32)
    lengths = np.concatenate((edge, rng.integers(1, cap + 1, max(rows - edge.size, 0)))
                             )[:rows].astype(np.int32)
    tl = torch.tensor(lengths, device=device)
    out = attention.dense_cached_attention(q, k, v, tl)
    some = np.unique(np.concatenate((np.arange(min(rows, 12)), [rows - 1])))
    ref = oatt.cached_fp64(*(x[some].float().cpu().numpy() for x in (q, k, v)), lengths[some])[0]
    check_bf16(f"decode split {rows}x{cap} {hq}/{hkv}", out[some], ref)

    kn, vn = (torch.tensor(rng.standard_normal((rows, 1, hkv, 64)), device=device).to(torch.bfloat16)
              for _ in range(2))
    pos = torch.tensor(rng.integers(0, cap, rows).astype(np.int32), device=device)
    pos[0], pos[-1] = 0, cap - 1
    kc, vc = k.clone(), v.clone()
    step, kc, vc = attention.cached_attention_step(q, kn, vn, kc, vc, pos, backend="hip")
    at = torch.arange(rows, device=device)
    k[at, pos.long()], v[at, pos.long()] = kn[:, 0], vn[:, 0]
    assert torch.equal(kc, k) and torch.equal(vc, v)
    assert torch.equal(step, attention.dense_cached_attention(q, k, v, pos + 1))
