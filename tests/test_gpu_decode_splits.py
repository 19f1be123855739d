"""The row decode's splits of an item (one wave, four, the most) at the lines between them."""

import numpy as np
import pytest
import torch

from _helpers import check_bf16
from mfattn.kernels import attention
from oracle import attention as oatt

pytestmark = pytest.mark.gpu


# rows x ceil(capacity / 128) items: up to 256 the most waves an item, up to 512 four, then one;
# up to 128 slots an item of several waves writes the output itself
@pytest.mark.parametrize("rows, cap", [(3, 127), (3, 128), (3, 129), (128, 200), (129, 200),
                                       (256, 130), (257, 130), (256, 128), (300, 128), (300, 100),
                                       (512, 64), (513, 64)])
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


@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("hkv, rows, cap", [(8, 520, 260), (4, 520, 520), (2, 1030, 520),
                                            (1, 1030, 1024)])
def test_caches_that_stream_v(hkv, rows, cap, group, device):
    """K and V of 264 to 277 MiB, above the 256 MiB from which V streams too, one wave an item:
    a plain decode against float64 on some rows, and a step with an append (the decode of the
    written cache, bit for bit)."""
    assert rows * cap * hkv * 64 * 4 > 256 << 20
    hq = hkv * group
    gen = torch.Generator(device=device).manual_seed(hq + cap)
    mk = lambda *s: torch.randn(s, generator=gen, device=device).bfloat16()  # noqa: E731
    q, kn, vn = mk(rows, 1, hq, 64), mk(rows, 1, hkv, 64), mk(rows, 1, hkv, 64)
    k, v = mk(rows, cap, hkv, 64), mk(rows, cap, hkv, 64)
    lengths = torch.randint(1, cap + 1, (rows,), generator=gen, device=device, dtype=torch.int32)
    lengths[:4] = torch.tensor([cap, 0, 1, 129], dtype=torch.int32)
    out = attention.dense_cached_attention(q, k, v, lengths)
    some = [0, 1, 2, 3, 7, rows // 2, rows - 1]
    ref = oatt.cached_fp64(*(x[some].float().cpu().numpy() for x in (q, k, v)),
                           lengths[some].cpu().numpy())[0]
    check_bf16(f"decode streamed {hq}/{hkv}", out[some], ref)
    pos = (lengths - 1).clamp(min=0)
    step, kc, vc = attention.cached_attention_step(q, kn, vn, k, v, pos, backend="hip")
    at = torch.arange(rows, device=device)
    assert torch.equal(kc[at, pos.long()], kn[:, 0]) and torch.equal(vc[at, pos.long()], vn[:, 0])
    assert torch.equal(step, attention.dense_cached_attention(q, kc, vc, pos + 1))
