"""bf16 decode of 3, 5, 6 and 7 query heads per KV head: fp32 probabilities in every split."""

import pytest
import torch

from mfattn.kernels import attention

pytestmark = pytest.mark.gpu


def _fp64(q, k, v, lengths):
    g = q.shape[2] // k.shape[2]
    out = []
    for b, n in enumerate(lengths):
        kk, vv = (x[b, :n].double().repeat_interleave(g, 1) for x in (k, v))
        p = torch.softmax((q[b].double() * kk).sum(-1) * 0.125, 0)
        out.append((p[..., None] * vv).sum(0))
    return torch.stack(out)


# rows x ceil(capacity / 128) items: the most waves an item, four (with and without a combine
# launch), one
@pytest.mark.parametrize("rows, cap", [(2, 1000), (260, 100), (40, 1100), (600, 100)])
@pytest.mark.parametrize("hq, hkv", [(24, 8), (40, 8), (48, 8), (56, 8), (12, 4), (28, 4), (10, 2),
                                     (6, 2), (7, 1), (5, 1)])
def test_error_is_the_rounding_of_the_output(rows, cap, hq, hkv, device):
    """The error against float64 is what rounding the float64 result to bf16 costs, within 2 %:
    probabilities, sums and products in fp32 are good to 1e-6, which moves a value across a
    rounding boundary 2**-8 apart in less than one case of a thousand; probabilities rounded to
    bf16 made the error 10 to 40 % larger."""
    gen = torch.Generator(device=device).manual_seed(rows + cap + hq)
    q, k, v = (torch.randn(s, generator=gen, device=device).bfloat16()
               for s in ((rows, 1, hq, 64), (rows, cap, hkv, 64), (rows, cap, hkv, 64)))
    lengths = torch.randint(cap // 2, cap + 1, (rows,), generator=gen, device=device,
                            dtype=torch.int32)
    out = attention.dense_cached_attention(q, k, v, lengths)[:, 0]
    some = list(range(0, rows, max(1, rows // 12)))
    ref = _fp64(q[some], k[some], v[some], lengths[some].tolist())
    rounding = (ref.bfloat16().double() - ref).norm()
    assert (out[some].double() - ref).norm() <= 1.02 * rounding


@pytest.mark.parametrize("rows, length", [(1, 37), (1, 1), (260, 61), (600, 77)])
@pytest.mark.parametrize("hq, hkv", [(24, 8), (12, 4), (10, 2), (7, 1)])
def test_an_infinite_last_value_stays_infinite(rows, length, hq, hkv, device):
    """A row's last value is infinite in one dimension: so is the output there, and only there
    (a load past the end that reads the last token again must not weigh it with 0)."""
    gen = torch.Generator(device=device).manual_seed(length)
    q, k, v = (torch.randn(s, generator=gen, device=device).bfloat16()
               for s in ((rows, 1, hq, 64), (rows, 100, hkv, 64), (rows, 100, hkv, 64)))
    v[:, length - 1, 0, 5] = float("inf")
    lengths = torch.full((rows,), length, dtype=torch.int32, device=device)
    out = attention.dense_cached_attention(q, k, v, lengths)[:, 0].float()
    inf = torch.zeros_like(out, dtype=torch.bool)
    inf[:, : hq // hkv, 5] = True
    assert (out[inf] == float("inf")).all() and torch.isfinite(out[~inf]).all()
