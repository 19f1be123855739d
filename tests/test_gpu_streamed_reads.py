"""Forward passes of 192 MiB and more read their rows as streams: the bits of the smaller calls."""

import pytest
import torch

from mfattn.kernels import convolution, prologue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [5, 6, 7, 8])  # 24 MiB a row: eight are at the line
def test_prologue_rows_equal_rows_alone(rows, device):
    gen = torch.Generator(device=device).manual_seed(rows)
    q, k = (torch.randn((rows, 4096, h, 64), generator=gen, device=device).bfloat16() for h in (16, 8))
    gain = torch.ones(64, device=device, dtype=torch.bfloat16)
    whole = prologue.qk_norm_rope(q, k, gain, gain, None, eps=1e-5, rope_theta=1e6)
    for r in (0, rows - 1):
        one = slice(r, r + 1)
        alone = prologue.qk_norm_rope(q[one], k[one], gain, gain, None, eps=1e-5, rope_theta=1e6)
        assert all(torch.equal(w[one], a) for w, a in zip(whole, alone))


@pytest.mark.parametrize("taps", [1, 3, 8])
@pytest.mark.parametrize("tokens", [4095, 4129, 6143, 6145])
def test_conv_rows_equal_rows_alone(taps, tokens, device):
    """Four rows of 1024 channels in four tensors are either side of 192 MiB at 6144 tokens."""
    gen = torch.Generator(device=device).manual_seed(taps)
    b, c, v = (torch.randn((4, tokens, 1024), generator=gen, device=device).bfloat16() for _ in range(3))
    w = torch.randn((1024, taps), generator=gen, device=device).bfloat16()
    seg = (torch.arange(tokens, device=device, dtype=torch.int32) // 37 + 1).repeat(4, 1)
    whole = convolution.gated_depthwise_convolution_segmented(b, c, v, w, seg, kernel_size=taps)
    for r in (0, 3):
        one = slice(r, r + 1)
        alone = convolution.gated_depthwise_convolution_segmented(b[one], c[one], v[one], w, seg[one],
                                                                  kernel_size=taps)
        assert torch.equal(whole[one], alone)
