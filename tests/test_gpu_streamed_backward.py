"""Backward passes of 256 MiB and more access their rows as streams: the bits of smaller calls."""

import pytest
import torch

from mfattn.kernels import convolution, prologue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("centered", [False, True])
@pytest.mark.parametrize("taps, dtype", [(1, torch.bfloat16), (3, torch.bfloat16), (4, torch.bfloat16),
                                         (5, torch.bfloat16), (3, torch.float32)])
def test_conv_rows_equal_rows_alone(taps, dtype, centered, device):
    """Inputs and gradients (seven tensors) are 256 MiB from 18725 rows of 1024 bf16 channels on:
    five rows of 3851 tokens are above the line, one row alone below it.  fp32 rows are half as
    long."""
    tokens = 3851 if dtype is torch.bfloat16 else 1931
    gen = torch.Generator(device=device).manual_seed(taps)
    b, c, v, do = (torch.randn((5, tokens, 1024), generator=gen, device=device).to(dtype)
                   for _ in range(4))
    w = torch.randn((1024, taps), generator=gen, device=device).to(dtype)
    seg = (torch.arange(tokens, device=device, dtype=torch.int32) // 37 + 1).repeat(5, 1)

    def grads(rows):
        leaves = [x[rows].clone().requires_grad_() for x in (b, c, v)]
        if centered:
            out = convolution.gated_centered_convolution(*leaves, w, seg[rows])
        else:
            out = convolution.gated_depthwise_convolution_segmented(*leaves, w, seg[rows],
                                                                    kernel_size=taps)
        return torch.autograd.grad(out, leaves, do[rows])

    whole = grads(slice(0, 5))
    for r in (0, 4):
        for name, x, y in zip("bcv", whole, grads(slice(r, r + 1))):
            assert torch.equal(x[r:r + 1], y), (name, r)


def test_prologue_rows_equal_rows_alone(device):
    """Rows, gradients and results of 16/8 heads are 256 MiB from 29128 tokens on: eight rows of
    3700 are above the line, one row alone below it."""
    gen = torch.Generator(device=device).manual_seed(1)
    q, k, dq, dk = (torch.randn((8, 3700, h, 64), generator=gen, device=device).bfloat16()
                    for h in (16, 8, 16, 8))
    gain = torch.ones(64, device=device, dtype=torch.bfloat16)

    def grads(rows):
        leaves = [x[rows].clone().requires_grad_() for x in (q, k)]
        out = prologue.qk_norm_rope(*leaves, gain, gain, None, eps=1e-5, rope_theta=1e6)
        return torch.autograd.grad(out, leaves, (dq[rows], dk[rows]))

    whole = grads(slice(0, 8))
    for r in (0, 7):
        assert all(torch.equal(x[r:r + 1], y) for x, y in zip(whole, grads(slice(r, r + 1)))), r
