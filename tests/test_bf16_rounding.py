"""fp32 -> bf16 on the hardware's conversion, bit for bit as torch rounds."""

import pytest
import torch

import mlc


class Narrow(torch.nn.Module):
    def forward(self, x):
        return x.to(torch.bfloat16)


@pytest.mark.gpu
def test_every_upper_half_with_the_halves_that_decide_rounding():
    """Every sign, exponent and upper mantissa (subnormals, infinities, NaN
    among them) with lower halves below, at and above the tie."""
    high = torch.arange(1 << 16, dtype=torch.int64) << 16
    low = torch.tensor([0, 1, 0x7fff, 0x8000, 0x8001, 0xffff])
    bits = (high[:, None] + low[None]).reshape(-1)
    x = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32).view(torch.float32)
    got = mlc.compile(Narrow(), (x.cuda(),))(x.cuda()).cpu()
    want = x.to(torch.bfloat16)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])
