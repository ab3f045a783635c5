"""The epilogues' exact-erf GELU over every bf16 value that it can tell apart."""
import pytest
import torch

from django_assistant_bot_amd import ops


@pytest.mark.gpu
def test_gelu_against_64_bits():
    bits = torch.arange(1 << 16, dtype=torch.int32, device="cuda").to(torch.int16)
    x = bits.view(torch.bfloat16)
    x = x[torch.isfinite(x.float())]
    x = torch.cat([x, x.new_zeros(-len(x) % 64)])
    got = ops.gelu(x.view(-1, 64)).view(-1).double()
    exp = x.double() * 0.5 * torch.special.erfc(-x.double() * 2 ** -0.5)
    err = (got - exp).abs()
    # the rounding to bf16 (2^-8 of the value), and the polynomial's relative error, largest where the result is smallest
    for low, rel in ((-1.0, 1e-6), (-3.0, 5e-5), (-6.0, 2e-3), (-12.0, 2e-2)):
        at = x.double() >= low
        # (a value below 2^-126 may be flushed)
        assert (err[at] <= (2.0 ** -8 + rel) * exp[at].abs() + 2.0 ** -126).all()
    assert (err[x.double() < -12.0] <= 1e-30).all()
