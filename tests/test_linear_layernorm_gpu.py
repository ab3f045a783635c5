"""A projection in K-slices that the LayerNorm behind it sums, and the sizes that are left to one launch."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# ends of the four ranges of the rule (tiles of 64 or 128, two or three slices), whole tiles and one row more or less, K whose
# slices are not equal
SIZES = [(705, 768, 3072, 3), (896, 768, 3072, 3), (1024, 768, 2048, 2), (897, 768, 2624, 2), (960, 768, 3072, 2), (1344, 768, 1536, 2), (1345, 768, 3072, 3),
         (1792, 768, 3072, 3), (1921, 768, 3072, 2), (2688, 768, 1536, 2), (1793, 384, 1536, 2), (2689, 384, 1600, 3),
         (5376, 384, 1536, 2), (575, 1024, 4096, 3), (1280, 1024, 4096, 3), (2048, 1024, 4096, 2)]


@pytest.mark.parametrize("M,N,K,slices", SIZES)
def test_slices_against_64_bits(M, N, K, slices):
    assert ops.native().slab_slices(M, N, K) == slices
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    x, w, b, res, gain, off = r(M, K), r(N, K) * K ** -0.5, r(N), r(M, N), 1 + r(N) * 0.25, r(N)
    got = ops.linear_layernorm(x, w, b, res, gain, off, 1e-12).double()
    z = x.double() @ w.double().t() + b.double() + res.double()
    exp = torch.nn.functional.layer_norm(z, (N,), gain.double(), off.double(), 1e-12)
    # fp32 sums over K, twice those over N (2^-24 a step of the sum of the terms' sizes), over the row's deviation; one rounding
    mags = (x.double().abs() @ w.double().abs().t()).amax(1, keepdim=True) + 8
    slack = (K + 2 * N) * 2.0 ** -24 * mags / z.std(1, keepdim=True) * (gain.double().abs() + exp.abs())
    assert ((got - exp).abs() <= 2.0 ** -8 * exp.abs() + slack).all()


def test_other_sizes_and_operands_take_two_launches():
    for M, N, K in ((704, 768, 3072), (961, 768, 3072), (1344, 768, 3072), (1000, 768, 2112), (900, 768, 768), (900, 512, 3072), (0, 768, 3072), (3100, 768, 3072), (900, 768, 1535), (769, 1024, 4096)):
        assert ops.native().slab_slices(M, N, K) == 0
    g = torch.Generator(device=DEV).manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    x, w, b, res, gain, off = r(832, 3072), r(768, 3072), r(768), r(832, 1536)[:, :768], r(768), r(768)
    exp = ops.layernorm(ops.linear(x, w, b, residual=res), gain, off, 1e-12)  # (the residual's rows lie 1536 apart)
    assert torch.equal(ops.linear_layernorm(x, w, b, res, gain, off, 1e-12), exp)
