"""The attention inside the encoder's output projection against the two launches it stands for."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

LENGTHS = [[1], [15], [16], [17], [19], [31, 1], [32], [33], [5, 0, 28], [64], [1] * 64, [7, 30, 3, 20], [0, 31, 0, 1, 0],
           [2] + [0] * 80 + [9]]


@pytest.mark.parametrize("H,D", [(64, 64), (384, 32), (768, 64), (1024, 64)])
@pytest.mark.parametrize("lens", LENGTHS, ids=lambda v: "-".join(map(str, v))[:24])
def test_attention_in_the_projection(H, D, lens):
    T, g = sum(lens), torch.Generator().manual_seed(H + sum(lens) + len(lens))
    if T > 32 and H > 768:
        pytest.skip("two launches")
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    qkv, w, b, x = r(T, 3 * H) * 2, r(H, H) * H ** -0.5, r(H), r(T, H)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device=DEV)
    q, k, v = (t.view(T, H // D, D) for t in qkv.split(H, 1))
    att = ops.flash_attention_packed(q, k, v, cu, cu, max(lens)).view(T, H)
    out = torch.full((T + 1, H), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.native().gemm_attn(qkv.data_ptr(), cu.data_ptr(), len(lens), D, D ** -0.5, w.data_ptr(), b.data_ptr(), x.data_ptr(),
                           out.data_ptr(), T, H, torch.cuda.current_stream().cuda_stream)
    assert (out[T] == 7.0).all()
    # the attention's bits are the same; the projection's fp32 sums differ in their order (H 2^-23 of the sum of their
    # terms' sizes), which its rounding and that of the sum with x can make one step of 2^-8 each
    y = att.double() @ w.double().t() + b.double()
    slack = (att.double().abs() @ w.double().abs().t() + b.double().abs()) * H * 2.0 ** -23
    exp = (y.to(torch.bfloat16).double() + x.double())
    assert ((out[:T].double() - exp).abs() <= y.abs() * 2.0 ** -8 + exp.abs() * 2.0 ** -8 + 2 * slack).all()


def test_sizes_that_are_left_to_two_launches():
    for T, H, D, batch in ((65, 768, 64, 1), (8, 768, 128, 1), (8, 1088, 64, 1), (8, 96, 32, 1), (8, 768, 64, 0), (33, 1024, 64, 1)):
        with pytest.raises(RuntimeError):
            ops.native().gemm_attn(16, 16, batch, D, 1.0, 16, 16, 16, 16, T, H, 0)
