"""Which form of the encoder's attention a batch of texts takes, and the 32 x 32 form where it is not chosen."""
import pytest
import torch

from django_assistant_bot_amd.ops import native


@pytest.mark.parametrize("units,max_len,packed", [
    (12, 19, False), (4800, 64, False),  # one 64-query block
    (12, 65, False), (12, 128, False), (128, 128, False), (129, 128, True),  # 256 and 258 workgroups of 64 queries
    (12, 256, False), (64, 256, False), (65, 256, True), (12, 257, True), (2, 512, True), (4800, 512, True)])
def test_short_texts_stay_on_the_64_query_form_while_each_block_has_a_cu(units, max_len, packed):
    assert native().flash_packed64_wins(units, max_len) is packed


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[65], [64, 65, 1], [127, 128, 129, 3], [191, 192, 193], [1], [255, 256, 257]])
@pytest.mark.parametrize("Hq,Hkv", [(12, 12), (8, 2)])
def test_the_32_x_32_form_at_its_edges(lens, Hq, Hkv):
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + Hq)
    T, D = sum(lens), 64
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device="cuda", generator=g).to(torch.bfloat16)
    q, k, v = (t.unflatten(1, (-1, D)) for t in qkv.split([Hq * D, Hkv * D, Hkv * D], 1))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    out = torch.full((T + 1, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
    native().flash_packed64(q.data_ptr(), q.stride(0), D, k.data_ptr(), v.data_ptr(), k.stride(0), D, out.data_ptr(), Hq * D, D,
                            cu.data_ptr(), len(lens), max(lens), Hq, Hkv, D ** -0.5, torch.cuda.current_stream().cuda_stream)
    assert (out[T] == 7.0).all()
    s0 = 0
    for n in lens:
        qs, ks, vs = (t[s0:s0 + n].double().transpose(0, 1).contiguous() for t in (q, k, v))
        ks, vs = ks.repeat_interleave(Hq // Hkv, 0), vs.repeat_interleave(Hq // Hkv, 0)
        p = torch.softmax(torch.matmul(qs, ks.transpose(1, 2).contiguous()) * D ** -0.5, -1)
        exp = torch.matmul(p, vs).transpose(0, 1)
        # the probabilities and the result are rounded to bf16 (2^-8 each) before / after sums of |p v|
        bound = 2.0 ** -8 * (torch.matmul(p, vs.abs()).transpose(0, 1) + exp.abs()) + 1e-4
        assert ((out[s0:s0 + n].double() - exp).abs() <= bound).all()
        s0 += n
