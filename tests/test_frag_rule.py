"""Which prefill projections gemm_frag takes, and in how many K-slices."""
from types import SimpleNamespace

import pytest
import torch

from django_assistant_bot_amd.models import LlamaModel
from django_assistant_bot_amd.ops import kernels
from django_assistant_bot_amd.ops.kernels import frag_plan, frag_slices, native


# faster there by measurement; slower, or outside what was measured (rows, N, K)
@pytest.mark.parametrize("M,N,K,takes", [(260, 2048, 2048, True), (515, 3072, 2048, True), (260, 6144, 4096, True), (1093, 2048, 2048, True),
                                         (140, 28672, 4096, True), (1093, 28672, 4096, False), (1093, 4096, 14336, False),
                                         (700, 10240, 8192, False), (2300, 4096, 4096, False), (64, 2048, 2048, False),
                                         (300, 768, 2048, False), (300, 2048, 512, False), (5000, 2048, 2048, False)])
def test_plan(M, N, K, takes):
    assert (frag_plan(M, N, K)[0][0] == "frag") == takes
    assert frag_plan(M, N, K, True, False)[0][0] != "frag"


def test_slices():
    assert frag_slices(260, 2048, 8192) > 1 and frag_slices(140, 4096, 14336) > 1
    assert frag_slices(1093, 4096, 14336) == frag_slices(400, 2048, 2048) == frag_slices(3000, 4096, 4096) == 0
    for M, N, K in ((3000, 4096, 6848), (3300, 4096, 6848), (2048, 6144, 1088), (3500, 4096, 1600)):  # no estimate of the whole product
        assert frag_plan(M, N, K) is None and frag_slices(M, N, K) == 0
    for M, N, K in ((140, 1024, 1024), (260, 2048, 8192), (515, 2048, 8192), (260, 4096, 14336)):
        s = frag_slices(M, N, K)
        assert s == 0 or K // 64 >= 4 * s


@pytest.mark.parametrize("slices", [0, 17])
def test_estimate_of_no_product(slices):
    assert native().frag_us(300, 2048, 1024, slices) == float("inf")


# tiles of 192 rows where they leave fewer rows past the prompt's end; else 128 or 256
@pytest.mark.parametrize("M,N,K,kind", [(768, 4096, 14336, "192"), (1300, 6144, 4096, "192"), (2300, 4096, 4096, "192"), (560, 16384, 2048, "192"),
                                        (400, 4096, 14336, "mid"), (1900, 4096, 14336, "mid"), (1093, 6144, 4096, "mid"), (700, 2304, 2048, "mid")])
def test_rows_of_a_tile(M, N, K, kind):
    assert frag_plan(M, N, K, True, False)[0][0] == kind


# a step's projections leave the stream only for sizes that gemm_bt gives to gemm_frag: whole 256 weight rows (qkv, hidden, MLP)
@pytest.mark.parametrize("qkv,hidden,mlp,serves", [(6144, 4096, 14336, True), (3072, 2048, 8192, True), (3200, 1920, 5120, False), (6528, 2176, 5888, False),
                                                   (3200, 2048, 8192, False), (3072, 1920, 8192, False), (1152, 896, 4864, False)])
def test_steps_that_are_not_streamed(qkv, hidden, mlp, serves):
    layer = SimpleNamespace(**{n: torch.empty(s, device="meta") for n, s in (("qkv_w", (qkv, hidden)), ("o_w", (hidden, hidden)), ("down_w", (hidden, mlp)))})
    model = SimpleNamespace(layers=[layer])
    for T in (129, 200, 256):
        assert LlamaModel._frag_serves(model, T) == serves


# a whole product runs on the operands themselves (views of them are host time that short prompts wait for), parts on theirs
def test_parts_of_a_plan(monkeypatch):
    calls = []
    monkeypatch.setattr(kernels, "gemm_frag", lambda a, b, **kw: calls.append((a, b, kw["out"], kw["residual"])))
    monkeypatch.setattr(kernels, "_gemm256_into", lambda a, b, o, bias, r, *rest: calls.append((a, b, o, r)))
    A, B, out, r = torch.zeros(600, 64), torch.zeros(512, 64), torch.zeros(600, 512), torch.zeros(600, 512)
    kernels._run_frag_plan((("frag", 600, 512), None), A, B, out, r, kernels.EPI_NONE, 1, None)
    assert all(x is y for x, y in zip(calls.pop(), (A, B, out, r)))
    for plan, cut in (((("256", 512, 512), ("frag", 88, 512)), (512, 0)), ((("256", 600, 256), ("frag", 600, 256)), (0, 256))):
        kernels._run_frag_plan(plan, A, B, out, r, kernels.EPI_NONE, 1, None)
        m, n = cut
        for got, (rows, cols) in zip(calls, ((slice(0, m or 600), slice(0, n or 512)), (slice(m, 600), slice(n, 512)))):
            for x, y in zip(got, (A[rows], B[cols], out[rows, cols], r[rows, cols])):
                assert x.data_ptr() == y.data_ptr() and x.shape == y.shape and x.stride() == y.stride()
        del calls[:]


# with gemm_frag behind the waves, too, the parts are the product
def test_plans_with_gemm_frag_behind_the_waves():
    seen = 0
    for M in (641, 700, 1100, 1200, 1280, 2420, 3100, 3500, 4097, 4200, 5000, 5500, 5900):
        for N, K in ((2048, 2048), (4096, 4096), (6144, 4096), (8192, 2048), (16384, 2048), (28672, 4096)):
            for cols in (True, False):
                plan = frag_plan(M, N, K, cols)
                if plan is None or plan[1] is None or plan[1][0] != "frag":
                    continue
                (_, m, n), (_, m2, n2) = plan
                assert (m == m2 == M and n + n2 == N and cols) or (n == n2 == N and m + m2 == M)
                assert n % 256 == 0 and (m == M or m % 256 == 0)
                seen += 1
    assert seen > 10
