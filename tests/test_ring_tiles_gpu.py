"""The encoder's ring kernel (gemm_small.hip) against an fp64 product: every tile at its edges, its K-slices, and
the sizes that it takes from the larger kernels."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# tile of the ring: one K-tile, fewer K-tiles than buffers, ragged rows and columns, many K-tiles
SHAPES = {0: [(1, 4, 64), (130, 388, 128)], 1: [(641, 772, 64), (641, 772, 448)], 2: [(1300, 772, 128), (1000, 1028, 448)],
          3: [(4000, 1028, 64), (641, 3076, 448)], 4: [(1300, 2308, 64), (641, 2308, 768)], 5: [(700, 3076, 1024), (3000, 772, 1024)],
          6: [(1700, 3076, 192), (1500, 3076, 448)], 7: [(2340, 3076, 128), (2600, 2308, 448)]}


def _operands(M, N, K, bias, res):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(*shape, pad=0, scale=1.0):  # a view of wider rows: strides other than the width
        t = torch.randn(*shape[:-1], shape[-1] + pad, device=DEV, generator=g) * scale
        return t.to(torch.bfloat16)[..., :shape[-1]]

    return rnd(M, K, pad=8), rnd(N, K, pad=16, scale=K ** -0.5), rnd(N) if bias else None, rnd(M, N, pad=4) if res else None


def _check(got, A, B, b, r, gelu):
    exp = A.double() @ B.double().t()
    if b is not None:
        exp = exp + b.double()
    if gelu:
        exp = torch.nn.functional.gelu(exp)
    # two roundings to bf16 (2^-8 of the value each: the product's and, with a residual, the sum's) and fp32 sums of K
    # products of size about K^-1/2 (error far below 1e-4 at these K)
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if r is not None:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got.double() - exp).abs() <= tol).all()


@pytest.mark.parametrize("tile,M,N,K", [(t, *s) for t, v in SHAPES.items() for s in v])
@pytest.mark.parametrize("gelu,bias,res", [(False, True, True), (True, True, False), (False, False, False)])
def test_every_tile(tile, M, N, K, gelu, bias, res):
    nat = ops.native()
    A, B, b, r = _operands(M, N, K, bias, res)
    wide = torch.empty(M + 1, N + 12, dtype=torch.bfloat16, device=DEV).fill_(7.0)
    out = wide[:M, :N]
    p = lambda t: 0 if t is None else t.data_ptr()  # noqa: E731
    nat.gemm_small(p(A), A.stride(0), p(B), B.stride(0), p(out), out.stride(0), p(b), p(r), 0 if r is None else r.stride(0), M, N, K,
                   int(gelu), nat.RING_TILE + 16 + tile, torch.cuda.current_stream().cuda_stream)
    _check(out, A, B, b, r, gelu)
    assert (wide[M:] == 7.0).all() and (wide[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K,slices,tile", [(1807, 384, 1536, 2, 2), (2029, 384, 1536, 2, 4), (1955, 768, 3072, 2, 5), (2695, 384, 1600, 3, 4)])
def test_slices(M, N, K, slices, tile):
    nat = ops.native()
    assert nat.slab_slices(M, N, K) == slices
    A, B, _, _ = _operands(M, N, K, False, False)
    A, B = A.contiguous(), B.contiguous()
    slabs = torch.full((slices + 1, M, N), 7.0, device=DEV)
    nat.gemm_slab(A.data_ptr(), B.data_ptr(), slabs.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream, tile)
    cut = [K // 64 * i // slices * 64 for i in range(slices + 1)]
    for i in range(slices):
        exp = A[:, cut[i]:cut[i + 1]].double() @ B[:, cut[i]:cut[i + 1]].double().t()
        assert (slabs[i].double() - exp).abs().max() <= 1e-4  # fp32 sums
    assert (slabs[slices] == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(6400, 768, 768), (5300, 1152, 384), (9000, 1000, 768)])
@pytest.mark.parametrize("shift", [0, 4])
def test_sizes_taken_from_the_larger_kernels(M, N, K, shift):
    """Rows that the ring's copies do not take (8 bytes off a 16-byte line) stay on those kernels, which do."""
    assert ops.kernels.small_tile(M, N, K) == -1 and ops.native().ring_wins(M, N, K, 0, 1)
    A, B, b, r = _operands(M, N, K, True, True)
    if shift:
        wide = torch.zeros(M, K + 8, dtype=torch.bfloat16, device=DEV)
        wide[:, shift:K + shift] = A
        A = wide[:, shift:K + shift]
    assert A.data_ptr() % 16 == 2 * shift
    _check(ops.gemm_bt(A, B, bias=b, residual=r), A, B, b, r, False)


@pytest.mark.parametrize("M,N,K", [(300, 768, 768), (1300, 3072, 768), (2200, 768, 3072), (9000, 1152, 384)])
def test_the_choice_of_a_tile_changes_no_bits(M, N, K):
    nat, s = ops.native(), torch.cuda.current_stream().cuda_stream
    A, B, b, r = _operands(M, N, K, True, True)

    def run(tile):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        nat.gemm_small(A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), out.data_ptr(), N, b.data_ptr(), r.data_ptr(), r.stride(0),
                       M, N, K, 0, tile, s)
        return out

    exp = run(nat.RING_TILE)
    assert all(torch.equal(run(nat.RING_TILE + 16 + t), exp) for t in SHAPES)
