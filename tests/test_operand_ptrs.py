"""The native look at a call's operands against the same questions asked one attribute at a time."""
import pytest
import torch

from django_assistant_bot_amd import ops

bf = torch.bfloat16
SHAPES = ((6, 4), (6,), (1, 4))


def good():
    return [torch.zeros(s, dtype=bf) for s in SHAPES]


def by_attribute(rows, dev):
    out = []
    for row in rows:
        for t, s in zip(row, SHAPES):
            if t.shape != s or t.dtype != bf or not t.is_contiguous() or t.device != dev:
                return None
            out.append(t.data_ptr())
    return out


FORMS = {
    "contiguous": lambda: torch.zeros(6, 4, dtype=bf),
    "part of a storage": lambda: torch.zeros(9, 4, dtype=bf)[2:8],
    "parameter": lambda: torch.nn.Parameter(torch.zeros(6, 4, dtype=bf), requires_grad=False),
    "transposed": lambda: torch.zeros(4, 6, dtype=bf).t(),
    "row stride": lambda: torch.zeros(6, 8, dtype=bf)[:, :4],
    "expanded": lambda: torch.zeros(1, 4, dtype=bf).expand(6, 4),
    "half": lambda: torch.zeros(6, 4, dtype=torch.half),
    "fp32": lambda: torch.zeros(6, 4),
    "other shape": lambda: torch.zeros(4, 6, dtype=bf),
    "one more axis": lambda: torch.zeros(6, 4, 1, dtype=bf),
    "meta": lambda: torch.zeros(6, 4, dtype=bf, device="meta"),
    "conjugate": lambda: torch.zeros(6, 4, dtype=torch.complex64).conj(),
}


@pytest.mark.parametrize("form", FORMS)
def test_operands(form):
    api = getattr(torch.Tensor, "__dlpack_c_exchange_api__", None)
    if api is None:
        pytest.skip("this torch has no exchange table")
    rows = [tuple(good()), (FORMS[form](), *good()[1:])]
    like = torch.zeros(3, dtype=torch.int32)
    got = ops.native().operand_ptrs(api, torch.Tensor, like, rows, SHAPES)
    assert got == by_attribute(rows, like.device)


def test_operands_that_are_left_to_the_caller():
    """What the table does not describe, or is no tensor, is None: the caller asks one by one."""
    api = getattr(torch.Tensor, "__dlpack_c_exchange_api__", None)
    if api is None:
        pytest.skip("this torch has no exchange table")
    like, ptrs = torch.zeros(3, dtype=torch.int32), ops.native().operand_ptrs
    assert ptrs(api, torch.Tensor, like, [tuple(good())[:2]], SHAPES) is None
    assert ptrs(api, torch.Tensor, like, [(None, *good()[1:])], SHAPES) is None
    assert ptrs(api, torch.Tensor, like, [good()], SHAPES) is None
    grad = torch.zeros(6, 4, dtype=bf, requires_grad=True)
    rows = [(grad, *good()[1:])]
    assert ptrs(api, torch.Tensor, like, rows, SHAPES) in (None, by_attribute(rows, like.device))
    assert ptrs(api, torch.Tensor, like, [], SHAPES) == []
