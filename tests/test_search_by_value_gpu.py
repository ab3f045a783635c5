"""A search's small host tensors in its launches' arguments (search.hip) against the same from tensors of the device."""
import numpy as np
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.engine.vector_index import VectorIndex

pytestmark = pytest.mark.gpu
DEV = "cuda"


# groups around a wave and at the most that a launch takes; words around a thread's four and a workgroup's 1024
@pytest.mark.parametrize("rows,groups,words", [(1, 1, 0), (1, 0, 1), (3, 64, 3), (3, 65, 5), (128, 128, 1023), (2, 128, 1024), (130, 0, 1025),
                                               (2, 2, 70_001)])
def test_unit_queries_writes_groups_and_clears(rows, groups, words):
    g = torch.Generator(device=DEV).manual_seed(rows + words)
    x = torch.randn(rows, 768, device=DEV, generator=g)
    host = torch.randint(-2 ** 31, 2 ** 31 - 1, (groups,), dtype=torch.int64).to(torch.int32) if groups else None
    room = torch.full((words + 64,), -1, dtype=torch.int32, device=DEV)
    q, there = ops.unit_queries(x, host, room[:words] if words else None)
    assert torch.equal(q, ops.unit_rows(x)) and not room[:words].any() and (room[words:] == -1).all()
    assert there is None if host is None else torch.equal(there.cpu(), host)


def test_unit_queries_takes_no_more_values_than_fit():
    x = torch.zeros(2, 64, device=DEV)
    for bad in (torch.zeros(129, dtype=torch.int32), torch.zeros(2, dtype=torch.int64), torch.zeros(2, dtype=torch.int32, device=DEV)):
        with pytest.raises(ValueError):
            ops.unit_queries(x, bad)


@pytest.mark.parametrize("n", [1, 32, 255, 257, 70_001])
@pytest.mark.parametrize("queries", [1, 128, 129])
def test_limits_of_the_host(n, queries):
    docs = torch.arange(n, device=DEV) // 3 - 5
    limits = torch.randint(-6, n // 3 + 2, (queries,))
    limits[0] = -2 ** 63
    limits[-1] = 2 ** 63 - 1
    start = torch.randint(-2 ** 31, 2 ** 31, (queries, (n + 31) // 32), device=DEV).to(torch.int32)
    for mask in (None, start):
        exp = ops.doc_lt_bits(docs, limits.to(DEV), None if mask is None else mask.clone())
        if queries > ops.native().HOST_VALUES:
            with pytest.raises(ValueError):
                ops.doc_lt_bits(docs, limits, None if mask is None else mask.clone())
        else:
            assert torch.equal(ops.doc_lt_bits(docs, limits, None if mask is None else mask.clone()), exp)


# queries around what the arguments hold, of an index that selects (20,000 rows)
@pytest.mark.parametrize("queries", [1, 128, 129])
@pytest.mark.parametrize("form", ["list", "host", "strided", "pinned", "device"])
def test_filters_of_any_form(queries, form):
    n = 20_000
    idx = VectorIndex(256, DEV, capacity=n)
    g = torch.Generator(device=DEV).manual_seed(queries)
    idx.add(np.arange(n), torch.randn(n, 256, device=DEV, generator=g), doc_ids=np.arange(n) // 4, groups=np.arange(n) % 3)
    q = torch.randn(queries, 256, device=DEV, generator=g)
    groups, limits = torch.arange(queries, dtype=torch.int32) % 4 - 1, 100 + 37 * torch.arange(queries)
    allowed = [np.arange(i % 7, n, 2 + i % 5) for i in range(queries)]
    s = idx.scores(q, groups.to(DEV))
    lists = torch.zeros(queries, n, dtype=torch.bool, device=DEV)
    for i, ids in enumerate(allowed):
        lists[i, torch.from_numpy(ids).to(DEV)] = True
    below = torch.arange(n, device=DEV)[None] // 4 < limits.to(DEV)[:, None]

    def of(t):
        return {"list": t.tolist(), "host": t, "strided": t.repeat_interleave(2)[::2], "pinned": t.pin_memory(),
                "device": t.to(DEV) if t.dtype == torch.int32 else t}[form]
    for kw, live in ((dict(), torch.ones_like(lists)), (dict(allowed=iter(allowed)), lists), (dict(doc_lt=of(limits)), below),
                     (dict(allowed=tuple(allowed), doc_lt=of(limits)), lists & below)):
        vals, ids, docs = idx.search(q, 30, q_groups=of(groups), **kw)
        exp = s.masked_fill(~live, float("-inf"))
        top = exp.topk(30, dim=1).values
        hit = ~torch.isinf(top)
        assert torch.equal(~torch.isinf(vals), hit) and torch.equal(ids >= 0, hit)
        assert ((vals - top)[hit].abs() <= 256 * 2.0 ** -22).all()  # two fp32 sums of 256 products of unit vectors
        at = exp.gather(1, ids.clamp(min=0))
        assert ((vals - at)[hit].abs() <= 256 * 2.0 ** -22).all() and torch.equal(docs[hit], ids[hit] // 4)


def test_empty_lists_allow_nothing():
    idx = VectorIndex(256, DEV, capacity=64)
    idx.add(np.arange(50), torch.randn(50, 256, device=DEV))
    q = torch.randn(2, 256, device=DEV)
    for allowed in ([[], []], [np.empty(0, np.int64), {99}], [[], [7]]):
        vals, ids, docs = idx.search(q, 5, allowed=allowed)
        assert ids[0].eq(-1).all() and ids[1].tolist() == ([7] if allowed[1] == [7] else [-1]) + [-1] * 4
    idx.remove(np.arange(50))
    assert idx.search(q, 5, allowed=[[1], [2]])[1].eq(-1).all()


# rows that are no whole fours and around a mask's words; queries around a fragment and the most that the scan takes
@pytest.mark.parametrize("dim,queries", [(256, 1), (256, 256), (512, 17), (768, 128), (1024, 2)])
@pytest.mark.parametrize("rows", [1, 5, 31, 33, 8190, 20_003])
def test_one_call_is_its_launches(rows, dim, queries):
    n, k = (max(rows, 4) + 3) // 4 * 4, min(max(rows // 3, 1), 60)
    g = torch.Generator(device=DEV).manual_seed(rows + dim)
    frag = ops.shuffle_weights(ops.unit_rows(torch.randn(-(-n // 128) * 128, dim, device=DEV, generator=g)))
    group, docs = (torch.arange(n, device=DEV) % 3).to(torch.int32), torch.arange(n, device=DEV) // 4
    group[rows:] = -1
    ids = torch.randperm(n, device=DEV, generator=g) + 9
    keys, order = ids[:rows].sort()
    x = torch.randn(queries, dim + 8, device=DEV, generator=g)[:, 8:]
    few = queries <= ops.native().HOST_VALUES
    groups = (torch.arange(queries) % 4 - 1).to(torch.int32) if few else None
    limits = torch.randint(0, rows // 4 + 2, (queries,)) if few else None
    lens = torch.randint(0, rows + 1, (queries,))
    off = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(DEV)
    flat = ids[torch.randint(0, n, (int(off[-1]),), device=DEV)]
    words = (rows + 31) // 32
    for gq, lists, lim in ((None, None, None), (groups, None, None), (None, True, None), (None, None, limits), (groups, True, limits)):
        lists = lists and (flat, off, int(lens.max()), keys, order)
        allow = None if lists is None else ops.allow_bits(*lists, words)
        if lim is not None:
            allow = ops.doc_lt_bits(docs[:rows], lim.to(DEV), allow)
        s, p = ops.scores_and_parts(ops.unit_rows(x), frag, n, group, None if gq is None else gq.to(DEV), allow)
        for got, exp in zip(ops.selected_search(x, frag, rows, group, ids, docs, k, gq, lists, lim), ops.top_hits(s, p, k, ids, docs)):
            assert torch.equal(got, exp)


def test_one_call_refuses_rows_that_its_launches_would_not_take():
    frag, x = torch.zeros(128, 256, dtype=torch.bfloat16, device=DEV), torch.zeros(2, 256, device=DEV)
    group, ids = torch.zeros(8, dtype=torch.int32, device=DEV), torch.zeros(8, dtype=torch.int64, device=DEV)
    wide = torch.zeros(8, 2, dtype=torch.int64, device=DEV)[:, 0]
    two = torch.zeros(3, dtype=torch.int64, device=DEV)
    for bad in (dict(row_group=ids), dict(row_group=wide.to(torch.int32).repeat_interleave(2)[::2]), dict(row_group=group.float()),
                dict(row_group=group.cpu()), dict(row_ids=group), dict(row_ids=wide), dict(row_ids=ids.cpu()), dict(row_docs=group),
                dict(row_docs=wide), dict(row_docs=ids.double()), dict(row_docs=ids.cpu()), dict(vecs=frag.cpu()),
                dict(lists=(ids, two, 1, ids, ids.cpu())), dict(lists=(ids.cpu(), two, 1, ids, ids)), dict(lists=(ids, two, 1, ids, group))):
        with pytest.raises((ValueError, TypeError)):
            ops.selected_search(**{**dict(x=x, vecs=frag, rows=8, row_group=group, row_ids=ids, row_docs=ids, k=4), **bad})


def test_one_call_refuses_what_its_launches_do():
    frag, x = torch.zeros(128, 256, dtype=torch.bfloat16, device=DEV), torch.zeros(2, 256, device=DEV)
    group, ids = torch.zeros(8, dtype=torch.int32, device=DEV), torch.zeros(8, dtype=torch.int64, device=DEV)
    i64 = torch.zeros(1, dtype=torch.int64)
    for bad in (dict(x=x[:, :128]), dict(x=x.to(torch.bfloat16)), dict(rows=9), dict(k=0), dict(k=9), dict(groups=group.cpu()[:1]),
                dict(groups=torch.zeros(2, dtype=torch.int64)), dict(limits=i64), dict(limits=i64.to(DEV)), dict(rows=129),
                dict(lists=(i64.to(DEV), i64.to(DEV), 1, i64.to(DEV), i64.to(DEV))), dict(lists=(i64, ids[:3], 1, ids, ids))):
        with pytest.raises(ValueError):
            ops.selected_search(**{**dict(x=x, vecs=frag, rows=8, row_group=group, row_ids=ids, row_docs=ids, k=4), **bad})
