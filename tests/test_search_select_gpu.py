"""Scores with their parts' maxima (index_scan.hip) and the selection from them (search.hip) against plain torch."""
import numpy as np
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.engine.vector_index import VectorIndex

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _key(x):
    """Floats in the kernels' order (-0 below 0), as integers."""
    bits = x.contiguous().view(torch.int32).long()
    return torch.where(bits < 0, -(bits & 0x7FFFFFFF) - 1, bits)


def _parts(s):
    n = s.shape[1]
    pad = torch.full((s.shape[0], -n % 16), float("-inf"), device=s.device)
    u = _key(torch.cat([s, pad], 1).view(s.shape[0], -1, 16).max(-1)[0]) + (1 << 31)  # unsigned ordered bits
    p = torch.randint(0, 1 << 30, (s.shape[0], -(-n // 64) * 4), device=s.device, dtype=torch.int32)  # (padding: anything)
    p[:, : u.shape[1]] = torch.where(u >= 1 << 31, u - (1 << 32), u).to(torch.int32)
    return p


# rows around a wave's 16, a tile's 32, the ring's refill (256 workgroups x 32 rows) and several rounds of it; queries
# around the 16 of a fragment and the groups' sizes
@pytest.mark.parametrize("dim,queries", [(256, 1), (256, 65), (256, 256), (512, 17), (768, 1), (768, 64), (768, 129), (1024, 5),
                                         (1024, 128)])
@pytest.mark.parametrize("n", [4, 28, 36, 8192, 8228, 70_020])
def test_scores_and_parts(n, dim, queries):
    g = torch.Generator(device=DEV).manual_seed(n + dim)
    q, v = (torch.nn.functional.normalize(torch.randn(m, dim, device=DEV, generator=g), dim=-1).to(torch.bfloat16)
            for m in (queries, -(-n // 128) * 128))
    group = (torch.arange(len(v), device=DEV) % 5 - 1).to(torch.int32)
    qg = (torch.arange(queries, device=DEV) % 6 - 1).clamp(max=3).to(torch.int32)
    words = (n + 31) // 32
    allow = torch.randint(-2 ** 31, 2 ** 31, (queries, words), device=DEV, generator=g).to(torch.int32)
    seen = (allow[:, torch.arange(n, device=DEV) // 32] >> (torch.arange(n, device=DEV) % 32)) & 1 == 1
    exact = q.double() @ v[:n].double().t()
    frag = ops.shuffle_weights(v)
    for gq, mask in ((None, None), (qg, None), (None, allow), (qg, allow)):
        s, p = ops.scores_and_parts(q, frag, n, group[:n].contiguous(), gq, mask)
        live = (group[:n] >= 0).expand(queries, -1)
        if gq is not None:
            live = live & ((gq[:, None] < 0) | (group[None, :n] == gq[:, None]))
        if mask is not None:
            live = live & seen
        assert torch.equal(torch.isinf(s), ~live)
        # a sum of dim exact products in fp32, up to 2^-23 of the running sum (unit vectors: below 1) lost a step
        assert ((s.double() - exact).abs().masked_fill(~live, 0) <= dim * 2.0 ** -23).all()
        u = (n + 15) // 16
        assert torch.equal(p[:, :u], _parts(s)[:, :u])


@pytest.mark.parametrize("n", [4, 60, 1024, 8192, 8196, 20_004, 70_000, 1_100_000])
@pytest.mark.parametrize("k", [1, 16, 250, 1024])
def test_top_hits(n, k):
    """Scores of any spread, equal ones (in row order where they are few enough to be ranked), rows that few or no scores
    pass, infinities."""
    k = min(k, n)
    g = torch.Generator(device=DEV).manual_seed(n + k)
    s = torch.randn(8, n, device=DEV, generator=g)
    s[1] = torch.round(s[1] * 3)  # thousands of equal scores
    s[2] = float("-inf")
    s[3, torch.rand(n, device=DEV, generator=g) < 0.98] = float("-inf")
    s[4, 40:] = float("-inf")
    s[5] = torch.where(s[5] > 0, s[5] * 1e-30, s[5] * 1e30)
    s[6, : n // 2: 2] = 0.0
    s[6, 1: n // 2: 2] = -0.0
    s[7, n // 3] = float("inf")
    ids, docs = torch.randperm(n + 3, device=DEV, generator=g), torch.arange(n + 3, device=DEV) // 3
    row_of = torch.empty_like(ids)
    row_of[ids] = torch.arange(n + 3, device=DEV)
    vals, got, gdocs = ops.top_hits(s, _parts(s), k, ids, docs)
    for m in range(len(s)):
        key = _key(s[m])
        at = torch.argsort(-key, stable=True)[:k]
        assert torch.equal(_key(vals[m]), key[at])
        hit = torch.isfinite(vals[m])
        assert torch.equal(got[m] >= 0, hit) and torch.equal(gdocs[m] >= 0, hit)
        rows = row_of[got[m][hit]]
        assert torch.equal(_key(s[m])[rows], _key(vals[m])[hit]) and rows.unique().numel() == rows.numel()
        assert torch.equal(gdocs[m][hit], docs[rows])
        if m not in (1, 6):
            assert torch.equal(rows, at[hit])


@pytest.mark.parametrize("n", [5, 8190, 20_003])
@pytest.mark.parametrize("flt", ["none", "group", "allowed", "doc_lt", "all"])
def test_search_by_selection_is_the_full_search(n, flt):
    """The route of searches that select against the scores of ``gemm_bt`` and ``topk_rows``: removed rows, k above the
    rows that are left, one query without a hit."""
    rng = np.random.default_rng(n)
    ids, docs = rng.permutation(n) + 7, np.arange(n) // 6
    idx = VectorIndex(768, DEV, capacity=n)
    g = torch.Generator(device=DEV).manual_seed(n)
    idx.add(ids, torch.randn(n, 768, device=DEV, generator=g), doc_ids=docs, groups=docs % 3)
    idx.remove(ids[: n // 4])
    q = torch.randn(6, 768, device=DEV, generator=g)
    kw = {}
    if flt in ("group", "all"):
        kw["q_groups"] = [0, 1, -1, 2, 1, 9]
    if flt in ("allowed", "all"):
        kw["allowed"] = [rng.choice(ids, max(1, n // (2 + i)), replace=False) for i in range(5)] + [np.empty(0, np.int64)]
    if flt in ("doc_lt", "all"):
        kw["doc_lt"] = [0, 1, n // 8, n // 6, 10 ** 9, 3]
    for k in (1, 250, 3000):
        idx.threshold_search = False
        ev, ei, ed = idx.search(q, k, **kw)
        idx.threshold_search = True
        assert idx._selects(6, not ("allowed" in kw or "doc_lt" in kw))
        gv, gi, gd = idx.search(q, k, **kw)
        assert idx.stats["threshold_searches"] == 0 and idx.stats["selected_searches"] > 0
        assert gv.shape == ev.shape and torch.equal(torch.isinf(gv), torch.isinf(ev))
        hit = ~torch.isinf(gv)
        assert ((gv - ev)[hit].abs() <= 768 * 2.0 ** -22).all()  # two fp32 sums of 768 products of unit vectors
        assert torch.equal(gi >= 0, hit) and torch.equal(gd >= 0, hit)
        same = gi == ei  # (neighbours that close may change places)
        assert torch.equal(gd[same], ed[same]) and same.float().mean() > 0.97


# n, k, rows that pass: together, one of so many, or values of so few kinds.  Fewer threads (64 rows each) than k see a score;
# fewer parts (16 rows) than k do; more than 4096 parts or 8192 scores reach the threads' bound; equal scores fill them.
FEW_THREADS = [(8_196, 250, "all", 1), (12_000, 250, "all", 1), (30_000, 500, "all", 1), (50_000, 1000, "all", 1),
               (16_384, 1024, "all", 1), (100_000, 1024, "all", 1), (1_000_000, 1024, "all", 1), (1_300_000, 1000, "all", 1),
               (100_000, 1000, "every", 4), (600_000, 250, "together", 12_000), (1_000_000, 1000, "together", 50_000),
               (1_100_000, 500, "together", 20_000), (60_000, 1000, "kinds", 1), (60_000, 250, "kinds", 3),
               (1_100_000, 700, "kinds", 1), (400_000, 1024, "kinds", 400)]


def _few_threads(n, k, kind, arg):
    g = torch.Generator(device=DEV).manual_seed(n + k)
    s = torch.randn(3, n, device=DEV, generator=g) * 0.05
    if kind == "every":
        s[:, torch.arange(n, device=DEV) % arg != 1] = float("-inf")
    elif kind == "together":
        s[:, : n // 3] = float("-inf")
        s[:, n // 3 + arg:] = float("-inf")
    elif kind == "kinds":
        s = torch.randint(0, arg, (3, n), device=DEV, generator=g).float() - arg // 2
    return s


@pytest.mark.parametrize("n,k,kind,arg", FEW_THREADS)
def test_top_hits_where_few_threads_see_a_score(n, k, kind, arg):
    s = _few_threads(n, k, kind, arg)
    ids, docs = torch.arange(n, device=DEV) + 5, torch.arange(n, device=DEV) // 3
    vals, got, gdocs = ops.top_hits(s, _parts(s), k, ids, docs)
    at = torch.argsort(-_key(s), dim=1, stable=True)[:, :k]  # (equal scores in row order)
    assert torch.equal(vals, s.gather(1, at))
    assert torch.equal(got, torch.where(torch.isinf(vals), -1, at + 5)) and torch.equal(gdocs, torch.where(torch.isinf(vals), -1, at // 3))


@pytest.mark.parametrize("n,k,kind,arg", FEW_THREADS)
def test_top_hits_costs_no_more_than_the_general_selection(n, k, kind, arg):
    """One workgroup that goes over a whole row again and again took up to ten times as long as the selection in chunks."""
    s = _few_threads(n, k, kind, arg)
    p, ids = _parts(s), torch.arange(n, device=DEV)

    def us(f):
        for _ in range(3):
            f()
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        torch.cuda.synchronize()
        a.record()
        for _ in range(20):
            f()
        b.record()
        b.synchronize()
        return 50 * a.elapsed_time(b)

    def general():
        vals, rows = ops.topk_rows(s, k)
        ops.hit_ids(vals, rows, ids, ids)
    new, old = (min(t) for t in zip(*((us(lambda: ops.top_hits(s, p, k, ids, ids)), us(general)) for _ in range(5))))  # in turn
    print(f"{n} {k} {kind} {arg}: {new:.1f} us, general {old:.1f}")
    assert new <= 1.15 * old


@pytest.mark.parametrize("n", [(1 << 22) - 4, 1 << 22])
def test_scores_of_more_than_one_buffer(n):
    """256 queries by 4.2M rows: the scan's stores reach 4 GB, beyond that the scores are ``gemm_bt``'s."""
    dim, queries = 256, 256
    g = torch.Generator(device=DEV).manual_seed(n)
    q = torch.nn.functional.normalize(torch.randn(queries, dim, device=DEV, generator=g), dim=-1).to(torch.bfloat16)
    v = torch.nn.functional.normalize(torch.randn(1 << 14, dim, device=DEV, generator=g), dim=-1).to(torch.bfloat16)
    frag = ops.shuffle_weights(v).repeat((1 << 22) // len(v), 1)  # (a row's 16 neighbours are whole blocks of the copy)
    group = torch.zeros(1 << 22, dtype=torch.int32, device=DEV)
    group[7::1000] = -1
    s = ops.scores_shuffled(q, frag, n, group)
    rows = torch.cat([torch.arange(0, n, 9973, device=DEV), torch.arange(n - 40, n, device=DEV)])
    exp = q.double() @ v[rows % len(v)].double().t()
    live = (group[rows] >= 0).expand(queries, -1)
    assert s.shape == (queries, n) and torch.equal(torch.isinf(s[:, rows]), ~live)
    assert ((s[:, rows].double() - exp).abs().masked_fill(~live, 0) <= dim * 2.0 ** -23).all()  # an fp32 sum of exact products


def test_a_callers_pinned_filters_may_be_refilled():
    """Groups and document limits in pinned buffers that the caller fills anew once ``search`` returns, while the device
    is still busy with what was queued before."""
    n = 20_000
    idx = VectorIndex(256, DEV, capacity=n)
    g = torch.Generator(device=DEV).manual_seed(0)
    idx.add(np.arange(n), torch.randn(n, 256, device=DEV, generator=g), doc_ids=np.arange(n) // 4, groups=np.arange(n) % 2)
    q = torch.randn(3, 256, device=DEV, generator=g)
    groups, limits = torch.tensor([0, 1, 0], dtype=torch.int32), torch.tensor([90, 4000, 2500])
    exp = idx.search(q, 20, q_groups=groups, doc_lt=limits)
    groups, limits = groups.pin_memory(), limits.pin_memory()
    torch.cuda._sleep(200_000_000)  # some 0.1 s
    got = idx.search(q, 20, q_groups=groups, doc_lt=limits)
    groups.fill_(1)
    limits.fill_(3)
    for a, b in zip(got, exp):
        assert torch.equal(a, b)


def test_a_capture_does_not_record_a_copy_of_filters(monkeypatch):
    """While a stream is captured the filters take the copy that is waited for (which the capture refuses): a recorded copy
    from a pinned buffer of the search's own would read whatever that memory holds at the replay."""
    idx = VectorIndex(256, DEV, capacity=64)
    pinned = []
    pin = torch.Tensor.pin_memory
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t, *a: pinned.append(t) or pin(t, *a))
    group = torch.tensor([1, 2], dtype=torch.int32)
    assert torch.equal(idx._there(group).cpu(), group) and len(pinned) == 1
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert torch.equal(idx._there(group).cpu(), group) and len(pinned) == 1
