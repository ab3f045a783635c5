"""Threshold search where the best rows are in the sample itself: the scan's score of the row that set the threshold may
differ from the sample's by the order of its sum."""
import numpy as np
import pytest
import torch

from django_assistant_bot_amd.engine.vector_index import VectorIndex

pytestmark = pytest.mark.gpu


# widths with a scan kernel of their own and without, a width without the fragment layout; the queries' chunks of the
# candidate lists go to another kernel than all of them together
@pytest.mark.parametrize("dim", [128, 192, 256, 384, 640, 768, 1280])
@pytest.mark.parametrize("queries,cand_bytes", [(1, None), (16, None), (100, None), (300, 44)])
def test_rows_of_the_sample_are_found(dim, queries, cand_bytes, monkeypatch):
    n, nq = 30_000, 400 if queries > 1 else 60
    g = torch.Generator(device="cuda").manual_seed(dim)
    q = torch.randn(nq, dim, device="cuda", generator=g)
    v = torch.randn(n, dim, device="cuda", generator=g)
    v[: 64 * nq: 64] = q + torch.randn(nq, dim, device="cuda", generator=g)  # query i's best row: 64 i
    idx = VectorIndex(dim, "cuda", capacity=n)
    idx.add(np.arange(n), v)
    for k in (1, 3):
        got = []
        for on in (False, True):
            idx.threshold_search, idx.threshold_min_rows, idx.select_rows = on, 1, 0
            if on and cand_bytes:
                cap = 4 * idx._sample_rank(k) * 64 + 4096
                monkeypatch.setattr(idx, "CAND_BYTES", 8 * cap * cand_bytes, raising=False)
            parts = [idx.search(q[i:i + queries], k) for i in range(0, nq, queries)]
            got.append([torch.cat(t) for t in zip(*parts)])
        (ev, ei, _), (gv, gi, _) = got
        assert idx.stats["threshold_searches"] > 0 and not idx.stats.get("selected_searches")
        assert torch.equal(ei[:, 0], 64 * torch.arange(nq, device="cuda")) and torch.equal(gi[:, 0], ei[:, 0])
        # two fp32 sums of dim products of unit vectors; ranks may change places only where scores are that close
        assert ((gv - ev).abs() <= dim * 2.0 ** -22).all() and (gi >= 0).all()
        monkeypatch.undo()
