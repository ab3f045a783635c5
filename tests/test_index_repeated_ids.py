"""Ids that one ``VectorIndex.add`` names twice: a row is written once, with what came last."""
import numpy as np
import pytest
import torch

from django_assistant_bot_amd.engine.vector_index import VectorIndex


def _check(device, dim, monkeypatch):
    written = []
    put = VectorIndex._put
    monkeypatch.setattr(VectorIndex, "_put", lambda self, rows, v: written.append(rows.tolist()) or put(self, rows, v))
    idx = VectorIndex(dim, device, capacity=64)
    idx.add(np.arange(40), torch.zeros(40, dim) + torch.eye(dim)[:1], doc_ids=np.arange(40), groups=np.zeros(40))
    v = torch.eye(dim)[2:10]
    #  (40, new and named twice, has two rows; 7 and 3 are in the index)
    idx.add([7, 3, 40, 7, 3, 40, 7, 5], v, doc_ids=[70, 30, 0, 71, 31, 1, 72, 50], groups=[0, 1, 0, 1, 0, 1, 2, 0])
    assert len(written[-1]) == len(set(written[-1])) == 5 and idx.n == 42
    for item, at, doc, group in ((7, 6, 72, 2), (3, 4, 31, 0), (5, 7, 50, 0), (40, 5, 1, 1)):
        row = int(idx.rows_of([item])[0])
        assert torch.equal(idx.rows_data([row])[0].float().cpu(), v[at])
        assert (int(idx.row_ids[row]), int(idx.row_docs[row]), int(idx.row_group[row])) == (item, doc, group)
    ids = idx.search(v[6], 1)[1]
    assert ids.tolist() == [[7]]


# ids of the index and new ones, with and without an id that is named twice
@pytest.mark.parametrize("ids", [[1, 3, 1], [3, 4, 3], [1, 3, 4], [3, 4, 5]])
@pytest.mark.parametrize("name", ["doc_ids", "groups"])
def test_one_value_for_all_rows(ids, name):
    for one in (5, [5], np.array([[5]])):
        idx = VectorIndex(32, "cpu", capacity=4)
        idx.add([1, 2], torch.eye(32)[:2])
        idx.add(ids, torch.eye(32)[2:5], **{name: one})
        kept = idx.row_docs if name == "doc_ids" else idx.row_group
        for i, item in enumerate(ids):
            row = int(idx.rows_of([item])[0])
            assert int(kept[row]) == 5
            if item not in ids[i + 1:]:
                assert torch.equal(idx.rows_data([row])[0].float(), torch.eye(32)[2 + i])
        assert len(idx) == 2 + len(set(ids) - {1, 2})


@pytest.mark.parametrize("ids", [[1, 3, 1], [3, 4, 3], [1, 3, 4], [3, 4, 5]])
@pytest.mark.parametrize("name", ["doc_ids", "groups"])
@pytest.mark.parametrize("bad", [[1, 2], [1, 2, 3, 4], [[1], [2], [3]]])
def test_what_is_refused_changes_nothing(ids, name, bad):
    idx = VectorIndex(32, "cpu", capacity=4)
    idx.add([1, 2], torch.eye(32)[:2], doc_ids=7)
    with pytest.raises((ValueError, RuntimeError)):
        idx.add(ids, torch.eye(32)[2:5], **{name: bad})
    assert len(idx) == idx.n == 2 and idx.search(torch.eye(32)[1], 2)[1].tolist() == [[2, 1]]
    assert idx.row_docs[:2].tolist() == [7, 7] and torch.equal(idx.rows_data([0, 1]).float(), torch.eye(32)[:2])


def test_a_row_is_written_once(monkeypatch):
    _check("cpu", 32, monkeypatch)


@pytest.mark.gpu
def test_a_row_is_written_once_on_the_gpu(monkeypatch):
    _check("cuda", 256, monkeypatch)
