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


def test_a_row_is_written_once(monkeypatch):
    _check("cpu", 32, monkeypatch)


@pytest.mark.gpu
def test_a_row_is_written_once_on_the_gpu(monkeypatch):
    _check("cuda", 256, monkeypatch)
