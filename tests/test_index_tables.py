"""The device tables a ``VectorIndex`` derives from its rows and keeps until the next update."""
import numpy as np
import torch

from django_assistant_bot_amd.engine.vector_index import VectorIndex


def _rows_by_table(idx, ids):
    keys, rows = (t.cpu().numpy() for t in idx._live_ids())
    assert (np.diff(keys) > 0).all()
    if not len(keys):
        return rows
    at = np.searchsorted(keys, ids)
    ok = (at < len(keys)) & (keys[np.minimum(at, len(keys) - 1)] == ids)
    return rows[at[ok]]


def test_id_table_names_the_rows_of_the_mapping():
    """Ids that one ``add`` names twice (the later vector is the item's), updates, removals, a compaction."""
    rng = np.random.default_rng(0)
    idx = VectorIndex(128, "cpu", capacity=64, dtype=torch.float32)
    asked = np.arange(-5, 4000)
    for step in range(4):
        ids = rng.integers(0, 3000, 2000)
        if step == 2:
            idx.remove(rng.integers(0, 3000, 2500))
        idx.add(ids, torch.from_numpy(rng.standard_normal((len(ids), 128)).astype(np.float32)))
        if step == 3:
            idx.compact()
        assert np.array_equal(_rows_by_table(idx, asked), idx.rows_of(asked))
    while len(idx):
        idx.remove(np.arange(3000))
        assert np.array_equal(_rows_by_table(idx, asked), idx.rows_of(asked))
