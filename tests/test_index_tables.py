"""The device tables a ``VectorIndex`` derives from its rows and keeps until the next update."""
import numpy as np
import pytest
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


@pytest.mark.parametrize("twice", [False, True])
def test_id_table_names_the_rows_of_the_mapping(twice, tmp_path):
    """Ids that one ``add`` names twice (the later vector is the item's) or once, updates, removals, a compaction, a
    snapshot."""
    rng = np.random.default_rng(0)
    idx = VectorIndex(128, "cpu", capacity=64, dtype=torch.float32)
    asked = np.arange(-5, 4000)
    for step in range(4):
        ids = rng.integers(0, 3000, 2000)
        ids = ids if twice else np.unique(ids)
        if step == 2:
            idx.remove(rng.integers(0, 3000, 2500))
        idx.add(ids, torch.from_numpy(rng.standard_normal((len(ids), 128)).astype(np.float32)))
        if step == 3:
            idx.compact()
        assert np.array_equal(_rows_by_table(idx, asked), idx.rows_of(asked)) and idx._twice == twice
    idx.save(str(tmp_path / "rows"))
    idx = VectorIndex.load(str(tmp_path / "rows"), "cpu")
    assert np.array_equal(_rows_by_table(idx, asked), idx.rows_of(asked))
    while len(idx):
        idx.remove(np.arange(3000))
        assert np.array_equal(_rows_by_table(idx, asked), idx.rows_of(asked))


class _Interrupted(VectorIndex):
    """Runs ``update`` once, after the id -> row mapping was read (as an update on another thread can)."""

    update = None

    def _then(self, got):
        update, self.update = self.update, None
        if update is not None:
            update(self)
        return got

    def _id_rows(self):
        return self._then(super()._id_rows())

    def _live_rows(self):
        return self._then(super()._live_rows())


UPDATES = {
    "add": lambda idx: idx.add([7, 900], torch.randn(2, 128)),
    "remove": lambda idx: idx.remove([0, 1, 2]),
    "compact": lambda idx: (idx.remove([3, 4]), idx.compact()),
}


@pytest.mark.parametrize("name", UPDATES)
@pytest.mark.parametrize("first,twice", [("rows_of", False), ("_live_ids", False), ("_live_ids", True)])
def test_tables_of_an_older_version_are_rebuilt(name, first, twice):
    idx = _Interrupted(128, "cpu", capacity=64, dtype=torch.float32)
    idx._twice = twice
    idx.add(np.arange(100), torch.randn(100, 128))
    asked = np.arange(1000)
    idx.update = UPDATES[name]
    idx.rows_of(asked) if first == "rows_of" else idx._live_ids()
    assert idx.update is None
    now = np.array(sorted(idx._row_of.items()))
    assert np.array_equal(idx.rows_of(asked), now[:, 1]) and np.array_equal(_rows_by_table(idx, asked), now[:, 1])


class _Replaced(VectorIndex):
    """Reads its tables just before a compaction replaces the id -> row mapping."""

    @property
    def _row_of(self):
        return self._mapping

    @_row_of.setter
    def _row_of(self, mapping):
        if hasattr(self, "_mapping"):
            self.rows_of([5])
            self._live_ids()
        self._mapping = mapping


def test_compaction_shows_its_version_last():
    idx = _Replaced(128, "cpu", capacity=64, dtype=torch.float32)
    idx._twice = True
    idx.add(np.arange(100), torch.randn(100, 128))
    idx.remove(np.arange(0, 100, 3))
    idx.compact()
    now = np.array(sorted(idx._row_of.items()))
    assert np.array_equal(idx.rows_of(np.arange(100)), now[:, 1])
    assert np.array_equal(_rows_by_table(idx, np.arange(100)), now[:, 1])


@pytest.mark.gpu
def test_tables_built_on_one_stream_are_read_on_another():
    """The id table and the row sample queued behind a long kernel on one stream and used at once on a second, which also
    outlives the entry: masks and scores as on one stream."""
    n, dim, k = 70_000, 128, 20
    g = torch.Generator(device="cuda").manual_seed(0)
    idx = VectorIndex(dim, "cuda", capacity=n + 10)
    idx.add(np.random.default_rng(0).permutation(n), torch.randn(n, dim, device="cuda", generator=g))
    idx.threshold_min_rows = 1
    q = torch.randn(4, dim, device="cuda", generator=g)
    allowed = [np.arange(i, n, 7) for i in range(4)]
    mask, (sample, groups) = idx.allow_mask(allowed), idx._sample_rows(n // 64 // 4 * 4)
    vals, ids, _ = idx.search(q, k)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for idx._twice in (False, True, False):  # (from the row metadata, from the mapping)
        idx._version += 1  # (rows as they were: both tables are built anew)
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(200_000_000)  # some 0.1 s
            for t in (*idx._live_ids(), *idx._sample_rows(n // 64 // 4 * 4)):
                assert t.is_cuda
        del t
        with torch.cuda.stream(b):
            got = idx.allow_mask(allowed)
            s2, g2 = (t.clone() for t in idx._sample_rows(n // 64 // 4 * 4))
            idx._id_table = idx._sample = None  # the tables are freed with b's reads in flight
            junk = [torch.full((n,), -1, device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        assert torch.equal(got, mask) and torch.equal(s2, sample) and torch.equal(g2, groups)
        with torch.cuda.stream(b):
            got = idx.search(q, k)
        torch.cuda.synchronize()
        assert torch.equal(got[0], vals) and torch.equal(got[1], ids)
        del junk
    idx.remove(np.arange(n))
    assert not idx.allow_mask(allowed).any()  # a table without ids
