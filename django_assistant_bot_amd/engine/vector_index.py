"""Exact in-HBM cosine top-k index: the pgvector replacement.

The reference stores 768-d vectors in PostgreSQL (``VectorField`` + HNSW m=16/ef_construction=64,
storage/models.py:32-58) and searches with ``qs.annotate(distance=CosineDistance(field, q))
.order_by('distance')[:n]`` (rag/services/search_service.py:185-196) -- approximate, on the CPU, one
query at a time.  Here rows live L2-normalised in bf16 in HBM (1M x 768 = 1.5 GB, noise next to
288 GB), every query of a batch is scored against every live row by the MFMA GEMM kernel with the
filter applied in its epilogue (row tombstones, per-query group = bot, optional allow-bitmask for
arbitrary QuerySet filters), and the exact top-k is selected by the radix-select kernel.
Recall is 1.0 by construction.  Distance semantics match pgvector: ``1 - cos``.

The index is a cache of the ORM (source of truth); it supports upsert, delete (tombstone + lazy
compaction), growth, and safetensors snapshots for warm starts.

On the GPU (bf16, dim % 128 == 0) the rows are held ONCE, in the ``ops.shuffle_weights`` fragment
layout: every 16-row x 32-k block is one coalesced 1 KB load for the scans of up to
256 queries (index_scan.hip / the streaming GEMM's candidate epilogue) and one LDS-DMA piece for the
phased GEMM above that and the generic-filter score GEMM.  (Round 2 kept a row-major copy beside
it: 2x the index HBM.)  Only the 1/64 row sample of the threshold search is gathered, and cached until
the next update.
"""
from __future__ import annotations

from itertools import accumulate

import numpy as np
import torch
import torch.nn.functional as F

from .. import ops


class VectorIndex:
    def __init__(self, dim: int, device=None, capacity: int = 4096, dtype=torch.bfloat16):
        self.dim = dim
        self.device = torch.device(device if device is not None else ("cuda" if torch.cuda.is_available() else "cpu"))
        self.dtype = dtype
        self._cap = 0
        self.n = 0  # rows in use (live + tombstoned)
        self.stats = {"threshold_searches": 0, "threshold_overflows": 0}
        self.vecs = self.row_ids = self.row_docs = self.row_group = None
        self._row_of: dict[int, int] = {}
        self._sorted = None  # lazily built (version, sorted ids, rows) for vectorised id -> row lookups
        # fragment layout (see the module docstring) for bf16 GPU indexes of a 128-multiple width
        self.frag = self.device.type == "cuda" and dtype == torch.bfloat16 and dim % 128 == 0
        self._version = 0  # bumped at the end of every update: invalidates the cached threshold sample and id tables
        self._sample = None
        self._id_table = None
        self._dead = 0
        self._twice = False  # an id may have live rows beside the mapping's one (see ``add``)
        self._grow(max(64, capacity))

    # ------------------------------------------------------------------ storage
    def _grow(self, cap: int):
        cap = (cap + 255) // 256 * 256  # whole 256-row tiles for the fragment-layout scans / GEMMs
        dev = self.device
        vecs = torch.zeros((cap, self.dim), dtype=self.dtype, device=dev)
        ids = torch.full((cap,), -1, dtype=torch.int64, device=dev)
        docs = torch.full((cap,), -1, dtype=torch.int64, device=dev)
        grp = torch.full((cap,), -1, dtype=torch.int32, device=dev)
        if self.n:
            if self.frag:  # the first ceil(n / 16) 16-row blocks are a contiguous prefix
                e = -(-self.n // 16) * 16 * self.dim
                vecs.view(-1)[:e] = self.vecs.view(-1)[:e]
            else:
                vecs[: self.n] = self.vecs[: self.n]
            ids[: self.n] = self.row_ids[: self.n]
            docs[: self.n] = self.row_docs[: self.n]
            grp[: self.n] = self.row_group[: self.n]
        self.vecs, self.row_ids, self.row_docs, self.row_group = vecs, ids, docs, grp
        self._cap = cap

    # exact threshold search (no score matrix) for large indexes on the GPU: see _threshold_search
    threshold_search = True
    threshold_min_rows = 1 << 19
    # 1/64 of the rows (4 x fewer sample bytes and sample scores than 1/16 for ~4 x more candidates:
    # 10M rows x 512 queries 10.79 -> 9.15 ms, 128 queries 4.70 -> 4.59; profiles/index_search.md)
    sample_stride = 64

    def _put(self, rows: torch.Tensor, v: torch.Tensor) -> None:
        if self.frag:
            ops.shuffle_rows_into(self.vecs, rows, v)
        else:
            self.vecs[rows] = v

    def rows_data(self, rows) -> torch.Tensor:
        """Row-major copy of the given rows (any layout)."""
        rows = torch.as_tensor(rows, dtype=torch.int64, device=self.device)
        if not self.frag:
            return self.vecs[rows]
        R, K = self.vecs.shape
        v5 = self.vecs.view(R // 16, K // 32, 4, 16, 8)
        return v5[rows // 16, :, :, rows % 16, :].reshape(rows.numel(), K)

    def __len__(self) -> int:
        return len(self._row_of)

    def __contains__(self, item_id: int) -> bool:
        return int(item_id) in self._row_of

    def add(self, ids, vectors, doc_ids=None, groups=None) -> None:
        """Upsert rows.  ids: int64 [n]; vectors [n, dim] (any float dtype / device); doc_ids int64 [n]
        (document each row belongs to); groups int32 [n] (e.g. bot id; must be >= 0), or one value for all rows.  What is
        refused leaves the index as it was."""
        ids = np.asarray(ids, dtype=np.int64).reshape(-1)
        n = len(ids)
        if n == 0:
            return
        v = torch.as_tensor(vectors).to(self.device, torch.float32).reshape(n, self.dim)
        v = F.normalize(v, dim=-1).to(self.dtype)

        def per_row(a):
            if a.ndim > 1 and a.size == a.shape[-1]:
                a = a.reshape(-1)
            return a if a.shape == (n,) else np.broadcast_to(a, (n,)).copy()
        docs = per_row(np.asarray(-1 if doc_ids is None else doc_ids, dtype=np.int64))
        grp = per_row(np.asarray(0 if groups is None else groups, dtype=np.int32))
        if (grp < 0).any():
            raise ValueError("groups must be >= 0 (negative marks deleted rows)")
        idl = ids.tolist()
        distinct = set(idl)
        if len(distinct) == n and not (self._row_of.keys() & distinct):
            # bulk insert of new ids (ingest): C-speed bookkeeping, contiguous rows
            if self.n + n > self._cap:
                self._grow(max(self.n + n, 2 * self._cap))
            rows = np.arange(self.n, self.n + n, dtype=np.int64)
            self._row_of.update(zip(idl, range(self.n, self.n + n)))
            self.n += n
        else:
            rows = np.empty(n, dtype=np.int64)
            fresh = []
            for i, x in enumerate(idl):
                r = self._row_of.get(x)
                if r is None:
                    fresh.append(i)
                else:
                    rows[i] = r
            if fresh:
                # (a new id that one call names twice gets two rows; the mapping keeps the later one)
                self._twice |= len({idl[i] for i in fresh}) < len(fresh)
                need = self.n + len(fresh)
                if need > self._cap:
                    self._grow(max(need, 2 * self._cap))
                for j, i in enumerate(fresh):
                    rows[i] = self.n + j
                    self._row_of[idl[i]] = self.n + j
                self.n += len(fresh)
            last = dict(zip(rows.tolist(), range(n))) if len(distinct) < n else rows
            if len(last) < n:  # an id of the index named twice: its later vector (writes to one row in one launch have no order)
                at = np.sort(np.fromiter(last.values(), dtype=np.int64, count=len(last)))
                rows, ids, docs, grp, v = rows[at], ids[at], docs[at], grp[at], v[torch.from_numpy(at).to(self.device)]
        pin = self.device.type == "cuda"

        def dev(a):
            x = torch.from_numpy(np.ascontiguousarray(a))
            return (x.pin_memory() if pin else x).to(self.device, non_blocking=True)
        r = dev(rows)
        self._put(r, v)
        self.row_ids[r] = dev(ids)
        self.row_docs[r] = dev(docs)
        self.row_group[r] = dev(grp)
        self._version += 1  # behind the writes: what another thread caches meanwhile is of the old version

    def remove(self, ids) -> int:
        rows = [self._row_of.pop(int(x)) for x in np.asarray(ids).reshape(-1).tolist() if int(x) in self._row_of]
        if rows:
            r = torch.as_tensor(rows, dtype=torch.int64, device=self.device)
            self.row_group[r] = -1
            self.row_ids[r] = -1
            self._version += 1
            self._dead += len(rows)
            if self._dead > 1024 and self._dead > self.n // 4:
                self.compact()
        return len(rows)

    def compact(self) -> None:
        live = (self.row_group[: self.n] >= 0).nonzero().flatten()
        m = live.numel()
        self._put(torch.arange(m, device=self.device), self.rows_data(live))
        self.row_ids[:m] = self.row_ids[live]
        self.row_docs[:m] = self.row_docs[live]
        self.row_group[:m] = self.row_group[live]
        self.row_group[m: self.n] = -1
        self.n = m
        self._dead = 0
        ids = self.row_ids[:m].cpu().numpy()
        self._row_of = {int(x): i for i, x in enumerate(ids.tolist())}
        self._version += 1

    # ------------------------------------------------------------------ search
    def _id_rows(self) -> np.ndarray:
        """int64 [2, items]: the item ids and the row of each (of one moment: an update may run on another thread)."""
        row_of = self._row_of.copy()
        return np.stack([np.fromiter(d, dtype=np.int64, count=len(row_of)) for d in (row_of.keys(), row_of.values())])

    def rows_of(self, ids) -> np.ndarray:
        """Row index of each live item id (ids that are not in the index are dropped).  Vectorised
        through a sorted (id, row) table rebuilt lazily after upserts / deletes."""
        ids = np.asarray(ids, dtype=np.int64).reshape(-1)
        table, version = self._sorted, self._version
        if table is None or table[0] != version:
            keys, vals = self._id_rows()
            order = np.argsort(keys, kind="stable")
            table = self._sorted = (version, keys[order], vals[order])
        _, keys, vals = table
        if not len(keys) or not len(ids):
            return np.zeros(0, dtype=np.int64)
        pos = np.searchsorted(keys, ids)
        pos = np.minimum(pos, len(keys) - 1)
        hit = keys[pos] == ids
        return vals[pos[hit]]

    def _pack_rows(self, row_mask: torch.Tensor) -> torch.Tensor:
        """bool [q, words*32] row mask (device) -> int32 bitmask [q, words] for the score epilogue."""
        q, nb = row_mask.shape
        w = row_mask.view(q, nb // 32, 32).to(torch.int64) << torch.arange(32, device=row_mask.device)
        packed = w.sum(-1)
        packed = packed - (packed >= (1 << 31)).to(torch.int64) * (1 << 32)
        return packed.to(torch.int32).contiguous()

    @staticmethod
    def _id_lists(allowed) -> list:
        return [np.fromiter(ids, dtype=np.int64) if isinstance(ids, (set, frozenset)) else
                np.asarray(ids, dtype=np.int64).reshape(-1) for ids in allowed]

    def _lists_there(self, lists):
        """(ids, offsets, longest list, keys, rows) as ``ops.allow_bits`` takes them: one copy, the lists behind their offsets;
        the ids are looked up on the device."""
        lens = [len(x) for x in lists]
        host = torch.empty(len(lists) + 1 + sum(lens), dtype=torch.int64, pin_memory=True)
        flat = host.numpy()
        flat[:len(lists) + 1] = list(accumulate(lens, initial=0))
        np.concatenate(lists, out=flat[len(lists) + 1:])
        dev = host.to(self.device, non_blocking=True)
        return dev[len(lists) + 1:], dev[:len(lists) + 1], max(lens), *self._live_ids()

    def allow_mask(self, allowed, mask=None) -> torch.Tensor:
        """Per-query allowed item ids (sets, lists or int arrays) -> int32 bitmask [q, ceil(n/32)] over
        rows, built on the device (no per-id Python loop).  ``mask``: one of zeros to set the bits of."""
        words = (self.n + 31) // 32
        lists = self._id_lists(allowed)
        if self.device.type == "cuda" and 0 < len(lists) <= 65535:
            return ops.allow_bits(*self._lists_there(lists), words, mask)
        m = torch.zeros((len(allowed), words * 32), dtype=torch.bool, device=self.device)
        for qi, ids in enumerate(lists):
            rows = self.rows_of(ids)
            if len(rows):
                m[qi, torch.from_numpy(rows).to(self.device)] = True
        return self._pack_rows(m)

    def _kept(self, slot: str, key, build):
        """Device tensors derived from the rows, built once and kept in ``slot`` until ``key`` changes.  They are built on
        the caller's stream and read on any: a reader on another stream waits for the build and holds the memory until
        its own work is done."""
        entry = getattr(self, slot)
        cuda = self.device.type == "cuda"
        handle = torch._C._cuda_getCurrentRawStream(self.vecs.device.index) if cuda else 0  # (a stream object: 3 us)
        if entry is None or entry[0] != key:
            with torch.inference_mode(False):
                tensors = build()
            event = torch.cuda.current_stream(self.vecs.device).record_event() if cuda else None
            entry = (key, tensors, handle, event)
            setattr(self, slot, entry)
        elif handle != entry[2]:
            stream = torch.cuda.current_stream(self.vecs.device)
            stream.wait_event(entry[3])
            for t in entry[1]:
                t.record_stream(stream)
        return entry[1]

    def _live_rows(self):
        """(item ids, rows) of the live rows, on the device."""
        live = (self.row_group[: self.n] >= 0).nonzero().flatten()
        return self.row_ids[live], live

    def _live_ids(self):
        """(sorted item ids, the row of each) on the device, rebuilt after an update.  From the row metadata (first search
        of 60k rows: 0.36 ms) unless an id may have a second live row: the mapping says which of them is its row (2.25
        ms)."""
        def build():
            if self._twice:
                host = torch.from_numpy(self._id_rows())
                ids, rows = (host.pin_memory() if self.device.type == "cuda" else host).to(self.device, non_blocking=True)
            else:
                ids, rows = self._live_rows()
            keys, order = ids.sort()
            return keys, rows[order]
        return self._kept("_id_table", self._version, build)  # (the version of before the build)

    def doc_lt_mask(self, limits, mask=None) -> torch.Tensor:
        """Rows whose document id is < limits[q] (the ingest dedup filter ``document__id__lt``),
        bitmask built from the row metadata on the device (``mask``: intersected with it, in place)."""
        if mask is not None and mask.shape[0] != len(limits):
            return mask & self.doc_lt_mask(limits)
        words = (self.n + 31) // 32
        lim = torch.as_tensor(np.asarray(limits, dtype=np.int64))
        lim = lim.contiguous() if self._by_value(lim) else self._there(lim)
        if self.device.type == "cuda" and lim.dim() == 1 and self.n and 0 < len(lim) <= 65535:
            return ops.doc_lt_bits(self.row_docs[: self.n], lim, mask)
        lim = lim.to(self.device)[:, None]
        m = torch.zeros((len(limits), words * 32), dtype=torch.bool, device=self.device)
        m[:, : self.n] = self.row_docs[None, : self.n] < lim
        m = self._pack_rows(m)
        return m if mask is None else mask & m

    @torch.inference_mode()
    def scores(self, queries: torch.Tensor, q_groups=None, allowed=None, doc_lt=None) -> torch.Tensor:
        """fp32 cosine similarities [q, n] (-inf for filtered / deleted rows).  Filters: ``q_groups``
        (per-query row group, e.g. bot + status bit), ``allowed`` (per-query item ids), ``doc_lt``
        (per-query document-id bound); masks are ANDed."""
        q, qg, allow, n = self._query(queries, q_groups, allowed, doc_lt)
        if self.frag:
            return ops.gemm_bt(q, self.vecs, epilogue=ops.EPI_SCORES, out_f32=True, row_group=self.row_group[:n],
                               q_group=qg, allow=allow, shuffled=True, n=n)
        return ops.gemm_bt(q, self.vecs[:n], epilogue=ops.EPI_SCORES, out_f32=True, row_group=self.row_group[:n],
                           q_group=qg, allow=allow)

    def _there(self, t: torch.Tensor) -> torch.Tensor:
        """A small host tensor on the index's device, without a wait for the copy from a pinned one of its own (a caller's
        pinned tensor comes back from ``pin_memory`` as it is, and may be refilled once the search returns).  A stream capture
        refuses the copy that is waited for; it would record the other, whose buffer a replay finds in other hands."""
        if self.device.type == "cuda" and not t.is_cuda and not torch.cuda.is_current_stream_capturing():
            own = t.pin_memory()
            if own is not t:
                return own.to(self.device, non_blocking=True)
        return t.to(self.device)

    def _by_value(self, t: torch.Tensor) -> bool:
        """Whether a small tensor can go into the arguments of the launch that reads it: of the host, a row of up to
        ``HOST_VALUES``.  (Not while a stream is captured: ``_there``.  A pinned one may be the target of a copy that the
        stream has yet to make: it is read in the stream's order.)"""
        return (self.device.type == "cuda" and not t.is_cuda and t.dim() == 1 and t.numel() <= ops.native().HOST_VALUES
                and not t.is_pinned() and not torch.cuda.is_current_stream_capturing())

    def _unit(self, queries, q_groups, clear=None):
        """(unit queries, their groups) on the device; ``clear``: a mask to be zeroed."""
        x = torch.as_tensor(queries).to(self.device, torch.float32)
        if q_groups is None and clear is None:
            return ops.unit_rows(x, self.dtype), None
        groups = None if q_groups is None else torch.as_tensor(q_groups, dtype=torch.int32)
        if not (x.is_cuda and self.dtype == torch.bfloat16 and len(x)):
            if clear is not None:
                clear.zero_()
            return ops.unit_rows(x, self.dtype), None if groups is None else self._there(groups)
        q, there = ops.unit_queries(x, groups.contiguous() if groups is not None and self._by_value(groups) else None, clear)
        return q, self._there(groups) if there is None and groups is not None else there

    def _query(self, queries, q_groups, allowed, doc_lt):
        """(unit queries, their groups, row mask, rows in whole fours) on the device."""
        mask, allowed = None, None if allowed is None else list(allowed)
        if allowed and self.device.type == "cuda" and len(allowed) <= 65535:
            mask = torch.empty((len(allowed), (self.n + 31) // 32), dtype=torch.int32, device=self.device)
        q, qg = self._unit(queries, q_groups, mask)
        allow = None if allowed is None else self.allow_mask(allowed, mask)
        if doc_lt is not None:
            allow = self.doc_lt_mask(doc_lt, allow)
        return q, qg, allow, (max(self.n, 4) + 3) // 4 * 4

    @torch.inference_mode()
    def search(self, queries, k: int, q_groups=None, allowed=None, doc_lt=None):
        """-> (similarity [q, k] fp32 desc, item ids [q, k] int64 (-1 = none), doc ids [q, k] int64).
        Group-only filters keep the exact threshold path (no score matrix) on large indexes."""
        queries = torch.as_tensor(queries)
        if queries.ndim == 1:
            queries = queries[None]
        nq = queries.shape[0]
        if self.n == 0 or k <= 0 or nq == 0:
            z = torch.full((nq, max(k, 0)), -1, dtype=torch.int64, device=self.device)
            return torch.full((nq, max(k, 0)), float("-inf"), device=self.device), z, z.clone()
        plain = allowed is None and doc_lt is None
        if self._selects(nq, plain, k):
            return self._selected_search(queries, k, q_groups, allowed, doc_lt)
        if self.device.type == "cuda" and plain and self.n >= self.threshold_min_rows and k <= 1024 and self.threshold_search:
            got = self._threshold_search(queries, k, q_groups)
            if got is not None:
                return got
        s = self.scores(queries, q_groups, allowed, doc_lt)
        vals, rows = ops.topk_rows(s, min(k, s.shape[1], 1024))
        return (vals, *ops.hit_ids(vals, rows, self.row_ids, self.row_docs))

    # From ``threshold_min_rows`` on: rows, and scores in all, up to which a search selects from its scores.  It saves the
    # sample and its two launches, the ranking's and the host read (some 45 us) and writes 4 B a row and query, and one
    # workgroup a query looks through its maxima.  Threshold / selection, us, rows of 768: 1M and 1 query 298 / 258, 4: 299 /
    # 282, 8: 301 / 293, 16: 298 / 303; 600k and 16 213 / 196, 32: 210 / 207; 2M and 1 517 / 514, 4: 517 / 555.  Of 256: 1M
    # and 16 143 / 129; of 1024: 1M and 8 368 / 369.  For more than 512 hits a bound takes longer than a threshold's list:
    # 1000 of 600k and 4 queries 247 / 235, 1M and 1 342 / 337, 4: 339 / 360, 1.4M and 1 432 / 441, 4: 433 / 484.
    select_rows, select_scores = 1_500_000, 8_000_000

    def _selects(self, nq: int, plain: bool, k: int = 1) -> bool:
        """Whether the scan writes the scores and their parts' maxima, and ``top_hits`` selects from them."""
        if not (self.threshold_search and self.frag and ops.scan_scores_ok(nq, (max(self.n, 4) + 3) // 4 * 4, self.dim)):
            return False
        rows, scores = self.select_rows, self.select_scores
        if k > 512:
            rows, scores = 2 * rows // 3, 3 * scores // 8
        return not plain or self.n < self.threshold_min_rows or self.n <= rows and nq * self.n <= scores

    def _selected_search(self, queries, k: int, q_groups, allowed, doc_lt):
        """Exact top-k in three launches and without a host read: unit queries, scores with the greatest of every 16 rows,
        selection.  (The bound below which parts are not looked into is the k-th greatest of those maxima.)  The usual filters
        and those launches are one call; others take a call for each."""
        rows, nq = self.n, queries.shape[0]
        n = (max(rows, 4) + 3) // 4 * 4
        groups = None if q_groups is None else torch.as_tensor(q_groups, dtype=torch.int32)
        allowed = None if allowed is None else list(allowed)
        limits = None if doc_lt is None else torch.as_tensor(np.asarray(doc_lt, dtype=np.int64))
        self.stats["selected_searches"] = self.stats.get("selected_searches", 0) + 1
        if ((groups is None or self._by_value(groups)) and (allowed is None or len(allowed) == nq <= 65535)
                and (limits is None or limits.numel() == nq and self._by_value(limits))):
            lists = None if allowed is None else self._lists_there(self._id_lists(allowed))
            return ops.selected_search(queries.to(self.device, torch.float32), self.vecs, rows, self.row_group, self.row_ids,
                                       self.row_docs, min(k, n, 1024), None if groups is None else groups.contiguous(), lists,
                                       None if limits is None else limits.contiguous())
        q, qg, allow, n = self._query(queries, groups, allowed, limits)
        scores, parts = ops.scores_and_parts(q, self.vecs, n, self.row_group[:n], qg, allow)
        return ops.top_hits(scores, parts, min(k, n, 1024), self.row_ids, self.row_docs)

    def _sample_rank(self, k: int) -> int:
        """Rank in the row sample whose score is taken as a search's threshold.  The sample holds Binomial(k, 1/stride)
        of a query's k best rows; this is five standard deviations and five rows past its mean (k 250: 19, about 1,200
        candidates; the sample's k-th best, a bound that cannot fail, gave 16,000)."""
        mean = k / self.sample_stride
        return min(k, int(np.ceil(mean + 5 * mean ** 0.5 + 5)), ops.kernels.RANK_MAX)

    def _slack(self, queries: int) -> float:
        """How far the sample's and the scan's scores of one row may lie apart, by which a threshold from the former is
        lowered.  Nothing where one kernel gives both (of the queries' chunks, too).  Else each is a sum of ``dim`` exact
        products in fp32, in some order and with up to 2^-23 of the running sum lost a step, and the lengths are 1 within
        the rounding to bf16.  (On 1M rows of 768 it lets 2 % more candidates through.)"""
        if self.frag and ops.native().index_scan_takes(queries, self.dim):
            return 0.0
        return self.dim * 2.0 ** -22 * (1 + 2.0 ** -6)

    def _threshold_search(self, queries, k: int, q_groups=None):
        """Exact top-k without the [q, n] score matrix: rows that score at least a threshold are appended to a list per
        query, and the list is ranked.  The threshold is the ``_sample_rank``-th best score of a strided row sample.
        It is exact whenever the list holds k rows (or the threshold cut nothing off), which the ranking kernel
        reports per query: one host read at the end, and the rare query that fails it takes ``_safe_search``."""
        q, qg = self._unit(queries, q_groups)
        n4 = (self.n + 3) // 4 * 4
        ns = (self.n // self.sample_stride) // 4 * 4
        if ns < k:  # (``_safe_search`` needs k rows in the sample)
            return None
        samp, samp_group = self._sample_rows(ns)
        if self.frag:
            s_scores = ops.scores_shuffled(q, samp, ns, samp_group, qg)
        else:
            s_scores = ops.gemm_bt(q, samp, epilogue=ops.EPI_SCORES, out_f32=True, row_group=samp_group, q_group=qg)
        r = self._sample_rank(k)
        cap = 4 * r * self.sample_stride + 4096
        step = max(1, self.CAND_BYTES // (8 * cap))
        slack = self._slack(q.shape[0])
        parts = []
        for i in range(0, q.shape[0], step):
            thr, cnt = ops.rank_value(s_scores[i:i + step], r, slack)
            lists = self._candidates(q[i:i + step], thr, cap, n4, None if qg is None else qg[i:i + step], cnt)
            parts.append(ops.rank_hits(*lists, thr, k, self.row_ids, self.row_docs))
        vals, ids, docs, status = parts[0] if len(parts) == 1 else (torch.cat(t) for t in zip(*parts))
        self.stats["threshold_searches"] += len(parts)
        failed = status.cpu().nonzero().flatten()
        if len(failed):
            self.stats["threshold_misses"] = self.stats.get("threshold_misses", 0) + len(failed)
            at = failed.to(self.device)
            fv, rows = self._safe_search(torch.as_tensor(queries)[failed], q[at], s_scores[at] - slack, k, n4,
                                         None if qg is None else qg[at],
                                         None if q_groups is None else [q_groups[i] for i in failed.tolist()])
            vals[at] = fv
            ids[at], docs[at] = ops.hit_ids(fv, rows.to(torch.int32), self.row_ids, self.row_docs)
        return vals, ids, docs

    def _safe_search(self, queries, q, s_scores, k: int, n4: int, qg, q_groups):
        """Threshold search with a bound that holds on any data: the k-th best score over the sample (``s_scores`` are less
        ``_slack``) is a lower bound for the k-th best over all rows, so the list always holds the top k unless it overflows.  A chunk whose
        list overflows is retried or scanned on its own (``_threshold_chunk``)."""
        tv, _ = ops.topk_rows(s_scores, k)
        thr = tv[:, k - 1].contiguous()
        # about k * stride scores clear the sample's k-th best (its rank in the whole index); the
        # lists hold twice that plus a fixed margin (the count's spread is ~sqrt(k) * stride).  Above
        # a byte budget for the [q, cap] lists the queries go through in chunks (k = 1024 at 512
        # queries asked for ~1 GB of candidate memory per search).
        cap = 2 * k * self.sample_stride + 4096
        per_chunk = max(1, self.CAND_BYTES // (8 * cap))
        parts = [self._threshold_chunk(queries, q, thr, k, cap, n4, qg, i, min(i + per_chunk, q.shape[0]), q_groups)
                 for i in range(0, q.shape[0], per_chunk)]
        if len(parts) == 1:
            return parts[0]
        return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])

    def _threshold_chunk(self, queries, q, thr, k: int, cap: int, n4: int, qg, i: int, j: int, q_groups):
        """Queries i:j of a threshold search.  A list that overflows its capacity (clustered data:
        far more rows than k x stride clear the sample's bound) is retried for THIS chunk with the
        capacity it needed, and past the memory budget this chunk alone takes the full score path
        -- never the whole batch."""
        qgs = None if qg is None else qg[i:j]
        got, cmax = self._threshold_candidates(q[i:j], thr[i:j], k, cap, n4, qgs)
        if got is None:
            cap2 = -(-cmax // 1024) * 1024
            if (j - i) * cap2 * 8 <= 4 * self.CAND_BYTES:
                self.stats["threshold_retries"] = self.stats.get("threshold_retries", 0) + 1
                got, _ = self._threshold_candidates(q[i:j], thr[i:j], k, cap2, n4, qgs)
        if got is None:  # this chunk through [chunk, n] score sub-batches
            self.stats["threshold_chunk_full"] = self.stats.get("threshold_chunk_full", 0) + 1
            step = max(1, (1 << 30) // (4 * max(1, self.n)))
            vs, rs = [], []
            for a in range(i, j, step):
                b = min(j, a + step)
                sc = self.scores(queries[a:b], None if q_groups is None else q_groups[a:b])
                v, r = ops.topk_rows(sc, min(k, sc.shape[1], 1024))
                vs.append(v)
                rs.append(r)
            got = (torch.cat(vs), torch.cat(rs))
        return got

    CAND_BYTES = 256 << 20  # candidate-list memory of one threshold search

    def _candidates(self, q, thr, cap: int, n4: int, qg, cnt=None):
        """Candidate lists (scores, rows, counts) of the filtered scores >= thr."""
        if self.frag:
            return ops.score_candidates_shuffled(q, self.vecs, n4, thr, cap, self.row_group[:n4], qg, cnt)
        return ops.score_candidates(q, self.vecs[:n4], thr, cap, self.row_group[:n4], qg, cnt)

    def _threshold_candidates(self, q, thr, k: int, cap: int, n4: int, qg):
        cand_val, cand_idx, cnt = self._candidates(q, thr, cap, n4, qg)
        cmax = int(cnt.max())
        if cmax > cap:
            self.stats["threshold_overflows"] += 1
            return None, cmax
        # only the filled prefix of the lists (the longest one, ~16k of the 36k-entry capacity at
        # k = 250 on unstructured data) is ranked; shorter lists are -inf past their count
        n_use = min(cap, max(k, -(-cmax // 64) * 64))
        vals, pos = ops.topk_rows(cand_val[:, :n_use], min(k, n_use))
        rows = torch.gather(cand_idx, 1, pos.long())
        return (vals, rows.masked_fill(torch.isinf(vals), 0)), cmax

    def _sample_rows(self, ns: int):
        """The strided 1/64 row sample (in the index's own layout) and its groups, cached until the next update."""
        def build():
            rows = torch.arange(0, ns * self.sample_stride, self.sample_stride, device=self.device)
            if self.frag:  # whole tiles of 128 rows: the last row again behind the sample
                padded = torch.arange(-(-ns // 128) * 128, device=self.device).clamp_(max=ns - 1) * self.sample_stride
                data = ops.shuffle_weights(ops.gather_shuffled_rows(self.vecs, padded))
            else:
                data = self.rows_data(rows).contiguous()
            return data, self.row_group[rows]
        return self._kept("_sample", (ns, self._version), build)

    # ------------------------------------------------------------------ persistence
    def save(self, path: str) -> None:
        from safetensors.torch import save_file

        n = self.n
        save_file({"vecs": self.rows_data(torch.arange(n, device=self.device)).contiguous().cpu(),
                   "ids": self.row_ids[:n].cpu(),
                   "docs": self.row_docs[:n].cpu(), "group": self.row_group[:n].cpu()}, path,
                  metadata={"dim": str(self.dim)})

    @classmethod
    def load(cls, path: str, device=None) -> "VectorIndex":
        from safetensors.torch import load_file

        st = load_file(path)
        idx = cls(st["vecs"].shape[1], device, capacity=max(64, st["vecs"].shape[0]), dtype=st["vecs"].dtype)
        n = st["vecs"].shape[0]
        idx._put(torch.arange(n, device=idx.device), st["vecs"].to(idx.device))
        idx.row_ids[:n] = st["ids"].to(idx.device)
        idx.row_docs[:n] = st["docs"].to(idx.device)
        idx.row_group[:n] = st["group"].to(idx.device)
        idx.n = n
        idx._row_of = {int(x): i for i, x in enumerate(st["ids"].tolist()) if x >= 0}
        idx._dead = n - len(idx._row_of)
        idx._twice = int((st["group"] >= 0).sum()) != len(idx._row_of)
        return idx
