"""Tensor-level wrappers of the gfx950 kernels.

Each function validates shapes / dtypes / devices on the host BEFORE launching (a hand-written
kernel that is fed a wrong shape faults the GPU), then enqueues on the current HIP stream, which
makes every op capturable into a HIP graph.  CPU tensors run ``ops.reference``.
"""
from __future__ import annotations

import functools
import math

import torch
import torch.nn.functional as F

from . import reference as ref
from ._lib import expect, expect_bf16_contig, native, ptr, same_device, stream

EPI_NONE, EPI_GELU, EPI_SWIGLU, EPI_SCORES = ref.EPI_NONE, ref.EPI_GELU, ref.EPI_SWIGLU, ref.EPI_SCORES
EPI_SWIGLU8, EPI_GEGLU8, EPI_REGLU8 = ref.EPI_SWIGLU8, ref.EPI_GEGLU8, ref.EPI_REGLU8
GLU8 = (EPI_SWIGLU8, EPI_GEGLU8, EPI_REGLU8)  # gated epilogues over 8-row [gate | up] groups
_GLU_ALL = (EPI_SWIGLU, *GLU8)


def _i32(t: torch.Tensor) -> None:
    if t.dtype != torch.int32 or not t.is_contiguous():
        raise TypeError("expected a contiguous int32 tensor")


# ----------------------------------------------------------------------------------------------
# normalisation / embeddings / pooling


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, residual: torch.Tensor | None = None):
    """RMSNorm over the last dim; with ``residual`` the input is ``x + residual`` and the sum is
    also returned (fused residual stream).  Returns (out, residual_out).

    ``x`` may also be split-K slabs [S, rows, cols] (fp32, or bf16: ``slab_dtype``) of the producing
    projection (``stream_gemm(..., splits=S)``): they are summed in fp32 (and rounded to bf16) inside
    the kernel."""
    slabs = x.dim() == 3 and x.dtype in (torch.float32, torch.bfloat16)
    if not x.is_cuda:
        if slabs:
            x = x.float().sum(0).to(torch.bfloat16)
        return ref.rmsnorm(x, w, eps, residual)
    expect_bf16_contig(w, residual)
    same_device(x, w, residual)
    cols = x.shape[-1]
    expect(w.numel() == cols, "rmsnorm weight size mismatch")
    if slabs:
        expect(x.is_contiguous(), "slabs must be contiguous")
        S, rows = x.shape[0], x.shape[1]
        shape = (rows, cols)
    else:
        expect_bf16_contig(x)
        rows = x.numel() // cols
        shape = tuple(x.shape)
    expect(residual is None or tuple(residual.shape) == shape, "residual shape mismatch")
    out = torch.empty(shape, dtype=torch.bfloat16, device=x.device)
    res_out = torch.empty(shape, dtype=torch.bfloat16, device=x.device) if residual is not None else None
    if slabs:
        native().rmsnorm_slabs(ptr(out), ptr(res_out), ptr(x), S, rows * cols, ptr(residual), ptr(w), rows, cols,
                               float(eps), stream(x), int(x.dtype == torch.bfloat16))
    else:
        native().rmsnorm(ptr(out), ptr(res_out), ptr(x), ptr(residual), ptr(w), rows, cols, float(eps), stream(x))
    return out, res_out


def layernorm(x, gamma, beta, eps, residual=None):
    if not x.is_cuda:
        return ref.layernorm(x, gamma, beta, eps, residual)
    expect_bf16_contig(x, gamma, beta, residual)
    same_device(x, gamma, beta, residual)
    cols = x.shape[-1]
    rows = x.numel() // cols
    expect(gamma.numel() == cols and beta.numel() == cols, "layernorm affine size mismatch")
    expect(residual is None or residual.shape == x.shape, "residual shape mismatch")
    out = torch.empty_like(x)
    native().layernorm(ptr(out), ptr(x), ptr(residual), ptr(gamma), ptr(beta), rows, cols, float(eps), stream(x))
    return out


def bert_embed(ids, pos_ids, type_ids, word, pos, typ, gamma, beta, eps):
    if not ids.is_cuda:
        return ref.bert_embed(ids, pos_ids, type_ids, word, pos, typ, gamma, beta, eps)
    _i32(ids)
    _i32(pos_ids)
    if type_ids is not None:
        _i32(type_ids)
    expect_bf16_contig(word, pos, typ, gamma, beta)
    expect(ids.shape == pos_ids.shape, "ids / position ids mismatch")
    H = word.shape[1]
    out = torch.empty((ids.numel(), H), dtype=word.dtype, device=ids.device)
    native().bert_embed(ptr(out), ptr(ids), ptr(pos_ids), ptr(type_ids), ptr(word), ptr(pos), ptr(typ), ptr(gamma),
                        ptr(beta), ids.numel(), H, float(eps), stream(ids))
    return out


def embed_gather(ids, table):
    if not ids.is_cuda:
        return ref.embed_gather(ids, table)
    _i32(ids)
    expect_bf16_contig(table)
    out = torch.empty((ids.numel(), table.shape[1]), dtype=table.dtype, device=ids.device)
    native().embed_gather(ptr(out), ptr(ids), ptr(table), ids.numel(), table.shape[1], stream(ids))
    return out


def mean_pool(hidden, cu_seqlens, normalize=False, want_bf16=False, out=None, rows=None):
    """Mean over each packed sequence (all tokens, as the reference).  Returns fp32 [B, H]
    (and a bf16 copy when ``want_bf16``).  ``out`` fp32 [n, H] and ``rows`` int32 [B] (distinct, inside [0, n)):
    sequence b goes to out[rows[b]], and out is returned."""
    if not hidden.is_cuda:
        res = ref.mean_pool(hidden, cu_seqlens, normalize)
        if out is not None:
            out[rows.long()] = res
            res, copy = out, res
        else:
            copy = res
        return (res, copy.to(torch.bfloat16)) if want_bf16 else res
    expect_bf16_contig(hidden)
    _i32(cu_seqlens)
    B = cu_seqlens.numel() - 1
    H = hidden.shape[1]
    expect(H <= 4096, "mean_pool supports hidden <= 4096")
    expect((out is None) == (rows is None), "mean_pool: out and rows together")
    if out is None:
        out = torch.empty((B, H), dtype=torch.float32, device=hidden.device)
    else:
        _i32(rows)
        same_device(hidden, out, rows)
        expect(out.dtype == torch.float32 and out.is_contiguous() and out.dim() == 2 and out.shape[1] == H
               and rows.numel() == B and out.shape[0] >= B, "mean_pool: out fp32 [n >= B, H], one row a sequence")
    ob = torch.empty((B, H), dtype=torch.bfloat16, device=hidden.device) if want_bf16 else None
    native().mean_pool(ptr(out), ptr(ob), ptr(hidden), ptr(cu_seqlens), B, H, int(bool(normalize)), stream(hidden), ptr(rows))
    return (out, ob) if want_bf16 else out


def encoder_forward(ids, pos_ids, cu_seqlens, max_seqlen: int, heads: int, eps: float, tables, layers):
    """Hidden states [T, H] of the packed token ids through a post-LN encoder in one native call, or None where an
    operand is not what it takes (the caller then runs the ops one by one, which report it).  ``tables``: word,
    position and type embeddings, gain and offset of their norm; ``layers``: per layer qkv, o, ln1, i, d, ln2 as pairs
    of a weight [N, K] and a bias, or a gain and an offset."""
    word = tables[0]
    if not ids.is_cuda or word.dim() != 2 or not layers:
        return None
    dev, bf, H, T = ids.device, torch.bfloat16, word.shape[1], ids.numel()
    F_ = layers[0][6].shape[0]
    if (T == 0 or max_seqlen <= 0 or H % 64 or F_ % 64 or heads <= 0 or H % heads or H // heads not in (32, 64, 128) or H > 4096
            or cu_seqlens.numel() < 2 or ids.shape != pos_ids.shape):
        return None
    for t in (ids, pos_ids, cu_seqlens):
        if t.dtype != torch.int32 or not t.is_contiguous() or t.device != dev:
            return None
    shapes = ((3 * H, H), (3 * H,), (H, H), (H,), (H,), (H,), (F_, H), (F_,), (H, F_), (H,), (H,), (H,))
    # twelve tensors a layer are looked at natively (144 of them 65 us -> 13); what that does not take is looked at here
    api = getattr(torch.Tensor, "__dlpack_c_exchange_api__", None)
    flat = None if api is None else native().operand_ptrs(api, torch.Tensor, ids, layers, shapes)
    if flat is None:
        flat = []
        for layer in layers:
            for t, shape in zip(layer, shapes):
                if t.shape != shape or t.dtype != bf or not t.is_contiguous() or t.device != dev:
                    return None
                flat.append(t.data_ptr())
    for t in tables:
        if t.shape[-1] != H or t.dtype != bf or not t.is_contiguous() or t.device != dev:
            return None
    x, y, att = (torch.empty((T, H), dtype=bf, device=dev) for _ in range(3))
    qkv, ffn = torch.empty((T, 3 * H), dtype=bf, device=dev), torch.empty((T, F_), dtype=bf, device=dev)
    slices = native().slab_slices(T, H, F_)
    slabs = torch.empty((slices, T, H), dtype=torch.float32, device=dev) if slices else None
    native().encoder_forward(ptr(ids), ptr(pos_ids), ptr(cu_seqlens), T, cu_seqlens.numel() - 1, int(max_seqlen), H, heads,
                             F_, float(eps), *(ptr(t) for t in tables), flat, ptr(x), ptr(y), ptr(att), ptr(qkv), ptr(ffn),
                             ptr(slabs), stream(ids))
    return x


def linear_layernorm(x, w, b, residual, gamma, beta, eps):
    """LayerNorm(x w^T + b + residual) of contiguous rows: in K-slices that the norm sums in 32 bits where that is the faster
    (``slab_slices`` in gemm_small.hip), else ``linear`` and ``layernorm``."""
    (M, K), N = x.shape, w.shape[0]
    slices = native().slab_slices(M, N, K) if x.is_cuda and w.dim() == 2 else 0
    operands = (x, w, b, residual, gamma, beta)
    if (not slices or any(t.dtype != torch.bfloat16 or not t.is_contiguous() or t.device != x.device for t in operands)
            or w.shape[1] != K or residual.shape != (M, N) or any(t.shape != (N,) for t in (b, gamma, beta))
            or (ptr(x) | ptr(w)) % 16 or (ptr(b) | ptr(residual) | ptr(gamma) | ptr(beta)) % 4):
        return layernorm(linear(x, w, b, residual=residual), gamma, beta, eps)
    slabs = torch.empty((slices, M, N), dtype=torch.float32, device=x.device)
    out = torch.empty_like(residual)
    native().gemm_slab(ptr(x), ptr(w), ptr(slabs), M, N, K, stream(x))
    native().layernorm_slabs(ptr(out), ptr(slabs), slices, ptr(b), ptr(residual), ptr(gamma), ptr(beta), M, N, float(eps),
                             stream(x))
    return out


# ----------------------------------------------------------------------------------------------
# element-wise


def gelu(x, bias=None, out=None):
    if not x.is_cuda:
        return ref.gelu(x, bias)
    expect_bf16_contig(x, bias)
    cols = x.shape[-1]
    out = torch.empty_like(x) if out is None else out
    native().gelu(ptr(out), ptr(x), ptr(bias), x.numel() // cols, cols, stream(x))
    return out


def silu_mul(x, interleaved=False, group: int | None = None):
    """x [..., 2F] = [gate | up] -> silu(gate) * up  [..., F].  ``group`` (or ``interleaved`` = 16):
    x columns are ``group``-wide [gate | up] groups (the projection of ``interleave_gate_up``
    weights; 0 = stacked halves)."""
    group = (16 if interleaved else 0) if group is None else int(group)
    if not x.is_cuda:
        if group:
            F2 = x.shape[-1]
            v = x.reshape(*x.shape[:-1], F2 // (2 * group), 2, group)
            x = torch.cat([v[..., 0, :].reshape(*x.shape[:-1], F2 // 2), v[..., 1, :].reshape(*x.shape[:-1], F2 // 2)], -1)
        return ref.silu_mul(x)
    expect(group in (0, 16), "the GPU silu_mul takes stacked or 16-column groups (8-row groups: EPI_SWIGLU8)")
    expect_bf16_contig(x)
    F2 = x.shape[-1]
    rows = x.numel() // F2
    out = torch.empty((*x.shape[:-1], F2 // 2), dtype=x.dtype, device=x.device)
    native().silu_mul(ptr(out), ptr(x), rows, F2 // 2, stream(x), int(group == 16))
    return out


def rope_kv_write(qkv, positions, cos_sin, k_cache, v_cache, slots, Hq, Hkv, D, write_q=True):
    """Applies RoPE to the q/k heads of ``qkv`` [T, (Hq+2Hkv)*D]; writes k, v into the paged caches
    [num_blocks, Hkv, block_size, D] at ``slots`` (int64, <0 skipped); returns q [T, Hq, D].
    ``qkv`` may also be split-K slabs [S, T, (Hq+2Hkv)*D] (fp32 or bf16), summed inside the kernel.
    ``write_q=False`` (bf16 ``qkv``): k / v only, returns None (the prefill attention rotates q on
    load: ``flash_attention_paged(..., rope=...)``)."""
    block_size = k_cache.shape[2]
    slabs = qkv.dim() == 3 and qkv.dtype in (torch.float32, torch.bfloat16)
    if not qkv.is_cuda:
        if slabs:
            qkv = qkv.float().sum(0).to(torch.bfloat16)
        return ref.rope_kv_write(qkv, positions, cos_sin, k_cache, v_cache, slots, Hq, Hkv, D, block_size)
    expect_bf16_contig(k_cache, v_cache)
    _i32(positions)
    expect(slots.dtype == torch.int64 and slots.is_contiguous(), "slots must be contiguous int64")
    expect(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous(), "cos_sin must be contiguous fp32")
    T = qkv.shape[-2]
    expect(qkv.shape[-1] == (Hq + 2 * Hkv) * D, "qkv width mismatch")
    expect(positions.numel() == T and slots.numel() == T, "positions / slots length mismatch")
    expect(tuple(k_cache.shape[1:]) == (Hkv, block_size, D) and k_cache.shape == v_cache.shape, "cache shape mismatch")
    expect(cos_sin.shape[1] == D // 2, "cos/sin table width mismatch")
    if not write_q:
        expect(not slabs, "write_q=False needs a bf16 qkv")
        expect_bf16_contig(qkv)
        native().rope_kv_write(ptr(qkv), qkv.stride(0), ptr(positions), ptr(cos_sin), 0, ptr(k_cache),
                               ptr(v_cache), ptr(slots), T, Hq, Hkv, D, block_size, stream(qkv))
        return None
    q = torch.empty((T, Hq, D), dtype=torch.bfloat16, device=qkv.device)
    if slabs:
        expect(qkv.is_contiguous(), "slabs must be contiguous")
        native().rope_kv_write(0, qkv.shape[-1], ptr(positions), ptr(cos_sin), ptr(q), ptr(k_cache), ptr(v_cache),
                               ptr(slots), T, Hq, Hkv, D, block_size, stream(qkv), ptr(qkv), qkv.shape[0],
                               T * qkv.shape[-1], int(qkv.dtype == torch.bfloat16))
    else:
        expect_bf16_contig(qkv)
        native().rope_kv_write(ptr(qkv), qkv.stride(0), ptr(positions), ptr(cos_sin), ptr(q), ptr(k_cache),
                               ptr(v_cache), ptr(slots), T, Hq, Hkv, D, block_size, stream(qkv))
    return q


# ----------------------------------------------------------------------------------------------
# attention


def _head_strides(t: torch.Tensor):
    # t viewed as [tokens, heads, D] with unit stride on D
    expect(t.stride(-1) == 1, "attention operands need unit stride on the head dim")
    return t.stride(0), t.stride(1)


def flash_attention_packed(q, k, v, cu_q, cu_k, max_seqlen_q, causal=False, scale=None, out=None):
    """Variable-length attention over packed sequences.  q [Tq, Hq, D], k/v [Tk, Hkv, D] may be
    strided views of a fused QKV buffer.  Returns [Tq, Hq, D] contiguous."""
    D = q.shape[-1]
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    if not q.is_cuda:
        return ref.flash_attention_packed(q, k, v, cu_q, cu_k, causal, scale)
    _i32(cu_q)
    _i32(cu_k)
    expect(q.dtype == torch.bfloat16 and k.dtype == torch.bfloat16 and v.dtype == torch.bfloat16, "bf16 required")
    expect(D in (32, 64, 128), "head dim must be 32, 64 or 128")
    Hq, Hkv = q.shape[1], k.shape[1]
    expect(Hq % Hkv == 0, "GQA requires Hq % Hkv == 0")
    expect(k.stride() == v.stride(), "k and v must share strides")
    qst, qsh = _head_strides(q)
    kst, ksh = _head_strides(k)
    for s in (qst, qsh, kst, ksh):
        expect(s % 8 == 0, "attention strides must be multiples of 8 elements (16 B)")
    out = torch.empty((q.shape[0], Hq, D), dtype=q.dtype, device=q.device) if out is None else out
    B = cu_q.numel() - 1
    native().flash_attention(ptr(q), qst, qsh, ptr(k), ptr(v), kst, ksh, 0, 0, 0, 0, 0, ptr(out), out.stride(0),
                             out.stride(1), ptr(cu_q), ptr(cu_k), 0, B, int(max_seqlen_q), Hq, Hkv, D,
                             int(bool(causal)), 0, float(scale), stream(q))
    return out


def flash_rope_ok(D: int, block_size: int) -> bool:
    """Whether flash_attention_paged can rotate q itself (the 32x32 D = 128 kernel's Q prologue)."""
    return D == 128 and block_size % 64 == 0


def flash_attention_paged(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, max_seqlen_q, causal=True, scale=None,
                          out=None, rope=None):
    """Prefill attention: q [Tq, Hq, D] packed by cu_q, keys/values of each sequence are its first
    ctx_lens[b] tokens in the paged caches (the query chunk is the tail of that context).
    ``rope=(positions int32 [Tq], cos_sin [max_pos, D/2, 2] fp32)``: q is the un-rotated projection
    and RoPE is applied on load (``flash_rope_ok``)."""
    D = q.shape[-1]
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    if not q.is_cuda:
        if rope is not None:
            pos, cs = rope
            T, Hq = q.shape[0], q.shape[1]
            q = ref.rope_q(q.reshape(T, Hq, D), pos, cs)
        return ref.flash_attention_paged(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, causal, scale)
    _i32(cu_q)
    _i32(ctx_lens)
    _i32(block_tables)
    expect_bf16_contig(k_cache, v_cache)
    expect(D in (32, 64, 128), "head dim must be 32, 64 or 128")
    Hq, Hkv, bs = q.shape[1], k_cache.shape[1], k_cache.shape[2]
    qst, qsh = _head_strides(q)
    out = torch.empty((q.shape[0], Hq, D), dtype=q.dtype, device=q.device) if out is None else out
    B = cu_q.numel() - 1
    expect(block_tables.shape[0] >= B and ctx_lens.numel() >= B, "block table / ctx_lens rows < batch")
    if rope is not None:
        pos, cs = rope
        _i32(pos)
        expect(flash_rope_ok(D, bs) and cs.dtype == torch.float32 and cs.is_contiguous() and pos.numel() == q.shape[0],
               "q RoPE in the attention needs D 128, block size % 64, fp32 cos/sin and one position per query")
        native().flash_attention_rope(ptr(q), qst, qsh, ptr(k_cache), ptr(v_cache), ptr(block_tables),
                                      block_tables.shape[1], bs, ptr(out), out.stride(0), out.stride(1), ptr(cu_q),
                                      ptr(ctx_lens), B, int(max_seqlen_q), Hq, Hkv, D, int(bool(causal)),
                                      float(scale), ptr(pos), ptr(cs), stream(q))
        return out
    native().flash_attention(ptr(q), qst, qsh, 0, 0, 0, 0, ptr(k_cache), ptr(v_cache), ptr(block_tables),
                             block_tables.shape[1], bs, ptr(out), out.stride(0), out.stride(1), ptr(cu_q), 0,
                             ptr(ctx_lens), B, int(max_seqlen_q), Hq, Hkv, D, int(bool(causal)), 1, float(scale),
                             stream(q))
    return out


class DecodeWorkspace:
    """Partition buffers of the split-K paged decode; allocated once (graph-capture safe)."""

    def __init__(self, max_batch, Hq, D, max_parts, device):
        self.max_parts = max_parts
        self.o = torch.empty((max_batch * Hq * max_parts * D,), dtype=torch.float32, device=device)
        self.m = torch.empty((max_batch * Hq * max_parts,), dtype=torch.float32, device=device)
        self.l = torch.empty((max_batch * Hq * max_parts,), dtype=torch.float32, device=device)
        # partition arrival counters of the in-launch combine (one per (sequence, kv head) <= Hq);
        # zero at rest: the last arriving workgroup resets its counter
        self.cnt = torch.zeros((max_batch * Hq,), dtype=torch.int32, device=device)


def decode_rope_ok(batch: int, Hkv: int, D: int, part_size: int) -> bool:
    """Decode steps whose rotary embedding and cache write ``paged_decode_rope`` does inside the attention."""
    return bool(native().decode_rope_ok(batch, Hkv, D, part_size))


def paged_decode_rope(qkv, positions, cos_sin, k_cache, v_cache, slots, Hq, block_tables, ctx_lens, part_size=512,
                      workspace: DecodeWorkspace | None = None, order=None, warm=None):
    """``rope_kv_write`` and ``paged_decode`` of a decode step in one launch (``decode_rope_ok``): ``qkv`` bf16 rows or split-K
    slabs, the step's token the last of each context."""
    slabs = qkv.dim() == 3
    Hkv, D = k_cache.shape[1], k_cache.shape[3]
    T, width = qkv.shape[-2:]
    expect(qkv.is_cuda and qkv.is_contiguous() and qkv.dtype in ((torch.float32, torch.bfloat16) if slabs else (torch.bfloat16,)),
           "paged_decode_rope: contiguous bf16 rows or slabs")
    expect(width == (Hq + 2 * Hkv) * D and positions.numel() == T and slots.numel() == T, "qkv width, positions and slots")
    _i32(positions)
    expect(slots.dtype == torch.int64 and slots.is_contiguous(), "slots must be contiguous int64")
    expect(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and cos_sin.shape[1] == D // 2, "cos_sin: fp32 [pos, D / 2, 2]")
    expect(workspace is not None and decode_rope_ok(T, Hkv, D, part_size), "paged_decode_rope: a workspace, batch, heads, partition")
    out = torch.empty((T, Hq, D), dtype=torch.bfloat16, device=qkv.device)
    rope = (ptr(qkv), int(qkv.dtype == torch.bfloat16), qkv.shape[0] if slabs else 1, width, ptr(positions), ptr(cos_sin), ptr(slots))
    return paged_decode(out, k_cache, v_cache, block_tables, ctx_lens, part_size, workspace, out=out, order=order, warm=warm, rope=rope)


def paged_decode(q, k_cache, v_cache, block_tables, ctx_lens, part_size=512, workspace: DecodeWorkspace | None = None,
                 scale=None, out=None, order=None, warm=None, rope=None):
    """q [B, Hq, D] (one new token per sequence) over the paged caches.  ``order`` (int32 [B], a
    permutation of the batch) is the order the (sequence, kv head) items are dispatched in: longest
    context first balances the two rounds of workgroups every CU runs at RAG batch sizes.  Any
    permutation is correct: the kernel bounds its partition walk by its own max over ctx_lens.

    ``warm`` = ``([(tensor, nbytes), ...up to 2], blocks)``: ``blocks`` workgroups appended to the
    launch read the first ``nbytes`` of each tensor into the Infinity Cache (the next projections'
    weights, while the latency-bound attention leaves the CUs idle); the output is unchanged."""
    B, Hq, D = q.shape
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    if not q.is_cuda:
        return ref.paged_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale)
    _i32(ctx_lens)
    _i32(block_tables)
    expect_bf16_contig(q, k_cache, v_cache)
    Hkv, bs = k_cache.shape[1], k_cache.shape[2]
    expect(D in (64, 128), "decode head dim must be 64 or 128")
    expect(Hq % Hkv == 0 and Hq // Hkv <= 16, "GQA group must be <= 16")
    expect(part_size % 128 == 0, "part_size must be a multiple of 128")
    expect(block_tables.shape[0] >= B and ctx_lens.numel() >= B, "block table / ctx_lens rows < batch")
    max_parts = workspace.max_parts if workspace is not None else 1
    if workspace is None:
        # single partition covering the longest allowed context
        part_size = max(part_size, ((block_tables.shape[1] * bs + 127) // 128) * 128)
        ws_o = ws_m = ws_l = ws_c = None
    else:
        expect(workspace.o.numel() >= B * Hq * max_parts * D and workspace.cnt.numel() >= B * Hkv,
               "decode workspace too small")
        ws_o, ws_m, ws_l, ws_c = workspace.o, workspace.m, workspace.l, workspace.cnt
    out = torch.empty_like(q) if out is None else out
    if order is not None:
        _i32(order)
        expect(order.is_cuda and order.numel() >= B, "decode order must hold the batch")
    wargs = {}
    if warm is not None and warm[1] > 0:
        ranges, blocks = warm
        expect(1 <= len(ranges) <= 2 and 0 < blocks <= 1024, "warm: 1-2 ranges, 1-1024 workgroups")
        for i, (t, nb) in enumerate(ranges):
            expect(t.is_cuda and t.is_contiguous() and 0 < nb <= t.numel() * t.element_size() and nb % 16 == 0,
                   "warm range must be a 16-B multiple inside a contiguous device tensor")
            wargs[f"w{i}"], wargs[f"w{i}_bytes"] = ptr(t), int(nb)
        wargs["w_blocks"] = int(blocks)
    if rope is not None:  # (``paged_decode_rope``: q is only its shape)
        wargs["rope"] = rope
    native().paged_decode_attention(ptr(q), ptr(k_cache), ptr(v_cache), ptr(block_tables), block_tables.shape[1], bs,
                                    ptr(ctx_lens), ptr(out), ptr(ws_o), ptr(ws_m), ptr(ws_l), ptr(ws_c), B, Hq, Hkv,
                                    D, int(part_size), int(max_parts), float(scale), stream(q), ptr(order), **wargs)
    return out


# ----------------------------------------------------------------------------------------------
# GEMM


# gemm_mid from the first row: at M <= 191 the 128 x 128 kernel re-reads the weights per row tile
# and leaves most CUs idle -- Llama-3-8B qkv / o / gate_up / down at M = 129-187: 54 / 54 / 72 / 181
# us against 31 / 29 / 67 / 47 (profiles/small_prefill_r6.md; decode-sized prefill steps of the
# fragment-layout decoder stream instead, models/llama.py PREFILL_STREAM_MAX_M)
GEMM_MID_MIN_M = 1


def _g256_fill(M: int, N: int) -> tuple[int, float]:
    """(256 x 256 tiles, share of the last-wave-padded CU slots they fill) of gemm256 on 256 CUs."""
    tiles = -(-M // 256) * (N // 256)
    return tiles, tiles / (-(-tiles // 256) * 256)


def use_gemm_mid(M: int, N: int, K: int, lda: int) -> bool:
    """Mid-M shapes on fragment-layout weights go to the stream-K kernel (gemm_mid.hip) where the
    256 x 256 kernel would leave CUs idle: fewer than GEMM256_FILL (192) tiles, or a last wave that
    leaves the chip under 70 % busy.  Measured (profiles/gemm_mid_r6.md): Llama-3-8B qkv / o / down
    at M = 384..2048 run 1.2-2.5x faster than the round-5 dispatch, gate_up at M = 640 / 768 (336
    tiles = 1.31 waves) 12 % faster than gemm256; gate_up at 384 / 512 / 1024 / 2048 and qkv at
    2048 stay on gemm256."""
    if M < GEMM_MID_MIN_M or N % 256 or not gemm_mid_ok(M, N, K, lda):
        return False
    tiles, fill = _g256_fill(M, N)
    return tiles < native().GEMM256_FILL or fill < 0.7


def use_gemm256(M: int, N: int, K: int, lda: int, ldb: int) -> bool:
    """Whether the phased 256x256 kernel takes a shape instead of the 128x128 one (``gemm256_wins`` in gemm256.hip)."""
    return native().gemm256_wins(M, N) and bool(native().gemm256_ok(M, N, K, lda, ldb))


def _g256_us(tiles: int, K: int) -> float:
    """Estimated time of gemm256: whole waves of 256 tiles, each K-step slower the more of the chip works (the clock, from
    some 144 workgroups on)."""
    if not tiles:
        return 0.0
    waves = -(-tiles // 256)
    return waves * K * (0.0133 + 0.0073 * max(0.5625, tiles / (256 * waves))) + 4 + 2 * waves


def _mid_us(M: int, tiles_n: int, K: int) -> float:
    """Estimated time of gemm_mid: lockstep groups of ceil(M / 128) workgroups share its (weight tile, K-step) plane;
    tiles that groups share are combined at the end (``gemm_mid_us`` in gemm_mid.hip)."""
    return native().gemm_mid_us(M, 256 * tiles_n, K)


def _mid(M: int, tiles_n: int, K: int):
    """(estimated us, kind) of a part on gemm_mid: on tiles of 192 rows where those are 3 % quicker by the estimates than the
    kernel that it takes by itself (26 of 108 sizes, 1.11 times as fast in the mean, the least 0.99): fewer rows past the
    prompt's end than with 256, fewer loads into a CU than with 128.  us, (768, 4096, 14336) 101 -> 89, (1093, 4096, 14336) 131 ->
    122, (1300, 6144, 4096) 77 -> 68, (2300, 4096, 4096) 84 -> 70, (1500, 16384, 2048) 105 -> 88."""
    us, us192 = _mid_us(M, tiles_n, K), native().gemm_mid_192_us(M, 256 * tiles_n, K)
    return (us192, "192") if us192 < 0.97 * us else (us, "mid")


@functools.lru_cache(maxsize=4096)
def _frag_plan(M: int, N: int, K: int, cols: bool, frag: bool):
    """``frag_plan`` and the estimate of its time."""
    tm, tn = -(-M // 256), N // 256
    mid_us, mid = _mid(M, tn, K)
    one = {"256": _g256_us(tm * tn, K), mid: mid_us}
    if use_gemm_mid(M, N, K, K):
        best = mid
    elif use_gemm256(M, N, K, K, K):
        best = "256"
    else:
        return None, float("inf")
    other = "256" if best == mid else mid
    if one[other] < 0.985 * one[best]:
        best = other
    plan, took, least = ((best, M, N), None), one[best], 0.95 * one[best]
    for waves in range(1, tm * tn // 256 + 1):
        n1, m1 = waves * 256 // tm, waves * 256 // tn
        if cols and 0 < n1 < tn:
            us, kind = _mid(M, tn - n1, K)
            us += _g256_us(tm * n1, K)
            if us < least:
                plan, took, least = (("256", M, 256 * n1), (kind, M, N - 256 * n1)), us, us
        if 0 < m1 < tm:
            us, kind = _mid(M - 256 * m1, tn, K)
            us += _g256_us(m1 * tn, K)
            if us < least:
                plan, took, least = (("256", 256 * m1, N), (kind, M - 256 * m1, N)), us, us
    us = native().frag_us(M, N, K, 1) if frag else float("inf")
    if us < 0.93 * took:
        return (("frag", M, N), None), us
    if frag and plan[1] is not None:  # the same division with gemm_frag behind the waves
        kind, m, n = plan[1]
        mid, us = _mid(m, n // 256, K)[0], native().frag_us(max(m, 65), n, K, 1)
        if us < 0.93 * mid:
            return (plan[0], ("frag", m, n)), took - mid + us
    return plan, took


def frag_plan(M: int, N: int, K: int, cols: bool = True, frag: bool = True):
    """How a projection with fragment-layout weights that both gemm256 and gemm_mid take is run: (first kernel, its
    rows, its columns) and the same of what remains (or None).  ``cols``: its columns may be divided; ``frag``: gemm_frag takes
    its operands.

    gemm256 alone pays a whole wave of 256 tiles for the last few (Llama-3-8B gate_up at M = 1093: 560 tiles, 235 us
    where two waves take 157), gemm_mid runs at about half its rate but divides evenly.  So the whole waves go to
    gemm256 and the remaining columns (or rows) to gemm_mid where the estimates (fitted to both kernels at the four
    projections of Llama-3-8B and Llama-3.2-1B, M = 300..5000, mostly within 10 %) gain more than 5 % over one kernel;
    between one or the other alone the old bounds (GEMM256_FILL, 70 % of a wave) decide unless the other's estimate is
    1.5 % lower.  us, before -> with the plan: gate_up M 513 137 -> 127, 1093 233 -> 213, 700 181 -> 148, qkv 1700 92 -> 77,
    2600 157 -> 118, o 2300 93 -> 72, down 2200 338 -> 236, 4300 533 -> 357.

    Outside that range the estimates only have to order the two kernels: over 24 shapes with N and K of 256..28,672 and M 1
    ..16,000 the plan differs from the old bounds 196 times and is 0.97..2.05 times as fast, median 1.53: few tiles of a
    short K are the quicker on gemm256 ((44, 512, 4096) 114 -> 62 us, (256, 4096, 512) 22.9 -> 14.6); the worst are (257,
    8192, 1024) 21.3 -> 22.0 and (1093, 4096, 1024) 22.4 -> 23.1.

    gemm_frag, whole, where its estimate is 7 % below: over M 96..2300 at 19 pairs of N 1024..28,672 and K 1024..14,336 that
    is 236 of 414 sizes, 1.64 times as fast in the mean, none slower (at 4 % below two of 271 are 7-9 % slower).  Behind whole
    waves of gemm256 in gemm_mid's place by the same line, where the product is divided without it, too (a call of Llama-3.2-1B,
    1,200 tokens 3,451 -> 3,391, 2,300 4,980 -> 4,870; where it alone makes the division pay, 1,300 tokens 3,497 -> 3,659)."""
    return _frag_plan(M, N, K, cols, frag)[0]


@functools.lru_cache(maxsize=4096)
def corner_plan(M: int, N: int, K: int):
    """(tile columns of 256 that gemm256 takes of the prompt's last rows, the estimate), or (0, None): all it takes of a product
    are whole waves of tiles, and gemm_frag what is left of the last row of them, where that is 1.5 % quicker by the estimates than
    ``frag_plan``.  The last rows are up to 256, often few; a tile of them takes as long as any.  us: (1093, 28672, 4096) GLU 234 ->
    219, (1600, 28672, 4096) 306 -> 285, (3333, 28672, 4096) 599 -> 552, (2760, 6144, 4096) 116 -> 104; a call of Llama-3-8B, 1,093
    tokens 15,890 -> 15,700, 1,600 21,214 -> 20,604, 2,400 27,957 -> 27,536, 3,332 38,536 -> 37,416; as before (0.997-1.003) at
    1,000, 4,000 and 7,900.  Left: (640, 28672, 4096), 80 of 336 tiles, alone 145 -> 135, but a call 10,775 -> 10,878."""
    tm, tn = -(-M // 256), N // 256
    waves = tm * tn // 256
    left = tm * tn - 256 * waves
    if tm < 2 or not waves or not 0 < left < tn or not native().gemm256_ok(M, N, K, K, K):
        return 0, None
    # (its weights, which gemm256 has read already, come from memory again, and slower than a projection's: 3.5 TB/s in calls)
    us = _g256_us(256 * waves, K) + max(native().frag_us(max(M - 256 * (tm - 1), 65), 256 * left, K, 1), 3 + 512 * left * K / 3.5e6)
    return (tn - left, us) if us < 0.985 * _frag_plan(M, N, K, True, True)[1] else (0, None)


def _run_corner(tail: int, A, B, out, residual, epilogue, b_group):
    """gemm256's whole waves and gemm_frag's corner behind them (``corner_plan``)."""
    m, n = (A.shape[0] - 1) // 256 * 256, 256 * tail
    _gemm256_into(A, B, out, None, residual, epilogue, True, b_group, tail)
    gemm_frag(A[m:], B[n:], residual=None if residual is None else residual[m:, n:], epilogue=epilogue,
              out=out[m:, n // (2 if epilogue in GLU8 else 1):], b_group=b_group)
    return out


@functools.lru_cache(maxsize=4096)
def frag_slices(M: int, N: int, K: int) -> int:
    """K-slices that ``gemm_frag`` leaves as fp32 slabs to the norm behind a projection with a residual, 0: the whole product
    is the quicker, or its time not known (K an odd multiple of 64 of several thousand rows, the 128 x 128 kernel's: (3500, 4096,
    1600) with the norm 68 whole, 97 in slices).  The norm reads them at some 4.5 TB/s.  us of product and norm, whole on the quickest kernel -> in slices:
    (260, 2048, 8192) 33.5 -> 23.8, (515, 2048, 8192) 39.8 -> 35.6, (140, 4096, 14336) 57 -> 39.7, (260, 4096, 14336) 62.6 ->
    55.4; (1093, 2048, 8192) 57.4 -> 53.1."""
    whole = corner_plan(M, N, K)[1] or _frag_plan(M, N, K, True, True)[1]
    if whole == float("inf"):
        return 0
    best, least = 0, 0.95 * whole
    for s in (2, 3, 4, 6, 8):
        us = native().frag_us(M, N, K, s) + 0.7 + 4 * s * M * N / 4.5e6 if K // 64 >= 4 * s else float("inf")
        if us < least:
            best, least = s, us
    return best


@functools.lru_cache(maxsize=4096)
def _frag_ok(M: int, N: int, K: int, lda: int) -> bool:
    return native().gemm_frag_ok(M, N, K, lda)


@functools.lru_cache(maxsize=4096)
def _gemm256_ok(M: int, N: int, K: int, lda: int) -> bool:
    """Whether gemm256 takes a projection with fragment-layout weights."""
    return bool(native().gemm256_ok(M, N, K, lda, K))


def gemm_frag(A, B, residual=None, epilogue=EPI_NONE, out=None, b_group: int = 1, glu_bias=None, slices: int = 0, tile: int = -1,
              checked: bool = False):
    """C = A . B^T (+ residual) or a GLU over 8-row [gate | up] groups, B a ``shuffle_weights`` copy, on tiles of 32 x 64 to 128 x
    256 (``gemm_frag.hip``).  ``slices`` S > 0: the K-slices' sums as fp32 slabs [S, M, N] for ``rmsnorm``.  ``tile`` (tests): that
    one instead of the one with the least estimate.  ``checked``: the operands and ``out`` have passed ``gemm_bt``'s checks."""
    M, K = A.shape
    N = B.shape[0]
    if checked:
        native().gemm_frag(ptr(A), A.stride(0), ptr(B), ptr(out), out.stride(0), ptr(residual),
                           residual.stride(0) if residual is not None else 0, ptr(glu_bias), 0, 0, M, N, K, epilogue, b_group, tile, stream(A))
        return out
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16, "bf16 CUDA operands required")
    expect(A.stride(-1) == 1 and B.is_contiguous() and B.shape[1] == K, "A K-contiguous, B a contiguous [N, K] copy")
    expect(_frag_ok(M, N, K, A.stride(0)), "gemm_frag: N % 32, K % 64, 16-B rows")
    expect(epilogue in (EPI_NONE, *GLU8) and b_group in (1, 8), "gemm_frag epilogues: none (+residual) or an 8-row-group GLU")
    n_out = N // 2 if epilogue in GLU8 else N
    if residual is not None:
        expect(epilogue == EPI_NONE and not slices and residual.dtype == torch.bfloat16 and residual.stride(-1) == 1
               and tuple(residual.shape) == (M, N), "residual must be bf16 [M, N]")
    _glu_bias(glu_bias, epilogue, N)
    if slices:
        expect(out is None and epilogue == EPI_NONE and 0 < slices <= K // 64, "slabs: a plain product, K-slices of whole K-tiles")
        slabs = torch.empty((slices, M, N), dtype=torch.float32, device=A.device)
    elif out is None:
        out = torch.empty((M, n_out), dtype=torch.bfloat16, device=A.device)
    expect(out is None or (out.dtype == torch.bfloat16 and out.stride(-1) == 1 and tuple(out.shape) == (M, n_out)), "bad output")
    native().gemm_frag(ptr(A), A.stride(0), ptr(B), ptr(out), out.stride(0) if out is not None else 0, ptr(residual),
                       residual.stride(0) if residual is not None else 0, ptr(glu_bias), ptr(slabs) if slices else 0, int(slices),
                       M, N, K, int(epilogue), int(b_group), int(tile), stream(A))
    return slabs if slices else out


def _frag_takes(A, B, out, residual, glu_bias) -> bool:
    """Whether ``gemm_frag`` takes a projection's operands (the kernels beside it take any alignment)."""
    return (_frag_ok(A.shape[0], B.shape[0], A.shape[1], A.stride(0)) and out.stride(0) % 8 == 0
            and (residual is None or residual.stride(0) % 8 == 0)
            and (ptr(A) | ptr(B) | ptr(out) | ptr(residual) | ptr(glu_bias)) % 16 == 0)


def _run_frag_plan(plan, A, B, out, residual, epilogue, b_group, glu_bias):
    """Runs the parts of a ``frag_plan``: the whole product, or views of the operands (a part starts at a whole tile)."""
    M, N = A.shape[0], B.shape[0]
    m = n = 0
    per = 2 if epilogue in GLU8 else 1  # weight rows per output column
    for part in plan:
        if part is None:
            continue
        kind, rows, cols = part
        a, b, o, r = A, B, out, residual
        if rows < M or cols < N:
            a, b = A[m:m + rows], B[n:n + cols]
            o = out[m:m + rows, n // per:(n + cols) // per]
            r = None if residual is None else residual[m:m + rows, n:n + cols]
        if kind == "frag":
            gemm_frag(a, b, residual=r, epilogue=epilogue, out=o, b_group=b_group, glu_bias=glu_bias, checked=True)
        elif kind != "256":
            gemm_mid(a, b, residual=r, epilogue=epilogue, out=o, variant=192 if kind == "192" else 0, b_group=b_group, glu_bias=glu_bias)
        else:
            _gemm256_into(a, b, o, glu_bias, r, epilogue, True, b_group)
        m, n = (rows, 0) if rows < M else (0, cols)
    return out


def small_tile(M: int, N: int, K: int) -> int:
    """Tile of ``gemm_small`` for a projection with row-major weights, -1: the 128 x 128 / 256 x 256 kernels (the rule,
    with its measurements: csrc/kernels/encoder.hip)."""
    return native().small_tile(M, N, K)


def _gemm_small_takes(A, B, out, bias, residual) -> bool:
    ldr = residual.stride(0) if residual is not None else 0
    return bool(native().gemm_small_ok(A.shape[0], B.shape[0], A.shape[1], A.stride(0), B.stride(0), out.stride(0), ldr)
                and not ((ptr(A) | ptr(B)) % 16 or (ptr(out) | ptr(bias) | ptr(residual)) % 8))


def _gemm_small_into(A, B, out, bias, residual, epilogue, tile: int | None = None) -> bool:
    """Runs a projection on ``gemm_small`` where it is the faster kernel (or on its given tile) and takes the operands; else
    False."""
    M, K = A.shape
    N = B.shape[0]
    if tile is None:
        tile = small_tile(M, N, K) if M and N else -1
        if tile < 0 and native().ring_wins(M, N, K, int(epilogue == EPI_GELU), int(residual is not None)):
            tile = native().RING_TILE
    if tile < 0 or not _gemm_small_takes(A, B, out, bias, residual):
        return False
    native().gemm_small(ptr(A), A.stride(0), ptr(B), B.stride(0), ptr(out), out.stride(0), ptr(bias), ptr(residual),
                        residual.stride(0) if residual is not None else 0, M, N, K, int(epilogue == EPI_GELU), tile, stream(A))
    return True


def gemm_bt(A, B, bias=None, residual=None, epilogue=EPI_NONE, out_f32=False, row_group=None, q_group=None,
            allow=None, out=None, shuffled=False, n=None, b_group: int = 1, glu_bias=None):
    """C = A . B^T (+bias) (+act) (+residual) on MFMA; A [M, K], B [N, K] (K-contiguous rows).

    ``shuffled``: B is a ``shuffle_weights`` copy (the layout the decode GEMM streams, so a model
    keeps ONE copy of every projection) of ``B.shape[0]`` rows, of which the first ``n`` (default:
    all) are the matrix; ``b_group`` 8: a ``shuffle_weights(w, 8)`` copy.  ``glu_bias`` (GLU8 epilogues):
    fp32 [N] = [gate | up], added before the gate's activation and the product."""
    expect(b_group == 1 or (shuffled and b_group == 8), "b_group: 1, or 8 with a shuffled copy")
    if shuffled:
        R = B.shape[0]
        N = R if n is None else int(n)
        expect(R % (16 * b_group) == 0 and B.shape[1] % 32 == 0 and B.is_contiguous() and R >= N,
               "shuffled B: contiguous [R, K] copy, R % (16 b_group) == 0, K % 32 == 0, R >= n")
        if not A.is_cuda:
            Bu = unshuffle_weights(B, b_group)[:N]
            return ref.gemm_bt(A, Bu, bias, residual, epilogue, out_f32, row_group, q_group, allow, glu_bias)
    if not A.is_cuda:
        return ref.gemm_bt(A, B, bias, residual, epilogue, out_f32, row_group, q_group, allow, glu_bias)
    expect(A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16, "bf16 operands required")
    expect(A.stride(-1) == 1 and B.stride(-1) == 1, "operands must be K-contiguous")
    M, K = A.shape
    N = (B.shape[0] if n is None else int(n)) if shuffled else B.shape[0]
    expect(B.shape[1] == K, "inner dims mismatch")
    expect(K % 64 == 0 and N % 4 == 0, "gemm_bt needs K % 64 == 0 and N % 4 == 0")
    expect(A.stride(0) % 8 == 0 and B.stride(0) % 8 == 0, "row strides must be multiples of 8")
    if bias is not None:
        expect_bf16_contig(bias)
        expect(bias.numel() == N, "bias size mismatch")
    n_out = N // 2 if epilogue in (EPI_SWIGLU, *GLU8) else N
    if epilogue == EPI_SWIGLU:
        expect(N % 32 == 0 and not out_f32, "swiglu epilogue needs N % 32 == 0 and bf16 output")
    if epilogue in GLU8:
        expect(N % 32 == 0 and not out_f32 and bias is None and residual is None,
               "swiglu8 epilogue needs N % 32 == 0, bf16 output, no bias / residual")
    _glu_bias(glu_bias, epilogue, N)
    if residual is not None:
        expect(residual.dtype == torch.bfloat16 and residual.stride(-1) == 1, "residual must be bf16 row-major")
        expect(tuple(residual.shape) == (M, n_out), "residual shape mismatch")
    allow_words = 0
    if allow is not None:
        expect(allow.dtype == torch.int32 and allow.is_contiguous() and allow.shape[0] == M, "allow mask shape")
        allow_words = allow.shape[1]
        expect(allow_words * 32 >= N, "allow mask too narrow")
    if row_group is not None:
        _i32(row_group)
        expect(row_group.numel() >= N, "row_group shorter than N")
    if q_group is not None:
        _i32(q_group)
        expect(q_group.numel() >= M, "q_group shorter than M")
    dtype = torch.float32 if out_f32 else torch.bfloat16
    if out is None:
        out = torch.empty((M, n_out), dtype=dtype, device=A.device)
    expect(out.dtype == dtype and out.stride(-1) == 1 and tuple(out.shape) == (M, n_out), "bad output buffer")
    plain = not out_f32 and row_group is None and q_group is None and allow is None
    if plain and shuffled and N == B.shape[0] and bias is None and epilogue in (EPI_NONE, *GLU8) and N % 256 == 0:
        lda = A.stride(0)
        frag = _frag_takes(A, B, out, residual, glu_bias)
        if frag and glu_bias is None and M > 256 and _gemm256_ok(M, N, K, lda):
            tail = corner_plan(M, N, K)[0]
            if tail:
                return _run_corner(tail, A, B, out, residual, epilogue, b_group)
        plan = (frag_plan(M, N, K, glu_bias is None, frag)
                if M >= GEMM_MID_MIN_M and _gemm256_ok(M, N, K, lda) else None)
        if plan is not None and all(q is None or q[0] not in ("mid", "192") or gemm_mid_ok(q[1], q[2], K, lda) for q in plan):
            return _run_frag_plan(plan, A, B, out, residual, epilogue, b_group, glu_bias)
        if use_gemm_mid(M, N, K, A.stride(0)):
            return gemm_mid(A, B, residual=residual, epilogue=epilogue, out=out, b_group=b_group, glu_bias=glu_bias)
    if plain and not shuffled and epilogue in (EPI_NONE, EPI_GELU) and _gemm_small_into(A, B, out, bias, residual, epilogue):
        return out
    if (epilogue in (EPI_NONE, EPI_GELU, EPI_SWIGLU, *GLU8) and plain and (not shuffled or N == B.shape[0])
            and use_gemm256(M, N, K, A.stride(0), B.stride(0))):
        rows = M
        if not shuffled and epilogue in (EPI_NONE, EPI_GELU) and _gemm_small_takes(A, B, out, bias, residual):
            rows = native().gemm256_rows(M, N, K, int(epilogue == EPI_GELU), int(residual is not None))
        _gemm256_into(A[:rows], B, out[:rows], bias if glu_bias is None else glu_bias, None if residual is None else residual[:rows],
                      epilogue, shuffled, b_group)
        if rows < M:
            took = _gemm_small_into(A[rows:], B, out[rows:], bias, None if residual is None else residual[rows:], epilogue, native().RING_TILE)
            expect(took, "gemm_bt: the rows behind the waves")  # (what it takes of all rows it takes of the last)
        return out
    native().gemm_bt(ptr(A), A.stride(0), ptr(B), B.stride(0), ptr(out), out.stride(0),
                     ptr(bias if glu_bias is None else glu_bias), ptr(residual),
                     residual.stride(0) if residual is not None else 0, M, N, K, int(epilogue), int(out_f32),
                     ptr(row_group), ptr(q_group), ptr(allow), allow_words, stream(A),
                     B.shape[0] if shuffled else 0, int(b_group))
    return out


def _glu_bias(glu_bias, epilogue, N: int) -> None:
    if glu_bias is not None:
        expect(epilogue in GLU8 and glu_bias.dtype == torch.float32 and glu_bias.is_contiguous() and glu_bias.numel() == N,
               "glu_bias: fp32 [gate | up] of a GLU8 epilogue")


def _gemm256_into(A, B, out, bias, residual, epilogue, shuffled, b_group=1, tail: int = 0):
    """``tail`` > 0: the last 256 rows' tiles over so many columns of 256 only."""
    M, K = A.shape
    native().gemm256(ptr(A), A.stride(0), ptr(B), B.stride(0), ptr(out), out.stride(0), ptr(bias), ptr(residual),
                     residual.stride(0) if residual is not None else 0, M, B.shape[0], K, int(epilogue), stream(A),
                     int(shuffled), int(b_group), int(tail))
    return out


def gemm256(A, B, bias=None, residual=None, epilogue=EPI_NONE, shuffled=False, b_group: int = 1):
    """The phased 256x256 kernel directly, for any M (``gemm_bt`` takes it from M >= 1024):
    tests and benchmarks.  N % 256 == 0, K % 128 == 0."""
    M, K = A.shape
    N = B.shape[0]
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16, "bf16 CUDA operands required")
    expect(bool(native().gemm256_ok(M, N, K, A.stride(0), B.stride(0))), "gemm256: N % 256, K % 128, 16-B rows")
    expect(not shuffled or (B.is_contiguous() and B.shape[1] == K), "shuffled B must be a contiguous [N, K] copy")
    n_out = N // 2 if epilogue in (EPI_SWIGLU, *GLU8) else N
    out = torch.empty((M, n_out), dtype=torch.bfloat16, device=A.device)
    return _gemm256_into(A, B, out, bias, residual, epilogue, shuffled, b_group)


_MID_WS: dict = {}


def _mid_workspace(device: torch.device, s: int):
    """Partial-tile slabs, ready flags and counts of ``gemm_mid``, one set per (device, stream): two streams
    running the kernel at once must not share them.  Flags and counts are zero at rest (every launch leaves
    them zero); the slabs' last 1024 bytes count the workgroups that ended."""
    key = (device.index, s)
    ws = _MID_WS.get(key)
    if ws is None:
        nat = native()
        slabs = torch.empty((nat.gemm_mid_slab_bytes() // 4,), dtype=torch.float32, device=device)
        slabs[-256:].zero_()
        cnt = torch.zeros((1 << 16,), dtype=torch.int32, device=device)
        ws = _MID_WS[key] = (slabs, cnt)
    return ws


def gemm_mid_ok(M: int, N: int, K: int, lda: int) -> bool:
    """Shapes ``gemm_mid`` serves: N % 256, K % 64, ceil(M / 128) <= 32 (M <= 4096)."""
    return bool(native().gemm_mid_ok(M, N, K, lda)) and -(-M // 128) * (N // 256) <= (1 << 16)


def gemm_mid(A, B, residual=None, epilogue=EPI_NONE, out=None, variant: int = 0, b_group: int = 1, glu_bias=None):
    """C = A . B^T (+ residual) or SwiGLU over 8-row [gate | up] groups, B a ``shuffle_weights`` copy:
    the mid-M kernels (``gemm_mid.hip``: grouped stream-K, 128 x 256 tiles or, by estimates, 256 x 256, in-launch combine)
    for M up to 4096 (mixed serving steps, single prompts).  Bit-reproducible: the split-K partials are
    summed in a fixed order.  ``variant``: 192 the kernel with tiles of so many rows where it takes the sizes; tests, A/B harness:
    32 / 64 the 128-row kernel with that K-step, 256 the 256-row one; + 1000 leaves split tiles uncombined (timing only)."""
    M, K = A.shape
    N = B.shape[0]
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16, "bf16 CUDA operands required")
    expect(A.stride(-1) == 1 and B.is_contiguous() and B.shape[1] == K, "A K-contiguous, B a contiguous [N, K] copy")
    expect(epilogue in (EPI_NONE, *GLU8), "gemm_mid epilogues: none (+residual) or an 8-row-group GLU")
    expect(gemm_mid_ok(M, N, K, A.stride(0)), "gemm_mid: N % 256, K % 64, M <= 4096, 16-B rows")
    expect(b_group in (1, 8), "gemm_mid: b_group 1 or 8")
    n_out = N // 2 if epilogue in GLU8 else N
    if residual is not None:
        expect(epilogue == EPI_NONE and residual.dtype == torch.bfloat16 and residual.stride(-1) == 1
               and tuple(residual.shape) == (M, N), "residual must be bf16 [M, N]")
    _glu_bias(glu_bias, epilogue, N)
    if out is None:
        out = torch.empty((M, n_out), dtype=torch.bfloat16, device=A.device)
    expect(out.dtype == torch.bfloat16 and out.stride(-1) == 1 and tuple(out.shape) == (M, n_out), "bad output")
    s = stream(A)
    slabs, cnt = _mid_workspace(A.device, s)
    native().gemm_mid(ptr(A), A.stride(0), ptr(B), ptr(out), out.stride(0), ptr(residual if glu_bias is None else glu_bias),
                      residual.stride(0) if residual is not None else 0, M, N, K, int(epilogue), ptr(slabs),
                      slabs.numel() * 4, ptr(cnt), cnt.numel(), s, int(variant), int(b_group))
    return out


def _candidate_lists(M: int, cap: int, device, cnt):
    """Candidate scores, rows and counts: padded and zeroed, or (``cnt``: the caller's zeroed counts) only allocated."""
    idx = torch.empty((M, cap), dtype=torch.int32, device=device)
    if cnt is not None:
        expect(cnt.dtype == torch.int32 and cnt.is_contiguous() and cnt.numel() == M, "cnt must be int32 [M]")
        return torch.empty((M, cap), dtype=torch.float32, device=device), idx, cnt
    return (torch.full((M, cap), float("-inf"), dtype=torch.float32, device=device), idx,
            torch.zeros(M, dtype=torch.int32, device=device))


def score_candidates(A, B, thr, cap, row_group=None, q_group=None, cnt=None):
    """Filtered cosine scores of A [M, K] against B [N, K] that are >= thr[m], appended per query
    (no [M, N] score matrix).  -> (cand_val fp32 [M, cap] (-inf padded), cand_idx int32 [M, cap]
    (defined for the first count entries of a row only), count int32 [M]; count > cap means the
    list overflowed).  ``cnt``: zeroed counts of the caller (``rank_value``); cand_val is then
    defined for the counted entries only."""
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16, "bf16 CUDA operands required")
    expect(A.stride(-1) == 1 and B.stride(-1) == 1 and A.stride(0) % 8 == 0 and B.stride(0) % 8 == 0,
           "operands must be K-contiguous with row strides % 8 == 0")
    M, K = A.shape
    N = B.shape[0]
    expect(B.shape[1] == K and K % 64 == 0 and N % 4 == 0, "score_candidates needs K % 64 == 0 and N % 4 == 0")
    expect(thr.dtype == torch.float32 and thr.is_contiguous() and thr.numel() >= M, "thr must be fp32 [M]")
    if row_group is not None:
        _i32(row_group)
        expect(row_group.numel() >= N, "row_group shorter than N")
    if q_group is not None:
        _i32(q_group)
        expect(q_group.numel() >= M, "q_group shorter than M")
    cand_val, cand_idx, cnt = _candidate_lists(M, cap, A.device, cnt)
    native().gemm_score_candidates(ptr(A), A.stride(0), ptr(B), B.stride(0), M, N, K, ptr(row_group), ptr(q_group),
                                   ptr(thr), ptr(cnt), ptr(cand_val), ptr(cand_idx), int(cap), stream(A))
    return cand_val, cand_idx, cnt


def score_candidates_shuffled(A, B_shuf, N, thr, cap, row_group=None, q_group=None, cnt=None):
    """``score_candidates`` over a copy of the rows in the ``shuffle_weights`` layout (``B_shuf``
    [R, K], R >= round_up(N, 128), R % 16 == 0): every 16-row x 32-k fragment is one coalesced 1 KB
    load (K 256, 512, 768 and 1..256 queries, K 1024 and 1..128: the persistent scan of
    index_scan.hip; more (K % 128 == 0): gemm256's candidate epilogue; the weight-streaming kernel's
    candidate epilogue otherwise)."""
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B_shuf.dtype == torch.bfloat16, "bf16 CUDA operands required")
    M, K = A.shape
    expect(shuffled_scan_ok(M, K) and A.stride(-1) == 1 and A.stride(0) % 8 == 0, "queries need K % 128 == 0")
    expect(B_shuf.is_contiguous() and B_shuf.shape[1] == K, "shuffled copy [R, K]")
    expect(B_shuf.shape[0] % 16 == 0 and B_shuf.shape[0] >= -(-N // 128) * 128, "shuffled copy needs round_up(N, 128) rows")
    expect(thr.dtype == torch.float32 and thr.is_contiguous() and thr.numel() >= M, "thr must be fp32 [M]")
    if row_group is not None:
        _i32(row_group)
        expect(row_group.numel() >= N, "row_group shorter than N")
    if q_group is not None:
        _i32(q_group)
        expect(q_group.numel() >= M, "q_group shorter than M")
    cand_val, cand_idx, cnt = _candidate_lists(M, cap, A.device, cnt)
    native().score_candidates_shuf(ptr(A), A.stride(0), ptr(B_shuf), M, int(N), K, ptr(row_group), ptr(q_group),
                                   ptr(thr), ptr(cnt), ptr(cand_val), ptr(cand_idx), int(cap), stream(A),
                                   B_shuf.shape[0])
    return cand_val, cand_idx, cnt


def scores_shuffled(A, B_shuf, N, row_group, q_group=None):
    """fp32 scores [M, N] of A [M, K] against the first N rows of a ``shuffle_weights`` copy (R >= round_up(N, 128)), -inf
    where the groups drop a row: the scan of index_scan.hip where it takes the shape, else ``gemm_bt``'s."""
    _expect_scores(A, B_shuf, N, row_group, q_group)
    if not (scan_scores_ok(A.shape[0], N, A.shape[1]) and A.stride(-1) == 1 and A.stride(0) % 8 == 0 and row_group.data_ptr() % 16 == 0):
        return gemm_bt(A, B_shuf, epilogue=EPI_SCORES, out_f32=True, row_group=row_group, q_group=q_group, shuffled=True, n=N)
    M, K = A.shape
    out = torch.empty((M, N), dtype=torch.float32, device=A.device)
    native().index_scan_scores(ptr(A), A.stride(0), ptr(B_shuf), M, int(N), K, ptr(row_group), ptr(q_group), 0, ptr(out), 0, 0,
                               stream(A))
    return out


def _expect_scores(A, B_shuf, N, row_group, q_group):
    M, K = A.shape
    expect(A.is_cuda and A.dtype == torch.bfloat16 and B_shuf.dtype == torch.bfloat16 and N > 0 and N % 4 == 0, "bf16, N % 4")
    expect(B_shuf.is_contiguous() and B_shuf.shape[1] == K and B_shuf.shape[0] % 16 == 0
           and B_shuf.shape[0] >= -(-N // 128) * 128, "shuffled copy [R, K]")
    _i32(row_group)
    expect(row_group.numel() >= N, "row_group shorter than N")
    if q_group is not None:
        _i32(q_group)
        expect(q_group.numel() >= M, "q_group shorter than M")


def scan_scores_ok(M: int, N: int, K: int) -> bool:
    """Shapes ``scores_and_parts`` serves: the scan's, and scores that one buffer can address."""
    return bool(native().index_scan_takes(M, K)) and 4 * M * N <= 0xffffff00


def scores_and_parts(A, B_shuf, N, row_group, q_group=None, allow=None):
    """(fp32 scores [M, N] as ``scores_shuffled`` gives them, also -inf where the int32 bitmask ``allow`` [M, ceil(N / 32)]
    has no bit; int32 [M, P] ordered bits of the greatest score of every 16 rows, P = round_up(ceil(N / 16), 4) with the
    last ones unwritten): what ``top_hits`` selects from."""
    _expect_scores(A, B_shuf, N, row_group, q_group)
    M, K = A.shape
    expect(scan_scores_ok(M, N, K) and A.stride(-1) == 1 and A.stride(0) % 8 == 0 and row_group.data_ptr() % 16 == 0,
           "scores_and_parts: the scan's shapes, 16-B rows")
    if allow is not None:
        _i32(allow)
        expect(allow.is_contiguous() and allow.shape == (M, (N + 31) // 32), "allow: int32 [M, ceil(N / 32)]")
    out = torch.empty((M, N), dtype=torch.float32, device=A.device)
    parts = torch.empty((M, ((N + 15) // 16 + 3) // 4 * 4), dtype=torch.int32, device=A.device)
    native().index_scan_scores(ptr(A), A.stride(0), ptr(B_shuf), M, int(N), K, ptr(row_group), ptr(q_group), ptr(allow), ptr(out),
                               ptr(parts), parts.shape[1], stream(A))
    return out, parts


def top_hits(scores, parts, k: int, row_ids, row_docs):
    """The k best of every row of ``scores_and_parts`` -> (scores fp32 [rows, k] descending, equal ones in row order, item
    ids, document ids int64; -inf / -1 past the rows that pass the filters), in one launch."""
    rows, n = scores.shape
    expect(scores.is_cuda and scores.dtype == torch.float32 and scores.is_contiguous() and n % 4 == 0
           and 1 <= k <= min(n, 1024), "top_hits: contiguous fp32 [rows, n], n % 4, k <= min(n, 1024)")
    _i32(parts)
    expect(parts.is_contiguous() and parts.shape[0] == rows and parts.shape[1] >= (n + 15) // 16 and parts.shape[1] % 4 == 0,
           "top_hits: the parts of these scores")
    expect(row_ids.dtype == torch.int64 and row_docs.dtype == torch.int64 and row_ids.is_contiguous()
           and row_docs.is_contiguous() and min(row_ids.numel(), row_docs.numel()) >= n, "row ids / documents: int64 [>= n]")
    vals = torch.empty((rows, k), dtype=torch.float32, device=scores.device)
    ids, docs = (torch.empty((rows, k), dtype=torch.int64, device=scores.device) for _ in range(2))
    native().top_hits(ptr(scores), rows, n, ptr(parts), parts.shape[1], int(k), ptr(row_ids), ptr(row_docs), ptr(vals),
                      ptr(ids), ptr(docs), stream(scores))
    return vals, ids, docs


def selected_search(x, vecs, rows: int, row_group, row_ids, row_docs, k: int, groups=None, lists=None, limits=None):
    """``top_hits`` of ``scores_and_parts`` of the unit rows of ``x`` (fp32 [q, K]) over the first ``rows`` rows of ``vecs``, in one
    call.  ``groups``: up to ``HOST_VALUES`` int32 of the host; ``lists``: (ids, offsets, longest, keys, rows) of
    ``allow_bits``, a list a query; ``limits``: int64 of the host, a bound on a row's document id a query."""
    M, K = x.shape
    n = (max(rows, 4) + 3) // 4 * 4
    nat = native()
    expect(x.is_cuda and x.dtype == torch.float32 and vecs.dtype == torch.bfloat16 and vecs.is_contiguous() and vecs.shape[1] == K
           and vecs.shape[0] % 16 == 0 and vecs.shape[0] >= -(-n // 128) * 128, "selected_search: fp32 [q, K] and a shuffled copy [R, K]")
    there, i64 = x.get_device(), torch.int64
    expect(vecs.get_device() == there and row_group.get_device() == there and row_group.dtype == torch.int32 and row_group.is_contiguous()
           and row_ids.get_device() == there and row_ids.dtype == i64 and row_ids.is_contiguous()
           and row_docs.get_device() == there and row_docs.dtype == i64 and row_docs.is_contiguous(),
           "selected_search: contiguous int32 groups, int64 row ids and documents, on the queries' device")
    expect(scan_scores_ok(M, n, K) and 1 <= k <= min(n, 1024) and row_group.data_ptr() % 16 == 0
           and min(row_group.numel(), row_ids.numel(), row_docs.numel()) >= n, "selected_search: the scan's shapes, rows' groups and ids")
    expect(groups is None or (not groups.is_cuda and groups.dtype == torch.int32 and groups.dim() == 1 and groups.is_contiguous()
                              and groups.numel() >= M), "q_group shorter than M")
    ids, offsets, longest, keys, key_rows = lists if lists is not None else (None, None, 0, None, None)
    for t in (ids, offsets, keys, key_rows) if lists is not None else ():
        expect(t.get_device() == there and t.dtype == i64 and t.is_contiguous(), "allow lists: contiguous CUDA int64 tensors")
    expect(lists is None or (offsets.numel() == M + 1 and keys.numel() == key_rows.numel()), "allow lists: one a query")
    expect(limits is None or (not limits.is_cuda and limits.dtype == torch.int64 and limits.is_contiguous() and limits.shape == (M,)),
           "limits: int64 of the host, one a query")
    x = x if x.stride(1) == 1 else x.contiguous()
    n_groups = 0 if groups is None else groups.numel()
    nb = nat.search_space(M, K, n, n_groups, int(lists is not None or limits is not None))
    space = torch.empty(nb, dtype=torch.uint8, device=x.device)
    vals = torch.empty((M, k), dtype=torch.float32, device=x.device)
    out_ids, out_docs = (torch.empty((M, k), dtype=torch.int64, device=x.device) for _ in range(2))
    nat.selected_search(x.data_ptr(), x.stride(0), M, K, vecs.data_ptr(), rows, n, row_group.data_ptr(), row_ids.data_ptr(),
                        row_docs.data_ptr(), ptr(groups), n_groups, int(lists is not None), ptr(ids), ptr(offsets), ptr(keys),
                        ptr(key_rows), 0 if keys is None else keys.numel(), int(longest), ptr(limits), int(k), space.data_ptr(), nb,
                        vals.data_ptr(), out_ids.data_ptr(), out_docs.data_ptr(), stream(x))
    return vals, out_ids, out_docs


def shuffled_scan_ok(M: int, K: int) -> bool:
    """Query counts / widths ``score_candidates_shuffled`` serves."""
    return M >= 1 and K % 128 == 0


def shuffle_rows_into(dst: torch.Tensor, rows: torch.Tensor, vals: torch.Tensor) -> None:
    """Writes ``vals`` [n, K] as rows ``rows`` of ``dst``, a [R, K] tensor in the ``shuffle_weights``
    layout (the incremental form of shuffle_weights, for copies that are updated in place)."""
    R, K = dst.shape
    v5 = dst.view(R // 16, K // 32, 4, 16, 8)
    rows = rows.to(dst.device, torch.long)
    v5[rows // 16, :, :, rows % 16, :] = vals.to(dst.dtype).reshape(-1, K // 32, 4, 8)


def _ref_stream_gemm(x, w, splits=1, epilogue=EPI_NONE, residual=None, norm_eps=0.0, glu_bias=None):
    """CPU semantics of ``stream_gemm`` (row-major ``w``): bf16 [M, N] / SwiGLU / fp32 slabs
    [S, M, N] whose sum is the product (slab 0 holds it, the others are zero).  ``norm_eps`` > 0:
    the product of the RMS-normalised rows of x (gains folded into w) before the epilogue."""
    if norm_eps > 0:
        xf = x.float()
        r = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + norm_eps)
        y = xf @ w.float().t() * r
        if epilogue in (EPI_SWIGLU, *GLU8):
            grp = 16 if epilogue == EPI_SWIGLU else 8
            v = y.view(y.shape[0], -1, 2, grp)
            act = ref.glu_act(v[:, :, 0], ref.epilogue_act(epilogue))
            y = (act * v[:, :, 1]).reshape(y.shape[0], -1)
        if splits > 1:
            return torch.cat([y[None], torch.zeros((splits - 1,) + tuple(y.shape))], 0)
        return y.to(torch.bfloat16)
    y = ref.gemm_bt(x, w, None, None, epilogue, out_f32=splits > 1, glu_bias=glu_bias)
    if splits > 1:
        return torch.cat([y[None], torch.zeros((splits - 1,) + tuple(y.shape), dtype=y.dtype)], 0)
    return y if residual is None else (y.float() + residual.float()).to(torch.bfloat16)


STREAM_KS = 128
STREAM_MAX_M = 256  # decode batches / prefill last-token LM heads up to this many rows stream the weights


def shuffle_weights(w: torch.Tensor, group: int = 1) -> torch.Tensor:
    """[N, K] row-major -> the same values in the fragment layout [N/16][K/32][64 lanes][8]: the
    16 x 32 tile an MFMA A fragment covers is 1 KB contiguous, in lane order (lane l = row l & 15,
    k 8 (l >> 4) .. + 8), so every weight load of the streaming kernel is one fully coalesced 1 KB
    read, and the prefill GEMMs' LDS-DMA copies whole blocks (gemm256 / gemm_bt ``shuffled``).
    ``group`` G > 1: the grouped form [N/(16G)][K/32][G][1 KB] -- the fragments of G consecutive
    16-row blocks adjacent for each 32-deep k chunk, so the decode GEMM's waves (one block each)
    stream neighbouring bytes (profiles/decode_stream_layout_r6.md); the kernels take it with
    ``w_group`` / ``b_group`` = G.  Returned with shape [N, K] (only the memory order changes)."""
    N, K = w.shape
    expect(N % (16 * group) == 0 and K % 32 == 0, "shuffle_weights needs N % (16 group) == 0 and K % 32 == 0")
    f = w.reshape(N // 16, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4)
    if group > 1:
        f = f.reshape(N // (16 * group), group, K // 32, 512).permute(0, 2, 1, 3)
    return f.contiguous().view(N, K)


def unshuffle_weights(w: torch.Tensor, group: int = 1) -> torch.Tensor:
    """Inverse of ``shuffle_weights``."""
    N, K = w.shape
    if group > 1:
        w = w.reshape(N // (16 * group), K // 32, group, 512).permute(0, 2, 1, 3)
    return w.reshape(N // 16, K // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).contiguous().view(N, K)


@functools.lru_cache(maxsize=None)
def stream_tile(cfg: int) -> tuple[int, int, bool]:
    """(weight rows a workgroup or -1, most rows of x, whether the weights are in fragment layout) of a ``stream_gemm``
    configuration."""
    nat = native()
    return nat.stream_gemm_bn(cfg), nat.stream_gemm_max_m(cfg), bool(nat.stream_gemm_shuffled(cfg))


def stream_gemm(x, w, splits=1, epilogue=EPI_NONE, residual=None, out=None, nt=False, cfg=0, norm_eps: float = 0.0,
                slab_dtype=torch.float32, w_group: int = 1, glu_bias=None):
    """Decode GEMM y = x w^T on the warp-specialised streaming kernel (``stream_gemm.hip``): bf16
    [M, N] (optional residual add), SwiGLU [M, N/2] over 16- / 8-row interleaved [gate | up] rows, or
    fp32 K-slice slabs [S, M, N] (their sum is the product; consumers sum them in their prologue or
    ``slab_reduce`` does).  ``cfg`` picks the tile / ring configuration
    (``native().stream_gemm_bn(cfg)`` weight rows per workgroup); ``nt`` streams the weights with
    non-temporal loads.  ``norm_eps`` > 0: x is an un-normalised residual stream and w carries the
    RMSNorm gains in its columns; the kernel scales row m by rsqrt(mean(x[m]^2) + eps) (the
    consumer-side RMSNorm of small decode batches).  ``slab_dtype`` bf16: the split-K slabs are the
    partial sums rounded to bf16 (half the bytes for the producer and its consumer; the rounding the TP
    path's all-reduce input has).  On the CPU ``w`` is row-major."""
    if not x.is_cuda:
        y = _ref_stream_gemm(x, w, splits=splits, epilogue=epilogue, residual=residual, norm_eps=norm_eps, glu_bias=glu_bias)
        return y.to(slab_dtype) if splits > 1 else y
    expect(norm_eps <= 0 or residual is None, "the consumer RMSNorm takes no residual add")
    expect(x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16, "bf16 operands required")
    expect(x.stride(-1) == 1 and w.stride(-1) == 1, "operands must be K-contiguous")
    M, K = x.shape
    N, K_w = w.shape[0], w.shape[1]
    bn, max_m, shuffled = stream_tile(cfg)
    if bn <= 0 or M > max_m:
        raise ValueError(f"stream_gemm cfg {cfg}: bad config or M too large")
    if K_w != K or N % bn or K % (splits * STREAM_KS):
        raise ValueError(f"stream_gemm needs N % {bn} == 0 and K % ({STREAM_KS}*splits) == 0")
    ldx, ldw = x.stride(0), w.stride(0)
    expect(ldx % 8 == 0 and ldw % 8 == 0, "row strides must be multiples of 8")
    if shuffled:
        expect(w.is_contiguous(), "shuffled-layout configurations take a contiguous shuffle_weights() tensor")
    if splits > 1:
        expect(epilogue == EPI_NONE and residual is None, "split-K writes raw slabs")
        expect(slab_dtype in (torch.float32, torch.bfloat16), "slabs are fp32 or bf16")
        if out is None:
            out = torch.empty((splits, M, N), dtype=slab_dtype, device=x.device)
        else:
            expect(out.dtype == slab_dtype and out.is_contiguous() and tuple(out.shape) == (splits, M, N), "bad slabs")
        ldo = N
    else:
        n_out = N // 2 if epilogue in _GLU_ALL else N
        if residual is not None:
            expect(epilogue == EPI_NONE and residual.dtype == torch.bfloat16 and residual.stride(-1) == 1
                   and tuple(residual.shape) == (M, N), "residual must be bf16 [M, N]")
        _glu_bias(glu_bias, epilogue, N)
        if epilogue == EPI_SWIGLU:
            expect(bn % 32 == 0, f"stream_gemm cfg {cfg}: EPI_SWIGLU needs 32-row tiles (use EPI_SWIGLU8)")
        if out is None:
            out = torch.empty((M, n_out), dtype=torch.bfloat16, device=x.device)
        else:
            expect(out.dtype == torch.bfloat16 and out.stride(-1) == 1 and tuple(out.shape) == (M, n_out), "bad output")
        ldo = out.stride(0)
    native().stream_gemm(x.data_ptr(), ldx, w.data_ptr(), ldw, out.data_ptr(), ldo,
                         ptr(residual if glu_bias is None else glu_bias),
                         residual.stride(0) if residual is not None else 0, M, N, K, splits, int(epilogue), stream(x),
                         int(bool(nt)), int(cfg), float(norm_eps), int(splits > 1 and out.dtype == torch.bfloat16),
                         int(w_group))
    return out


def norm_stream_ok(M: int, N: int, K: int, splits: int, bn: int) -> bool:
    """Shapes ``norm_stream`` serves: up to 4 rows, K of 256..4096, slices of up to 32,768 elements."""
    return bool(native().norm_stream_ok(M, N, K, splits, bn))


def norm_stream(x, gain, eps, residual, w, splits=1, bn=64, epilogue=EPI_NONE, slab_dtype=torch.float32, w_group: int = 1):
    """``stream_gemm(rmsnorm(x, gain, eps, residual)[0], w, ...)`` of a few decode rows in one launch (norm_stream.hip) ->
    (product, new residual or None).  x: bf16 rows or split-K slabs [S, M, K]; w: a ``shuffle_weights`` copy; ``bn``: weight
    rows a workgroup, 64 or 128."""
    slabs = x.dim() == 3
    S, (M, K), N = x.shape[0] if slabs else 1, x.shape[-2:], w.shape[0]
    expect(x.is_cuda and x.is_contiguous() and x.dtype in ((torch.float32, torch.bfloat16) if slabs else (torch.bfloat16,)),
           "norm_stream: contiguous bf16 rows or slabs")
    expect_bf16_contig(gain, residual, w)
    same_device(x, gain, residual, w)
    expect(gain.numel() == K and w.shape[1] == K and norm_stream_ok(M, N, K, splits, bn), "norm_stream: shapes")
    expect(residual is None or tuple(residual.shape) == (M, K), "residual shape mismatch")
    expect(epilogue == EPI_NONE or (epilogue == EPI_SWIGLU8 and splits == 1), "norm_stream: slabs, rows or SwiGLU of 8-row groups")
    expect(N % (16 * w_group) == 0 and slab_dtype in (torch.float32, torch.bfloat16), "whole groups; fp32 or bf16 slabs")
    new = None if residual is None else torch.empty_like(residual)
    if splits > 1:
        out = torch.empty((splits, M, N), dtype=slab_dtype, device=x.device)
    else:
        out = torch.empty((M, N // 2 if epilogue else N), dtype=torch.bfloat16, device=x.device)
    native().norm_stream(ptr(x), S, int(x.dtype == torch.float32), ptr(residual), ptr(gain), ptr(new), float(eps), ptr(w), ptr(out),
                         out.shape[-1], M, N, K, splits, int(slab_dtype == torch.float32), int(epilogue != EPI_NONE), int(w_group),
                         int(bn), stream(x))
    return out, new


def norm_rows(x, gain, eps, w, splits=1, bn=64, epilogue=EPI_NONE, slab_dtype=torch.float32, w_group: int = 1):
    """``norm_stream`` of up to 8 complete rows (bf16 [M, K], no slabs, no residual) -> product."""
    (M, K), N = x.shape, w.shape[0]
    expect(x.is_cuda, "norm_rows: rows on the GPU")
    expect_bf16_contig(x, gain, w)
    same_device(x, gain, w)
    expect(gain.numel() == K and w.shape[1] == K and native().norm_rows_ok(M, N, K, splits, bn), "norm_rows: shapes")
    expect(epilogue == EPI_NONE or (epilogue == EPI_SWIGLU8 and splits == 1), "norm_rows: slabs, rows or SwiGLU of 8-row groups")
    expect(N % (16 * w_group) == 0 and slab_dtype in (torch.float32, torch.bfloat16), "whole groups; fp32 or bf16 slabs")
    if splits > 1:
        out = torch.empty((splits, M, N), dtype=slab_dtype, device=x.device)
    else:
        out = torch.empty((M, N // 2 if epilogue else N), dtype=torch.bfloat16, device=x.device)
    native().norm_rows(ptr(x), ptr(gain), float(eps), ptr(w), ptr(out), out.shape[-1], M, N, K, splits, int(slab_dtype == torch.float32),
                       int(epilogue != EPI_NONE), int(w_group), int(bn), stream(x))
    return out


def rows_stream(x, w, residual, w_group: int = 1, tile: int = -1):
    """x w^T (rounded to bf16) + residual of up to 8 decode rows, w a ``shuffle_weights`` copy (rows_stream.hip).  ``tile`` (tests):
    that form of the kernel."""
    (M, K), N = x.shape, w.shape[0]
    expect(x.is_cuda and x.dtype == torch.bfloat16 and x.stride(1) == 1, "rows_stream: bf16 rows on the GPU")
    expect_bf16_contig(w, residual)
    same_device(x, w, residual)
    expect(w.shape[1] == K and tuple(residual.shape) == (M, N), "rows_stream: shapes")
    expect(native().rows_stream_ok(M, N, K, x.stride(0), w_group), "rows_stream: up to 8 rows, whole groups, K % 64")
    out = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
    native().rows_stream(ptr(x), x.stride(0), ptr(w), ptr(residual), ptr(out), M, N, K, int(w_group), stream(x), int(tile))
    return out


def slab_reduce(slabs, residual=None, out=None):
    """fp32 / bf16 slabs [S, M, N] -> bf16 [M, N] (fp32 sum rounded to bf16, then + residual)."""
    if not slabs.is_cuda:
        y = slabs.float().sum(0).to(torch.bfloat16)
        return y if residual is None else (y.float() + residual.float()).to(torch.bfloat16)
    S, M, N = slabs.shape
    expect(slabs.dtype in (torch.float32, torch.bfloat16) and slabs.is_contiguous() and N % 8 == 0, "bad slabs")
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=slabs.device)
    if residual is not None:
        expect(residual.dtype == torch.bfloat16 and tuple(residual.shape) == (M, N) and residual.stride(-1) == 1,
               "residual must be bf16 [M, N]")
    native().slab_reduce(ptr(out), out.stride(0), ptr(slabs), S, M, N, ptr(residual),
                         residual.stride(0) if residual is not None else 0, stream(slabs),
                         int(slabs.dtype == torch.bfloat16))
    return out


def interleave_gate_up(w_gate: torch.Tensor, w_up: torch.Tensor, group: int = 16) -> torch.Tensor:
    """[F, H] gate and up weights -> [2F, H] interleaved in ``group``-row groups [g | u | g | u ...]
    (16: the layout the SWIGLU epilogue of gemm_bt / gemm256 consumes; 8: EPI_SWIGLU8)."""
    Fd, H = w_gate.shape
    assert Fd % group == 0
    g = w_gate.reshape(Fd // group, group, H)
    u = w_up.reshape(Fd // group, group, H)
    return torch.stack([g, u], dim=1).reshape(2 * Fd, H).contiguous()


def regroup_gate_up(w: torch.Tensor, src: int = 16, dst: int = 8) -> torch.Tensor:
    """Re-interleave [2F, H] gate|up weights from ``src``-row to ``dst``-row groups."""
    n2, H = w.shape
    v = w.reshape(n2 // (2 * src), 2, src, H)
    gate, up = v[:, 0].reshape(n2 // 2, H), v[:, 1].reshape(n2 // 2, H)
    return interleave_gate_up(gate, up, dst)


# ----------------------------------------------------------------------------------------------
# selection


SAMPLE_FAST_MAX_K = 64
_CHUNK = 256 * 32


def sample_workspace(rows: int, vocab: int, device) -> torch.Tensor:
    ncand = -(-vocab // _CHUNK) * SAMPLE_FAST_MAX_K
    return torch.empty((rows * ncand * 8,), dtype=torch.uint8, device=device)


def sample_tokens(logits, temperature, top_k, top_p, seed: int, counters, generator=None, out=None,
                  fast: bool | None = None, workspace: torch.Tensor | None = None):
    """temperature / top_k (int32) / top_p per row; counters int64 per row (advanced in-kernel).

    ``fast`` (every row has 0 < top_k <= 64, the reference's 50 included) selects the two-stage kernel:
    per-chunk register-resident top-64 over many workgroups, then a per-row merge + top-p + sample."""
    if not logits.is_cuda:
        return ref.sample_hf(logits, temperature, top_k, top_p, generator)
    rows, vocab = logits.shape
    expect(logits.stride(-1) == 1, "logits rows must be contiguous")
    expect(logits.dtype in (torch.float32, torch.bfloat16), "logits must be fp32 or bf16")
    expect(temperature.dtype == torch.float32 and temperature.numel() >= rows, "temperature")
    expect(top_p.dtype == torch.float32 and top_p.numel() >= rows, "top_p")
    _i32(top_k)
    expect(counters.dtype == torch.int64 and counters.numel() >= rows, "counters")
    out = torch.empty((rows,), dtype=torch.int32, device=logits.device) if out is None else out
    if fast is None:
        fast = False
    ncand = -(-vocab // _CHUNK) * SAMPLE_FAST_MAX_K
    if fast and ncand <= 1024:
        ws = workspace if workspace is not None else sample_workspace(rows, vocab, logits.device)
        expect(ws.numel() >= rows * ncand * 8, "sampling workspace too small")
        native().sample_tokens_2stage(ptr(logits), int(logits.dtype == torch.float32), logits.stride(0), rows, vocab,
                                      ptr(temperature), ptr(top_k), ptr(top_p), int(seed) & ((1 << 64) - 1),
                                      ptr(counters), ptr(out), ptr(ws), ws.numel(), stream(logits))
    else:
        native().sample_tokens(ptr(logits), int(logits.dtype == torch.float32), logits.stride(0), rows, vocab,
                               ptr(temperature), ptr(top_k), ptr(top_p), int(seed) & ((1 << 64) - 1), ptr(counters),
                               ptr(out), 0, stream(logits))
    return out


def mask_logits(logits, mask, row_flags, vocab: int | None = None, word_offset: int = 0):
    """In place: logits[r, t] = -inf where bit t of ``mask[r]`` (int32 words, bit t % 32 of word
    t // 32) is clear, for the rows whose ``row_flags[r]`` (int32) is non-zero (JSON-constrained
    decoding).  Vocab-parallel slices: the first ``vocab`` columns of ``logits`` are tokens
    32 * ``word_offset`` ... (mask words ``word_offset`` ...).  Returns ``logits``."""
    rows = logits.shape[0]
    vocab = logits.shape[1] if vocab is None else int(vocab)
    words = -(-vocab // 32)
    expect(mask.dtype == torch.int32 and mask.is_contiguous() and mask.shape[0] >= rows
           and mask.shape[1] >= word_offset + words, "mask: int32 [rows, >= ceil(vocab / 32) words past the offset]")
    if not logits.is_cuda:
        m = mask[:rows, word_offset:word_offset + words]
        bits = (m.view(torch.int32).unsqueeze(-1) >> torch.arange(32, dtype=torch.int32)) & 1
        allow = bits.reshape(rows, -1)[:, :vocab].bool() | (row_flags[:rows] == 0).unsqueeze(1)
        logits[:, :vocab].masked_fill_(~allow, float("-inf"))
        return logits
    expect(logits.stride(-1) == 1 and logits.dtype in (torch.float32, torch.bfloat16), "logits: fp32/bf16 rows")
    _i32(row_flags)
    native().mask_logits(ptr(logits), int(logits.dtype == torch.float32), logits.stride(0), rows, vocab,
                         ptr(mask) + 4 * int(word_offset), words, ptr(row_flags), stream(logits), mask.stride(0))
    return logits


def sample_candidates(logits, vocab: int, index_base: int = 0, out=None):
    """Stage 1 of vocab-parallel sampling: each 8192-token chunk's top-64 of the first ``vocab``
    columns of ``logits`` as (order-preserving uint32 key, token id + ``index_base``) -> int32
    [2, rows, ncand] (keys, then ids).  The TP ranks all-gather these and ``sample_merge`` draws
    from the union (GPU only)."""
    expect(logits.is_cuda and logits.stride(-1) == 1 and logits.dtype in (torch.float32, torch.bfloat16),
           "logits: CUDA fp32/bf16 rows")
    rows = logits.shape[0]
    ncand = sample_candidates_per_row(vocab)
    if out is None:
        out = torch.empty((2, rows, ncand), dtype=torch.int32, device=logits.device)
    # (a row slice of a larger [2, R, ncand] buffer is fine: each half is rows x ncand contiguous)
    expect(out.dtype == torch.int32 and tuple(out.shape) == (2, rows, ncand) and out.stride(2) == 1
           and out.stride(1) == ncand, "candidates: int32 [2, rows, ncand] with contiguous halves")
    native().sample_candidates(ptr(logits), int(logits.dtype == torch.float32), logits.stride(0), rows, int(vocab),
                               int(index_base), ptr(out[0]), ptr(out[1]), ncand, stream(logits))
    return out


def sample_candidates_per_row(vocab: int) -> int:
    return -(-int(vocab) // _CHUNK) * SAMPLE_FAST_MAX_K


def sample_merge(cands, temperature, top_k, top_p, seed: int, counters, vocab: int, out=None):
    """Stage 2 of vocab-parallel sampling: ``cands`` int32 [2, rows, n] (every rank's
    ``sample_candidates`` side by side along n, n <= 1024) -> sorted top-k -> HF top-p ->
    multinomial with the per-row counter RNG (advanced in-kernel): the replicated head's draw."""
    two, rows, n = cands.shape
    expect(two == 2 and n <= 1024 and cands.dtype == torch.int32 and cands.is_contiguous(),
           "candidates: contiguous int32 [2, rows, <= 1024]")
    out = torch.empty((rows,), dtype=torch.int32, device=cands.device) if out is None else out
    _i32(top_k)
    native().sample_merge(ptr(cands[0]), ptr(cands[1]), n, rows, int(vocab), ptr(temperature), ptr(top_k), ptr(top_p),
                          int(seed) & ((1 << 64) - 1), ptr(counters), ptr(out), stream(cands))
    return out


def topk_rows(scores, k, index_base=0, want_global=False):
    """Exact per-row top-k of fp32 scores, sorted descending.  Returns (values, idx int32) or, with
    ``want_global``, (values, idx + index_base as int64).  Long rows use the two-stage kernel."""
    rows, n = scores.shape
    expect(1 <= k <= min(n, 1024), "1 <= k <= min(n, 1024)")
    if rows == 0:  # e.g. a rank with no queries in a sharded search (an empty view's strides are arbitrary)
        return (torch.empty((0, k), dtype=torch.float32, device=scores.device),
                torch.empty((0, k), dtype=torch.int64 if want_global else torch.int32, device=scores.device))
    if not scores.is_cuda:
        v, i = ref.topk_rows(scores, k)
        return (v, i.long() + index_base) if want_global else (v, i)
    expect(scores.dtype == torch.float32 and scores.stride(-1) == 1, "scores must be fp32 with contiguous rows")
    vals = torch.empty((rows, k), dtype=torch.float32, device=scores.device)
    if want_global:
        idx = torch.empty((rows, k), dtype=torch.int64, device=scores.device)
        i32, i64 = 0, ptr(idx)
    else:
        idx = torch.empty((rows, k), dtype=torch.int32, device=scores.device)
        i32, i64 = ptr(idx), 0
    if n >= 4 * _CHUNK:
        kc = -(-k // 64) * 64
        ncand = -(-n // _CHUNK) * kc
        ws = torch.empty((rows * ncand * 8,), dtype=torch.uint8, device=scores.device)
        native().topk_rows_2stage(ptr(scores), scores.stride(0), rows, n, k, ptr(vals), i32, int(index_base), i64,
                                  ptr(ws), ws.numel(), stream(scores))
    else:
        native().topk_rows(ptr(scores), scores.stride(0), rows, n, k, ptr(vals), i32, int(index_base), i64,
                           stream(scores))
    return vals, idx


def unit_rows(x, dtype=torch.bfloat16):
    """x / max(|x|, 1e-12) of every row, fp32 [rows, cols] -> bf16 (``F.normalize`` and the rounding in one launch)."""
    if not x.is_cuda or dtype != torch.bfloat16:
        return F.normalize(x, dim=-1).to(dtype)
    expect(x.dtype == torch.float32 and x.dim() == 2, "unit_rows: fp32 [rows, cols]")
    x = x if x.stride(1) == 1 else x.contiguous()
    out = torch.empty(x.shape, dtype=dtype, device=x.device)
    native().unit_rows(ptr(x), x.stride(0), ptr(out), x.shape[0], x.shape[1], stream(x))
    return out


def unit_queries(x, groups=None, clear=None):
    """``unit_rows`` of a search's queries on the GPU and what else it begins with, in one launch: ``groups``, int32 of the host and
    at most ``HOST_VALUES``, on the device (-> second result, else None); ``clear``, a contiguous int32 tensor, zeroed."""
    expect(x.is_cuda and x.dtype == torch.float32 and x.dim() == 2, "unit_rows: fp32 [rows, cols]")
    x = x if x.stride(1) == 1 else x.contiguous()
    out = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    n, there = 0, None
    if groups is not None:
        n = groups.numel()
        expect(not groups.is_cuda and groups.dtype == torch.int32 and groups.dim() == 1 and groups.is_contiguous()
               and n <= native().HOST_VALUES and x.shape[0], "unit_queries: a few int32 groups of the host, for queries")
        there = torch.empty(n, dtype=torch.int32, device=x.device)
    if clear is not None:
        expect(clear.device == x.device and clear.dtype == torch.int32 and clear.is_contiguous() and x.shape[0], "unit_queries: int32 words")
    native().unit_rows(ptr(x), x.stride(0), ptr(out), x.shape[0], x.shape[1], stream(x), ptr(groups), n, ptr(there), ptr(clear),
                       0 if clear is None else clear.numel())
    return out, there


RANK_MAX = 64  # largest rank of ``rank_value``


def rank_value(scores, r: int, slack: float = 0.0):
    """(r-th largest score of every row of fp32 [rows, n] less ``slack``, -inf when r > n; zeroed int32 [rows] for the counts of the
    scan that takes the value as its threshold)."""
    rows, n = scores.shape
    expect(scores.is_cuda and scores.dtype == torch.float32 and scores.stride(1) == 1, "scores: CUDA fp32 rows")
    expect(n > 0 and 1 <= r <= RANK_MAX, f"rank_value: 1 <= r <= {RANK_MAX}, n > 0")
    thr = torch.empty(rows, dtype=torch.float32, device=scores.device)
    cnt = torch.empty(rows, dtype=torch.int32, device=scores.device)
    native().rank_value(ptr(scores), scores.stride(0), rows, n, int(r), float(slack), ptr(thr), ptr(cnt), stream(scores))
    return thr, cnt


def rank_hits(cand_val, cand_idx, cnt, thr, k: int, row_ids, row_docs):
    """The k best of every row's candidate list (``score_candidates`` with threshold ``thr``) -> (scores fp32 [rows, k]
    descending, item ids, document ids int64 (-inf / -1 past the last), status int32 [rows]).  A non-zero status marks
    a row whose list overflowed or holds fewer than k entries although its threshold cut rows off; its outputs are
    undefined."""
    rows, cap = cand_val.shape
    expect(1 <= k <= 1024 and cand_idx.shape == cand_val.shape and cnt.numel() >= rows and thr.numel() >= rows
           and cand_val.is_contiguous() and cand_idx.is_contiguous(), "rank_hits: lists [rows, cap], k <= 1024")
    expect(row_ids.dtype == torch.int64 and row_docs.dtype == torch.int64 and row_ids.is_contiguous()
           and row_docs.is_contiguous(), "row ids / documents: int64")
    dev = cand_val.device
    vals = torch.empty((rows, k), dtype=torch.float32, device=dev)
    ids, docs = (torch.empty((rows, k), dtype=torch.int64, device=dev) for _ in range(2))
    status = torch.empty(rows, dtype=torch.int32, device=dev)
    native().rank_hits(ptr(cand_val), ptr(cand_idx), ptr(cnt), ptr(thr), cap, rows, int(k), ptr(row_ids), ptr(row_docs),
                       ptr(vals), ptr(ids), ptr(docs), ptr(status), stream(cand_val))
    return vals, ids, docs, status


def hit_ids(vals, rows, row_ids, row_docs):
    """(item ids, document ids) int64 of ranked rows; -1 where the score is infinite (no row left)."""
    if not vals.is_cuda:
        at, dead = rows.long(), torch.isinf(vals)
        return row_ids[at].masked_fill(dead, -1), row_docs[at].masked_fill(dead, -1)
    expect(rows.dtype == torch.int32 and rows.is_contiguous() and vals.is_contiguous() and rows.shape == vals.shape,
           "hit_ids: contiguous scores and int32 rows")
    expect(row_ids.dtype == torch.int64 and row_docs.dtype == torch.int64 and row_ids.is_contiguous()
           and row_docs.is_contiguous() and row_ids.numel() == row_docs.numel(), "row ids / documents: int64")
    ids, docs = (torch.empty(rows.shape, dtype=torch.int64, device=vals.device) for _ in range(2))
    native().hit_ids(ptr(vals), ptr(rows), ptr(row_ids), ptr(row_docs), ptr(ids), ptr(docs), rows.numel(),
                     row_ids.numel(), stream(vals))
    return ids, docs


def allow_bits(ids, offsets, longest: int, keys, rows, words: int, mask=None):
    """int32 bitmask [q, words] of the rows whose item id is in list q of ``ids`` (int64, list q = ids[offsets[q] :
    offsets[q + 1]], none longer than ``longest``); ``keys`` sorted int64 ids of the live rows, ``rows`` int64 their rows.
    ``mask``: one of zeros, whose bits are set."""
    for t in (ids, offsets, keys, rows):
        expect(t.is_cuda and t.dtype == torch.int64 and t.is_contiguous(), "allow_bits: contiguous CUDA int64 tensors")
    q = offsets.numel() - 1
    expect(q >= 1 and keys.numel() == rows.numel(), "allow_bits: offsets of every list, one row per key")
    if mask is None:
        mask = torch.zeros((q, words), dtype=torch.int32, device=ids.device)
    expect(mask.dtype == torch.int32 and tuple(mask.shape) == (q, words) and mask.is_contiguous() and mask.is_cuda, "mask shape")
    native().allow_bits(ptr(ids), ptr(offsets), ptr(keys), ptr(rows), keys.numel(), ptr(mask), int(words), q, int(longest),
                        stream(ids))
    return mask


def doc_lt_bits(docs, limits, mask=None):
    """int32 bitmask [q, ceil(n / 32)] of the rows with docs[r] < limits[q] (int64, on the device, or up to ``HOST_VALUES`` of
    the host); ``mask``: intersected in place."""
    n, q = docs.numel(), limits.numel()
    expect(docs.is_cuda and docs.dtype == torch.int64 and limits.dtype == torch.int64 and docs.is_contiguous()
           and limits.is_contiguous() and (limits.is_cuda or q <= native().HOST_VALUES), "doc_lt_bits: contiguous int64 tensors")
    words = (n + 31) // 32
    out = torch.empty((q, words), dtype=torch.int32, device=docs.device) if mask is None else mask
    expect(out.dtype == torch.int32 and tuple(out.shape) == (q, words) and out.is_contiguous(), "mask shape")
    native().doc_lt_bits(ptr(docs), ptr(limits), n, ptr(out), words, q, int(mask is not None), stream(docs), int(not limits.is_cuda))
    return out


def gather_shuffled_rows(src, rows):
    """Row-major bf16 copy of the given rows (int64, inside [0, R)) of ``src``, a [R, K] ``shuffle_weights`` copy."""
    expect(src.is_cuda and src.dtype == torch.bfloat16 and src.is_contiguous() and src.shape[0] % 16 == 0
           and src.shape[1] % 32 == 0, "gather_shuffled_rows: a [16 n, 32 m] shuffled bf16 copy")
    expect(rows.is_cuda and rows.dtype == torch.int64 and rows.is_contiguous(), "rows: contiguous CUDA int64")
    out = torch.empty((rows.numel(), src.shape[1]), dtype=src.dtype, device=src.device)
    native().gather_rows(ptr(src), ptr(rows), ptr(out), rows.numel(), src.shape[1], stream(src))
    return out


def linear(x, w, b=None, residual=None, act=None):
    """y = x W^T (+b) (+act) (+residual) on the native MFMA GEMMs (``gemm_bt``: the phased 256x256
    kernel for large token counts, the 128x128 kernel otherwise), epilogues fused.

    Widths the kernels do not tile (K % 64, N % 4) are zero-padded to the next native shape (zero
    k-columns add nothing to a dot product; padded output columns are sliced off), so every GPU
    call runs the native kernel -- there is no torch fallback (``ops/_lib.py`` dispatch rule)."""
    epi = {None: EPI_NONE, "gelu": EPI_GELU, "swiglu": EPI_SWIGLU}[act]
    if not x.is_cuda:
        return ref.gemm_bt(x, w, b, residual, epi)
    K, N = x.shape[-1], w.shape[0]
    expect(epi != EPI_SWIGLU or N % 32 == 0, "swiglu linear needs 16-row [gate | up] groups (N % 32 == 0)")
    x2 = x.reshape(-1, K)
    r2 = residual.reshape(x2.shape[0], -1) if residual is not None else None
    pk, pn = (-K) % 64, (-N) % 4
    if pk or pn:
        x2 = F.pad(x2, (0, pk)) if pk else x2
        w = F.pad(w, (0, pk, 0, pn))
        b = F.pad(b, (0, pn)) if (b is not None and pn) else b
        r2 = F.pad(r2, (0, pn)) if (r2 is not None and pn) else r2
    y = gemm_bt(x2, w, b, r2, epi)
    if pn:
        y = y[:, :N].contiguous()
    return y.view(*x.shape[:-1], y.shape[-1])
