"""Verify-attention and KV-store operators with the reference's signatures.

Drop-in for ``paged_attention_verify`` and ``store_kvcache`` of
src/myvllm/layers/attention.py (:615-668 and :71-112) and for the verify
branch of ``Attention.forward`` (:689-731).  Both operators launch the
gfx950 kernels of libnaivspec.so on torch's current stream; there is no
PyTorch fallback.
"""

from __future__ import annotations

import ctypes

import torch
import torch.nn as nn

from naivllm_amd import _lib
from naivllm_amd.utils.context import get_context

_INDEX_DTYPES = {
    "block_tables": torch.int32,
    "context_lens": torch.int64,
    "cu_seqlens_q": torch.int32,
    "positions": torch.int64,
    "slot_mapping": torch.int64,
}


def _as(t: torch.Tensor, name: str) -> torch.Tensor:
    want = _INDEX_DTYPES[name]
    if t.dtype != want:
        t = t.to(want)
    return t if t.is_contiguous() else t.contiguous()


def _check_cache(cache: torch.Tensor, name: str) -> tuple[int, int, int, int]:
    if cache.dim() != 4:
        raise ValueError(f"{name} must be (num_blocks, block_size, num_kv_heads, head_dim), got {tuple(cache.shape)}")
    if not cache.is_contiguous():
        raise ValueError(f"{name} must be contiguous")
    return tuple(cache.shape)


def verify_attention_workspace_bytes(batch_size: int, num_heads: int, num_kv_heads: int, head_dim: int,
                                     block_size: int, max_num_blocks: int, max_q_len: int,
                                     dtype: torch.dtype, kv_split_tokens: int = 0) -> int:
    return int(_lib.lib().nsv_verify_attention_workspace_size(
        batch_size, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks, max_q_len,
        _lib.dtype_code(dtype), kv_split_tokens))


ATTN_KERNELS = {0: "d-sliced", 1: "key-split", 2: "fp32"}


def verify_attention_plan(batch_size: int, num_heads: int, num_kv_heads: int, head_dim: int, block_size: int,
                          max_num_blocks: int, max_q_len: int, dtype: torch.dtype, kv_split_tokens: int = 0,
                          cus: int = 0) -> tuple[str, int]:
    """(kernel, most key splits of a sequence) that paged_attention_verify runs
    for this shape on a device with ``cus`` compute units (0: the current
    one); a context shorter than the table may be cut into fewer."""
    kind, splits = ctypes.c_int(), ctypes.c_int()
    rc = _lib.lib().nsv_verify_attention_plan(batch_size, num_heads, num_kv_heads, head_dim, block_size,
                                             max_num_blocks, max_q_len, _lib.dtype_code(dtype), kv_split_tokens,
                                             cus, ctypes.addressof(kind), ctypes.addressof(splits))
    _lib.check(rc, "verify_attention_plan")
    return ATTN_KERNELS[kind.value], splits.value


def paged_attention_verify(
    query: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    cu_seqlens_q: torch.Tensor,
    positions: torch.Tensor,
    scale: float,
    num_heads: int,
    num_kv_heads: int,
    head_dim: int,
    block_size: int,
    block_m: int,
    *,
    max_q_len: int | None = None,
    kv_split_tokens: int = 0,
    out: torch.Tensor | None = None,
    allocation_free: bool = False,
    tile_references: bool = False,
) -> torch.Tensor:
    """Verify a chunk of drafted tokens against the paged KV cache.

    Same arguments and result as the reference (layers/attention.py:615-668):
      query (T, H, D); k_cache/v_cache (num_blocks, block_size, Hkv, D);
      block_tables (B, max_num_blocks), -1 padded; context_lens (B,);
      cu_seqlens_q (B+1,); positions (T,), -1 marks an inert pad row;
      block_m >= every per-sequence query length.
    Returns (T, H, D) in query's dtype.  Keyword-only extras: ``max_q_len``
    (a tighter bound than block_m: fewer padded MFMA rows and partials),
    ``kv_split_tokens`` (keys per workgroup split, 0 = automatic), ``out``
    (a preallocated result) and ``allocation_free`` (run through
    nsv_verify_attention_noalloc: the library's fixed per-device scratch
    instead of a workspace, ``out`` required, index tensors already int32 /
    int64 and contiguous, so the call allocates nothing), ``tile_references``
    (an exponent reference per tile of keys, nsv_verify_attention_tile_refs;
    not with allocation_free).  Rows at position
    -1 come back as zeros (the reference leaves them meaningless; nothing
    reads them).
    """
    if query.dim() != 3 or query.shape[1] != num_heads or query.shape[2] != head_dim:
        raise ValueError(f"query must be (T, {num_heads}, {head_dim}), got {tuple(query.shape)}")
    nb, bs, hkv, d = _check_cache(k_cache, "k_cache")
    if tuple(v_cache.shape) != (nb, bs, hkv, d) or not v_cache.is_contiguous():
        raise ValueError("k_cache and v_cache must have the same contiguous shape")
    if bs != block_size or hkv != num_kv_heads or d != head_dim:
        raise ValueError("cache shape disagrees with block_size / num_kv_heads / head_dim")
    if query.dtype != k_cache.dtype or v_cache.dtype != k_cache.dtype:
        raise ValueError("query and caches must share one dtype")
    if not query.is_cuda:
        raise ValueError("paged_attention_verify runs on the GPU; query is on the CPU")
    query = query.contiguous()
    block_tables = _as(block_tables, "block_tables")
    context_lens = _as(context_lens, "context_lens")
    cu_seqlens_q = _as(cu_seqlens_q, "cu_seqlens_q")
    positions = _as(positions, "positions")
    batch_size, max_num_blocks = block_tables.shape
    qlen_bound = int(max_q_len if max_q_len is not None else block_m)
    code = _lib.dtype_code(query.dtype)
    h = _lib.lib()
    if out is not None and (tuple(out.shape) != tuple(query.shape) or out.dtype != query.dtype
                            or out.device != query.device or not out.is_contiguous()):
        raise ValueError(f"out must be a contiguous {query.dtype} tensor of shape {tuple(query.shape)} on "
                         f"{query.device}")
    if allocation_free:
        if out is None:
            raise ValueError("allocation_free=True needs a preallocated out")
        if tile_references:
            raise ValueError("allocation_free=True takes no tile_references")
        rc = h.nsv_verify_attention_noalloc(
            out.data_ptr(), query.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), block_tables.data_ptr(),
            context_lens.data_ptr(), cu_seqlens_q.data_ptr(), positions.data_ptr(), float(scale), batch_size,
            query.shape[0], num_heads, num_kv_heads, head_dim, block_size, max_num_blocks, qlen_bound, code,
            kv_split_tokens, _lib.stream_ptr(query.device))
        _lib.check(rc, "paged_attention_verify (allocation-free)")
        return out
    if out is None:
        out = torch.empty_like(query)
    ws_bytes = int(h.nsv_verify_attention_workspace_size(
        batch_size, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks, qlen_bound, code,
        kv_split_tokens))
    stream = _lib.stream_ptr(query.device)
    name = "verify_attention"
    if tile_references and not torch.cuda.is_current_stream_capturing():
        # (prefill steps may run beside another stream's rounds: scratch of
        # their own per stream, of which torch has a fixed pool)
        name = f"verify_attention on stream {stream}"
    ws = _lib.workspace(query.device, ws_bytes, name)
    rc = (h.nsv_verify_attention_tile_refs if tile_references else h.nsv_verify_attention)(
        out.data_ptr(), query.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        block_tables.data_ptr(), context_lens.data_ptr(), cu_seqlens_q.data_ptr(), positions.data_ptr(),
        float(scale), batch_size, query.shape[0], num_heads, num_kv_heads, head_dim, block_size,
        max_num_blocks, qlen_bound, code, kv_split_tokens,
        _lib.ptr(ws), ws_bytes, stream)
    _lib.check(rc, "paged_attention_verify")
    return out


def store_kvcache(
    key: torch.Tensor,
    value: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
    block_size: int,
) -> None:
    """Scatter (T, Hkv, D) key/value rows into the paged caches at
    ``slot_mapping`` (slot -1 = skip), as layers/attention.py:71-112."""
    num_tokens, num_kv_heads, head_dim = key.shape
    key = key.contiguous()
    value = value.contiguous()
    if k_cache.shape != v_cache.shape:
        raise ValueError("K and V cache shapes must match")
    if slot_mapping.numel() != num_tokens:
        raise ValueError("Slot mapping size must match number of tokens")
    nb, bs, hkv, d = _check_cache(k_cache, "k_cache")
    if not v_cache.is_contiguous():
        raise ValueError("v_cache must be contiguous")
    if (bs, hkv, d) != (block_size, num_kv_heads, head_dim):
        raise ValueError("cache shape disagrees with key shape / block_size")
    if key.dtype != k_cache.dtype or value.dtype != v_cache.dtype:
        raise ValueError("key/value and caches must share one dtype")
    slot_mapping = _as(slot_mapping, "slot_mapping")
    rc = _lib.lib().nsv_store_kv(
        key.data_ptr(), value.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), slot_mapping.data_ptr(),
        num_tokens, num_kv_heads, head_dim, block_size, _lib.dtype_code(key.dtype),
        _lib.stream_ptr(key.device))
    _lib.check(rc, "store_kvcache")


def _prefill_lengths(seqlens_q, seqlens_k) -> tuple[list[int], list[int]]:
    """The lengths as lists of ints, checked."""
    seqlens_q, seqlens_k = [int(x) for x in seqlens_q], [int(x) for x in seqlens_k]
    if len(seqlens_q) != len(seqlens_k):
        raise ValueError("seqlens_q and seqlens_k differ in length")
    for i, (ql, kl) in enumerate(zip(seqlens_q, seqlens_k)):
        if not 0 < ql <= kl:
            raise ValueError(f"prefill sequence {i}: {ql} query rows over {kl} keys")
    return seqlens_q, seqlens_k


def _prefill_work(seqlens_q, seqlens_k, num_heads: int, num_kv_heads: int, block_size: int | None, cus: int,
                  pinned: bool) -> tuple[torch.Tensor, list[int]]:
    """nsv_prefill_tiles into a host tensor; returns (its words, [tiles,
    merges, tile_rows, slots])."""
    seqlens_q, seqlens_k = _prefill_lengths(seqlens_q, seqlens_k)
    n = len(seqlens_q)
    q, k, counts = (ctypes.c_int64 * n)(*seqlens_q), (ctypes.c_int64 * n)(*seqlens_k), (ctypes.c_int32 * 4)()
    words = 4096
    while True:
        buf = torch.empty(words, dtype=torch.int32, pin_memory=pinned)
        rc = _lib.lib().nsv_prefill_tiles(q, k, n, num_heads, num_kv_heads, block_size or 0, cus, buf.data_ptr(),
                                          words, counts)
        need = 8 * counts[0] + 4 * counts[1]
        if rc == 0 or need <= words:
            break
        words = need
    _lib.check(rc, "prefill_tiles")
    return buf[:need], list(counts)


def prefill_tiles(seqlens_q, seqlens_k, num_heads: int, num_kv_heads: int, block_size: int | None, cus: int):
    """The prefill kernel's work list for sequences of seqlens_q new rows
    ending seqlens_k keys each (nsv_prefill_tiles); block_size None: K/V are
    the sequences' keys back to back.  Host only.
    Returns (tiles [n, 8] int32, merges [m, 4] int32, tile_rows, slots)."""
    work, (nt, nm, rows, slots) = _prefill_work(seqlens_q, seqlens_k, num_heads, num_kv_heads, block_size, cus, False)
    return work[:8 * nt].view(nt, 8).numpy(), work[8 * nt:].view(nm, 4).numpy(), rows, slots


class _StepList:
    """A prefill step's metadata on the device, in one transfer (``work``).

    The transfer is enqueued on the stream that is current here and not waited
    for; a call on another stream waits for it on the device (use_on)."""

    def _send(self, work: torch.Tensor, device, ahead: bool) -> None:
        self.work = work.to(device, non_blocking=ahead)
        stream = torch.cuda.current_stream(device)
        self.stream = stream.cuda_stream
        self.ready = torch.cuda.Event() if ahead else None  # the transfer is done
        if ahead:
            self.ready.record(stream)

    def use_on(self, stream) -> None:
        """Order work enqueued on ``stream`` after the transfer, and keep the
        list's memory until that work is done.  A capture on another stream
        can hold no wait for an event from outside it, and needs none:
        torch.cuda.graph waits for the device before it begins, and whoever
        replays the graph keeps the plan."""
        if stream.cuda_stream == self.stream or torch.cuda.is_current_stream_capturing():
            return
        if self.ready is not None:
            stream.wait_event(self.ready)
        self.work.record_stream(stream)


def _send_ahead() -> bool:
    """As _lib.upload: a step's transfer is not waited for, except inside a
    capture, which refuses the wait."""
    return not torch.cuda.is_current_stream_capturing()


class PrefillPlan(_StepList):
    """The prefill kernel's work list of one step on the device."""

    def __init__(self, seqlens_q, seqlens_k, num_heads: int, num_kv_heads: int, block_size: int | None, device):
        cus = torch.cuda.get_device_properties(device).multi_processor_count
        ahead = _send_ahead()
        work, (self.ntiles, self.nmerges, self.tile_rows, self.slots) = _prefill_work(
            seqlens_q, seqlens_k, num_heads, num_kv_heads, block_size, cus, ahead)
        self.num_heads, self.num_kv_heads, self.block_size = num_heads, num_kv_heads, block_size
        self.sequences, self.rows, self.keys = len(seqlens_q), int(sum(seqlens_q)), int(sum(seqlens_k))
        self._send(work, device, ahead)


class PrefillRows(_StepList):
    """The verify kernel's metadata of a prefill step of a few rows per
    sequence (verify_serves_prefill) on the device: context_lens, positions
    and cu_seqlens_q, one entry per sequence or row."""

    def __init__(self, seqlens_q, seqlens_k, device):
        ql, kl = _prefill_lengths(seqlens_q, seqlens_k)
        n, rows, ahead = len(ql), sum(ql), _send_ahead()
        work = torch.empty(n + rows + n // 2 + 1, dtype=torch.int64, pin_memory=ahead)
        work[:n] = torch.tensor(kl, dtype=torch.int64)
        work[n:n + rows] = torch.cat([torch.arange(k - q, k) for q, k in zip(ql, kl)])
        work[n + rows:].view(torch.int32)[:n + 1] = torch.tensor([0] + ql).cumsum(0)
        self.sequences, self.rows, self.max_q_len = n, rows, max(ql)
        self._send(work, device, ahead)
        self.context_lens, self.positions = self.work[:n], self.work[n:n + rows]
        self.cu_seqlens_q = self.work[n + rows:].view(torch.int32)[:n + 1]


def verify_serves_prefill(seqlens_q, seqlens_k, num_heads: int, num_kv_heads: int, block_size: int,
                          max_num_blocks: int) -> bool:
    """Whether a paged bf16 prefill step runs on the verify kernel, one block
    of rows per sequence, and not on the prefill kernel.

    The prefill kernel's waves hold 32 rows of one query head and a workgroup
    two heads of a kv head, so a short suffix behind a long prefix leaves most
    of its waves without rows and a group of 4 or more heads reads its K/V
    twice or more; the verify kernel packs the group's rows.  MI355X,
    graph-replayed, prefill -> verify kernel, us per layer: 16/8 heads, one
    sequence of 9 rows behind 1,024 keys 14.7 -> 8.8, behind 16,384 47 -> 28,
    eight of 24 behind 4,096 61 -> 30; 32/8 heads, eight of 4 behind 4,096 98 ->
    26, of 12 99 -> 31.  The lines: up to 48 packed rows (the key-split kernel's
    three row tiles) wherever that kernel takes the table and 8 pairs or more
    are there, beyond one row tile (2 pairs and 16 rows of 3 heads: 17 -> 22);
    where it does not take the table (24,000 keys in pages of one or 16 tokens)
    groups of more than two heads only (32/8 heads 524 -> 342, 16/8 274 -> 336).
    Up to 64 packed rows (the verify kernel's most) groups of more than two
    heads with 1,536 keys or more: 32/8 heads, eight of 16 rows behind 4,096
    keys 101 -> 77, behind 1,024 24 -> 27; 16/8 heads, of 32 63 -> 77."""
    group, pairs, longest = num_heads // num_kv_heads, len(seqlens_q) * num_kv_heads, max(seqlens_k, default=0)
    rows = group * max(seqlens_q, default=0)
    if rows < 1 or rows > 64 or max_num_blocks * block_size >= 1 << 22:
        return False
    key_split = block_size >= 16 and max_num_blocks <= 1024
    if rows <= 48:
        return (pairs >= 8 or rows <= 16) and (key_split or group > 2)
    return pairs >= 8 and key_split and group > 2 and longest >= 1536


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """t on 16 bytes, as the loads of the prefill kernel that go straight to
    LDS need it: a view at an odd offset is copied (what torch allocates is
    aligned)."""
    return t if t.data_ptr() % 16 == 0 else t.clone()


def prefill_attention(query: torch.Tensor, k: torch.Tensor, v: torch.Tensor, plan: PrefillPlan, scale: float,
                      head_dim: int, block_tables: torch.Tensor | None = None) -> torch.Tensor:
    """Causal attention of a prefill step's rows (bf16): query [rows, H, D];
    k, v the step's own [keys, Hkv, D], or with block_tables the paged caches
    [num_blocks, block_size, Hkv, D] (layers/attention.py:123-363)."""
    H, Hkv = plan.num_heads, plan.num_kv_heads
    if not query.is_cuda:
        raise ValueError("prefill_attention runs on the GPU; query is on the CPU")
    if query.dtype != torch.bfloat16 or k.dtype != query.dtype or v.dtype != query.dtype:
        raise ValueError("query, k and v must be bfloat16")
    if query.dim() != 3 or tuple(query.shape[1:]) != (H, head_dim) or query.shape[0] < plan.rows:
        raise ValueError(f"query must be (at least {plan.rows}, {H}, {head_dim}), got {tuple(query.shape)}")
    max_blocks = 0
    if block_tables is None:
        if tuple(k.shape) != tuple(v.shape) or tuple(k.shape[1:]) != (Hkv, head_dim) or k.shape[0] < plan.keys:
            raise ValueError(f"k and v must be (at least {plan.keys}, {Hkv}, {head_dim}), got {tuple(k.shape)}")
        k, v = k.contiguous(), v.contiguous()
    else:
        nb, bs, hkv, d = _check_cache(k, "k_cache")
        if tuple(v.shape) != (nb, bs, hkv, d) or not v.is_contiguous():
            raise ValueError("k_cache and v_cache must have the same contiguous shape")
        if (bs, hkv, d) != (plan.block_size, Hkv, head_dim):
            raise ValueError("cache shape disagrees with block_size / num_kv_heads / head_dim")
        block_tables = _as(block_tables, "block_tables")
        if block_tables.shape[0] < plan.sequences:
            raise ValueError(f"{plan.sequences} sequences but {block_tables.shape[0]} block-table rows")
        max_blocks = block_tables.shape[1]
    query = query.contiguous()
    if (query.data_ptr() | k.data_ptr() | v.data_ptr()) % 16:
        query, k, v = _aligned(query), _aligned(k), _aligned(v)
    out = torch.empty_like(query)
    # (the plan's list is the only memory that calls on several streams or
    # threads share, and they only read it)
    stream = torch.cuda.current_stream(query.device)
    plan.use_on(stream)
    part = torch.empty(plan.slots * H * plan.tile_rows * (head_dim + 2), dtype=torch.float32,
                       device=query.device) if plan.slots else None
    tiles = plan.work.data_ptr()
    rc = _lib.lib().nsv_prefill_attention(
        out.data_ptr(), query.data_ptr(), k.data_ptr(), v.data_ptr(), _lib.ptr(block_tables), tiles, plan.ntiles,
        plan.tile_rows, tiles + plan.ntiles * 32, plan.nmerges, float(scale), H, Hkv, head_dim,
        plan.block_size or 1, max_blocks, _lib.ptr(part), stream.cuda_stream)
    _lib.check(rc, "prefill_attention")
    return out


_prefill_plan: tuple = (None, None)  # (the Context it was built for, its tensors)


def _prefill_rows(ctx, num_heads: int, num_kv_heads: int, device) -> tuple:
    """Verify-kernel metadata of an fp32 prefill step, built once per Context.

    Sequence i has seqlens_q[i] new rows at positions seqlens_k[i] -
    seqlens_q[i] .. seqlens_k[i] - 1.  Its rows are cut into causal blocks of
    q_block = 64 // G rows (G query heads per kv head: the kernel holds up to
    64 query rows per (sequence, kv head)); each block is one entry of the
    kernel's batch with context = the block's last position + 1, so every
    row attends exactly keys 0 .. its position.  Block-table row of block j:
    the sequence's row of context.block_tables (paged prefill) or, without
    block tables, the sequence's keys in the step's own contiguous K/V read
    as one-token pages (cu_seqlens_k[i] + p for position p).
    Returns (block_tables, context_lens, cu_seqlens_q, positions, q_block)."""
    import numpy as np

    global _prefill_plan
    if _prefill_plan[0] is ctx:
        return _prefill_plan[1]
    if ctx.seqlens_q is None or ctx.seqlens_k is None:
        raise ValueError("a prefill step needs context.seqlens_q and context.seqlens_k")
    q_block = max(1, 64 // (num_heads // num_kv_heads))
    paged = ctx.block_tables is not None
    tables = ctx.block_tables.cpu().numpy() if paged else None
    width = tables.shape[1] if paged else max(ctx.seqlens_k)
    bt, lens, cu, pos = [], [], [0], []
    k_start = 0
    for i, (ql, kl) in enumerate(zip(ctx.seqlens_q, ctx.seqlens_k)):
        if not 0 < ql <= kl:
            raise ValueError(f"prefill sequence {i}: {ql} query rows over {kl} keys")
        if paged:
            row = tables[i].astype(np.int32)
        else:
            row = np.full(width, -1, dtype=np.int32)
            row[:kl] = np.arange(k_start, k_start + kl, dtype=np.int32)
        for b0 in range(kl - ql, kl, q_block):
            b1 = min(kl, b0 + q_block)
            bt.append(row)
            lens.append(b1)
            cu.append(cu[-1] + (b1 - b0))
        pos.append(np.arange(kl - ql, kl, dtype=np.int64))
        k_start += kl
    t = lambda x, dt: torch.from_numpy(np.ascontiguousarray(x, dtype=dt)).to(device)  # noqa: E731
    out = (t(np.stack(bt), np.int32), t(lens, np.int64), t(cu, np.int32), t(np.concatenate(pos), np.int64), q_block)
    _prefill_plan = (ctx, out)
    return out


class Attention(nn.Module):
    """Attention layer of the reference (layers/attention.py:670-767):
    writes this step's K/V into the paged cache at context.slot_mapping,
    then attends from the query rows the global Context describes:
      * verify (context.is_verify): a chunk of drafted tokens per sequence
        with a causal mask from absolute positions (:704-731);
      * prefill (context.is_prefill, :733-757): every new prompt row of each
        sequence, causally over its keys.  With context.block_tables (a
        prompt behind a cached prefix) the keys come from the paged cache,
        the step's own K/V already stored in it, as the reference's
        paged_attention_prefill (:328-363); without, from the step's
        contiguous K/V, as its varlen flash path (:257-325).  bf16 runs on
        the prefill kernel (``prefill_attention``), paged steps of a few rows
        per sequence on the verify kernel (``verify_serves_prefill``), fp32 on
        the verify kernel over causal blocks of rows (``_prefill_rows``);
      * decode (neither flag): one query row per sequence attending its
        whole context (:759-767), served by the same verify kernel with
        each row at position context_lens - 1."""

    def __init__(self, num_heads: int, head_dim: int, scale: float = 1.0, num_kv_heads: int | None = None,
                 block_size: int = 16):
        super().__init__()
        self.num_heads = num_heads
        self.head_dim = head_dim
        self.scale = scale
        self.num_kv_heads = num_kv_heads if num_kv_heads is not None else num_heads
        self.block_size = block_size
        self.k_cache = self.v_cache = torch.tensor([])

    def _prefill_bf16(self, context, q, k, v, scale: float) -> torch.Tensor:
        """The prefill branch on the prefill kernel, or on the verify kernel
        for a few rows per sequence; the step's work list is built by its
        first layer and kept with the step's Context."""
        paged = context.block_tables is not None
        if context.seqlens_q is None or context.seqlens_k is None:
            raise ValueError("a prefill step needs context.seqlens_q and context.seqlens_k")
        bs = self.block_size if paged else None
        key = (self.num_heads, self.num_kv_heads, bs, q.device)
        plans = context.__dict__.setdefault("prefill_plans", {})
        if paged and verify_serves_prefill(context.seqlens_q, context.seqlens_k, self.num_heads, self.num_kv_heads, bs,
                                           context.block_tables.shape[1]):
            return self._prefill_few(context, plans, q, scale)
        plan = plans.get(key)
        if plan is None:
            plan = plans[key] = PrefillPlan(context.seqlens_q, context.seqlens_k, self.num_heads, self.num_kv_heads,
                                            bs, q.device)
        if paged:
            return prefill_attention(q, self.k_cache, self.v_cache, plan, scale, self.head_dim,
                                     context.block_tables.to(q.device))
        return prefill_attention(q, k.reshape(-1, self.num_kv_heads, self.head_dim),
                                 v.reshape(-1, self.num_kv_heads, self.head_dim), plan, scale, self.head_dim)

    def _prefill_few(self, context, plans: dict, q, scale: float) -> torch.Tensor:
        """A paged prefill step of a few rows per sequence as one verify call."""
        rows = plans.get(q.device)
        if rows is None:
            rows = plans[q.device] = PrefillRows(context.seqlens_q, context.seqlens_k, q.device)
        if q.shape[0] < rows.rows:
            raise ValueError(f"query must have at least {rows.rows} rows, got {q.shape[0]}")
        tables = context.block_tables.to(q.device)
        if tables.shape[0] < rows.sequences:
            raise ValueError(f"{rows.sequences} sequences but {tables.shape[0]} block-table rows")
        rows.use_on(torch.cuda.current_stream(q.device))
        return paged_attention_verify(
            q, self.k_cache, self.v_cache, tables[:rows.sequences], rows.context_lens, rows.cu_seqlens_q, rows.positions,
            scale, self.num_heads, self.num_kv_heads, self.head_dim, self.block_size, 64, max_q_len=rows.max_q_len,
            tile_references=True)

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        context = get_context()
        k_cache, v_cache = self.k_cache, self.v_cache
        if k_cache.numel() > 0 and v_cache.numel() > 0 and context.slot_mapping is not None:
            store_kvcache(k.reshape(-1, self.num_kv_heads, self.head_dim),
                          v.reshape(-1, self.num_kv_heads, self.head_dim),
                          k_cache, v_cache, context.slot_mapping, self.block_size)
        scale = self.scale / (self.head_dim ** 0.5)
        q = q.reshape(-1, self.num_heads, self.head_dim)
        if context.is_prefill and not context.is_verify:
            if context.cu_seqlens_q is None:
                raise ValueError("cu_seqlens_q must be provided for varlen attention")
            if q.dtype == torch.bfloat16:
                o = self._prefill_bf16(context, q, k, v, scale)
                return o.reshape(o.shape[0], self.num_heads * self.head_dim)
            bt, lens, cu, positions, q_block = _prefill_rows(context, self.num_heads, self.num_kv_heads, q.device)
            if context.block_tables is not None:
                kc, vc, bs = k_cache, v_cache, self.block_size
            else:  # the step's own keys, one token per page
                kc = k.reshape(-1, 1, self.num_kv_heads, self.head_dim).contiguous()
                vc = v.reshape(-1, 1, self.num_kv_heads, self.head_dim).contiguous()
                bs = 1
            o = paged_attention_verify(q, kc, vc, bt, lens, cu, positions, scale, self.num_heads, self.num_kv_heads,
                                       self.head_dim, bs, max(16, q_block), max_q_len=q_block)
            return o.reshape(o.shape[0], self.num_heads * self.head_dim)
        if context.is_verify:
            max_q_len = max(context.seqlens_q)
            cu, positions = context.cu_seqlens_q, context.positions
        else:
            # decode: row b is the newest token of sequence b
            max_q_len = 1
            cu = torch.arange(0, q.shape[0] + 1, dtype=torch.int32, device=q.device)
            positions = context.context_lens.to(torch.int64) - 1
        block_m = max(16, 1 << (max_q_len - 1).bit_length())
        o = paged_attention_verify(
            q, k_cache, v_cache, context.block_tables, context.context_lens, cu, positions, scale,
            self.num_heads, self.num_kv_heads, self.head_dim, self.block_size, block_m, max_q_len=max_q_len)
        return o.reshape(o.shape[0], self.num_heads * self.head_dim)
