"""Qwen3 verify forward on the MI355X path.

The target model of the verification round (src/myvllm/models/qwen3.py:
Qwen3Attention :11-123, Qwen3MLP :129-151, Qwen3DecoderLayer :159-227,
Qwen3Model :233-281, Qwen3ForCausalLM :287-344): embedding, N decoder
layers (RMSNorm, fused QKV projection, per-head q/k RMSNorm, NeoX RoPE,
paged KV store + paged verify attention, o_proj, RMSNorm with residual,
SwiGLU MLP), final norm, LM head over every row.  Up to fused_rows() verify
rows every layer runs on this library's gfx950 kernels, 6 launches per
layer: the QKV projection (with the input RMSNorm as its prologue), the
pre-attention epilogue (q/k RMSNorm + RoPE + paged KV store), verify
attention, o_proj (with the residual add as its epilogue), gate_up
(post-attention RMSNorm prologue, SiLU * up epilogue) and down (residual
add epilogue). Up to WIDE_ROWS rows they run on the weight-streaming
projections where the hidden size is above WIDE_HIDDEN (8 launches per layer),
other batches on hipBLASLt between this library's residual-RMSNorm, epilogue,
attention and SiLU kernels. The LM head runs on this library's streaming kernel
up to lm_head_rows() rows (79 at hidden 1024, 19 at hidden 4096: the
activations staged in one CU's LDS), from a copy of its weight packed in that
kernel's load order, on the weight-streaming kernel from the same copy up to
WIDE_ROWS, and on hipBLASLt beyond. Weights are random (seeded): no checkpoint
is loaded.

The forward takes the verify metadata explicitly (positions, slots, block
tables, context lengths, cu_seqlens) so a whole forward is capturable in a
hipGraph with static buffers, as the reference's verify graphs are
(engine/model_runner.py:648-721).
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch
import torch.nn.functional as F

from naivllm_amd import _lib
from naivllm_amd.layers.attention import (PrefillPlan, PrefillRows, paged_attention_verify, prefill_attention,
                                          verify_serves_prefill)


@dataclass
class Qwen3Config:
    vocab_size: int = 151936
    hidden_size: int = 1024
    num_layers: int = 28
    num_heads: int = 16
    num_kv_heads: int = 8
    head_dim: int = 128
    intermediate_size: int = 3072
    rms_norm_eps: float = 1e-6
    rope_theta: float = 1_000_000.0
    max_position: int = 40960
    tie_word_embeddings: bool = True

    @staticmethod
    def qwen3_0_6b(**kw) -> "Qwen3Config":
        return Qwen3Config(**kw)

    @staticmethod
    def qwen3_8b(**kw) -> "Qwen3Config":
        base = dict(hidden_size=4096, num_layers=36, num_heads=32, num_kv_heads=8, head_dim=128,
                    intermediate_size=12288, tie_word_embeddings=False)
        base.update(kw)
        return Qwen3Config(**base)


def rope_cache(cfg: Qwen3Config, device) -> torch.Tensor:
    """[max_position, head_dim] = [cos | sin] of NeoX rotary embedding
    (layers/rotary_embedding.py:48-72), fp32."""
    d = cfg.head_dim
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, d, 2, dtype=torch.float64) / d))
    pos = torch.arange(cfg.max_position, dtype=torch.float64)
    f = torch.outer(pos, inv)
    return torch.cat([torch.cos(f), torch.sin(f)], dim=-1).float().contiguous().to(device)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, out: torch.Tensor,
             residual: torch.Tensor | None = None, residual_out: torch.Tensor | None = None) -> None:
    """out = rmsnorm(x + residual) * weight; x + residual goes to
    residual_out (layers/layernorm.py:18-35)."""
    T, E = x.shape
    rc = _lib.lib().nsv_rms_norm(x.data_ptr(), _lib.ptr(residual), _lib.ptr(residual_out), weight.data_ptr(),
                                 out.data_ptr(), T, E, eps, _lib.stream_ptr(x.device))
    _lib.check(rc, "rms_norm")


def embed_rms_norm(ids: torch.Tensor, embed: torch.Tensor, weight: torch.Tensor, eps: float, residual_out, out,
                   positions: torch.Tensor | None = None, cos_sin: torch.Tensor | None = None,
                   rope_out: torch.Tensor | None = None) -> None:
    """The forward's prologue (nsv_embed_rms_norm): residual_out = embed[ids],
    out = rmsnorm(residual_out) * weight, and rope_out [T, D] = cos_sin rows
    at the (clamped) positions when given."""
    ids = ids.to(torch.int64).contiguous()
    T, E = residual_out.shape
    D = cos_sin.shape[1] if cos_sin is not None else 0
    rc = _lib.lib().nsv_embed_rms_norm(
        ids.data_ptr(), embed.data_ptr(), embed.shape[0], weight.data_ptr(), eps, residual_out.data_ptr(),
        out.data_ptr(), T, E, _lib.ptr(positions), _lib.ptr(cos_sin), cos_sin.shape[0] if cos_sin is not None else 0,
        D, _lib.ptr(rope_out), _lib.stream_ptr(residual_out.device))
    _lib.check(rc, "embed_rms_norm")


def qk_norm_rope_store(qkv, q_norm_w, k_norm_w, cos_sin, positions, slot_mapping, q_out, k_cache, v_cache,
                       H: int, Hkv: int, D: int, eps: float) -> None:
    """The pre-attention epilogue (nsv_qk_norm_rope_store).  positions None:
    cos_sin holds the rotary row of each step row ([T, D])."""
    rc = _lib.lib().nsv_qk_norm_rope_store(
        qkv.data_ptr(), q_norm_w.data_ptr(), k_norm_w.data_ptr(), cos_sin.data_ptr(), cos_sin.shape[0],
        _lib.ptr(positions), slot_mapping.data_ptr(), q_out.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        qkv.shape[0], H, Hkv, D, eps, _lib.stream_ptr(qkv.device))
    _lib.check(rc, "qk_norm_rope_store")


def decode_fits(hidden: int, attn_dim: int, intermediate: int) -> bool:
    """Whether every projection's reduction suits nsv_linear_decode, and the
    partial sums of the hidden size fit its prologue (at most 256 slots)."""
    return all(k in (1024, 2048, 3072, 4096) for k in (hidden, attn_dim, intermediate)) and hidden // 4 <= 256


def decode_ss_rows(M: int, N: int) -> int:
    """Partial-sum rows a decode-shaped residual epilogue writes (nsv_linear_decode)."""
    return int(_lib.lib().nsv_linear_decode_ss_rows(M, N))


def ss_rows(M: int, N: int, K: int, has_norm: bool = False) -> int:
    """Rows of partial sums of r^2 a residual-epilogue linear writes (one per
    16- or 8-column tile of the output)."""
    return int(_lib.lib().nsv_linear_ss_rows(M, N, K, int(has_norm)))


def lm_head(x: torch.Tensor, packed: torch.Tensor, y: torch.Tensor) -> None:
    """y = x @ W.T (ParallelLMHead.forward's F.linear) from W's copy written
    by nsv_lm_head_pack, on the streaming kernel (nsv_lm_head): the same bits
    as linear(x, W, y)."""
    M, K = x.shape
    N = y.shape[1]
    if (tuple(packed.shape) != (N, K) or y.shape[0] != M or not (x.is_contiguous() and y.is_contiguous())
            or not (x.dtype == packed.dtype == y.dtype == torch.bfloat16)):
        raise ValueError("lm_head: x [M, K], packed [N, K] and y [M, N], contiguous bf16")
    rc = _lib.lib().nsv_lm_head(x.data_ptr(), packed.data_ptr(), y.data_ptr(), M, N, K, _lib.stream_ptr(x.device))
    _lib.check(rc, "lm_head")


def linear(x: torch.Tensor, weight: torch.Tensor, y: torch.Tensor | None = None, *,
           norm_w: torch.Tensor | None = None, ss_in: torch.Tensor | None = None, eps: float = 1e-6,
           swiglu: bool = False, resid: torch.Tensor | None = None, ss_out: torch.Tensor | None = None,
           decode: bool = False) -> None:
    """y = h @ weight.T on this library's few-row kernel (nsv_linear), or,
    decode=True, on its one-wave-per-column kernel for one or two rows
    (nsv_linear_decode: ss_out then has decode_ss_rows(M, N) rows).

    h = rmsnorm(x) * norm_w when norm_w is given (x is then the residual
    stream and ss_in [n, M] the producer's partial sums of x^2), else x.
    swiglu: weight is [gate; up] and y = silu(gate) * up.  resid: instead of
    writing y, add the product into the residual stream resid [M, N] and
    write the new partial sums of resid^2 to ss_out [ss_rows(M, N, K), M]."""
    M, K = x.shape
    N = weight.shape[0]
    epi = 2 if resid is not None else (1 if swiglu else 0)
    nss = ss_in.shape[0] if ss_in is not None else 0
    h = _lib.lib()
    if decode:
        rc = h.nsv_linear_decode(x.data_ptr(), _lib.ptr(norm_w), _lib.ptr(ss_in), nss, eps, weight.data_ptr(),
                                 _lib.ptr(y), _lib.ptr(resid), _lib.ptr(ss_out), M, N, K, epi,
                                 _lib.stream_ptr(x.device))
        _lib.check(rc, "linear_decode")
        return
    nbytes = h.nsv_linear_workspace_size(M, N, K)
    ws = _lib.workspace(x.device, nbytes, "linear")
    rc = h.nsv_linear(x.data_ptr(), _lib.ptr(norm_w), _lib.ptr(ss_in), nss, eps, weight.data_ptr(),
                      _lib.ptr(y), _lib.ptr(resid), _lib.ptr(ss_out), M, N, K, epi, _lib.ptr(ws),
                      ws.numel() if ws is not None else 0, _lib.stream_ptr(x.device))
    _lib.check(rc, "linear")


def wide_splits(M: int, N: int, K: int, swiglu: bool = False, packed: bool = False) -> int:
    """Workgroups nsv_wide_linear cuts the reduction over (0: not its shape)."""
    return int(_lib.lib().nsv_wide_linear_splits(M, N, K, int(swiglu), int(packed)))


def dense_bf16(t: torch.Tensor | None, M: int, N: int, device) -> bool:
    """Whether t is what the projections write: contiguous bf16 [M, N] on device."""
    return (t is not None and tuple(t.shape) == (M, N) and t.dtype == torch.bfloat16 and t.is_contiguous()
            and t.device == device)


def _check_partials(partials: torch.Tensor | None, splits: int, T: int, N: int, device) -> None:
    if (partials is None or partials.dtype != torch.float32 or not partials.is_contiguous()
            or partials.device != device or partials.numel() < splits * T * N):
        raise ValueError(f"partials: contiguous fp32 of at least {splits} x {T} x {N} on {device}")


def _check_cuda(t: torch.Tensor, what: str) -> None:
    if not t.is_cuda:
        raise ValueError(f"{what} runs on the GPU; its input is on {t.device}")


def wide_linear(x: torch.Tensor, weight: torch.Tensor, y: torch.Tensor | None, partials: torch.Tensor | None = None, *,
                swiglu: bool = False, packed: bool = False) -> None:
    """y = x @ weight.T on the weight-streaming kernel of up to 128 rows
    (nsv_wide_linear); with wide_splits > 1 the fp32 partial sums go to
    ``partials`` ([splits, M, N] at its start) instead.  swiglu: weight is
    [gate; up] and y = silu(gate) * up.  packed: weight in the LM head's
    packed layout."""
    M, K = x.shape
    N = weight.shape[0]
    if (weight.shape[1] != K or not (x.is_contiguous() and weight.is_contiguous())
            or not (x.dtype == weight.dtype == torch.bfloat16)):
        raise ValueError(f"wide_linear: x [M, K] and weight [N, K], contiguous bf16; got {tuple(x.shape)} {x.dtype}, "
                         f"{tuple(weight.shape)} {weight.dtype}")
    splits = wide_splits(M, N, K, swiglu, packed)
    if splits > 1:
        _check_partials(partials, splits, M, N, x.device)
    elif not dense_bf16(y, M, N // 2 if swiglu else N, x.device):
        raise ValueError(f"wide_linear: y must be a contiguous bf16 [{M}, {N // 2 if swiglu else N}] on {x.device}")
    _check_cuda(x, "wide_linear")
    rc = _lib.lib().nsv_wide_linear(x.data_ptr(), weight.data_ptr(), _lib.ptr(y), _lib.ptr(partials), M, N, K,
                                    int(swiglu), int(packed), _lib.stream_ptr(x.device))
    _lib.check(rc, "wide_linear")


def rms_norm_sum(partials: torch.Tensor, splits: int, weight: torch.Tensor, eps: float, out: torch.Tensor,
                 residual: torch.Tensor, residual_out: torch.Tensor | None = None) -> None:
    """rms_norm whose x is the sum of a split projection's partials."""
    T, E = out.shape
    _check_partials(partials, splits, T, E, out.device)
    if (not all(dense_bf16(t, T, E, out.device) for t in (out, residual, residual if residual_out is None else residual_out))
            or tuple(weight.shape) != (E,) or weight.dtype != torch.bfloat16):
        raise ValueError(f"rms_norm_sum: out, residual and residual_out [{T}, {E}] and weight [{E}], contiguous bf16")
    _check_cuda(out, "rms_norm_sum")
    rc = _lib.lib().nsv_rms_norm_sum(partials.data_ptr(), splits, residual.data_ptr(), _lib.ptr(residual_out),
                                     weight.data_ptr(), out.data_ptr(), T, E, eps, _lib.stream_ptr(out.device))
    _lib.check(rc, "rms_norm_sum")


def qk_norm_rope_store_sum(partials, splits: int, q_norm_w, k_norm_w, rope_rows, slot_mapping, q_out, k_cache, v_cache,
                           H: int, Hkv: int, D: int, eps: float) -> None:
    """qk_norm_rope_store (one rotary row per step row) whose qkv is the sum
    of a split projection's partials."""
    T = q_out.shape[0]
    _check_partials(partials, splits, T, (H + 2 * Hkv) * D, q_out.device)
    if not (rope_rows.shape[0] >= T and slot_mapping.numel() >= T and rope_rows.is_contiguous()
            and rope_rows.dtype == torch.float32 and slot_mapping.dtype == torch.int64 and slot_mapping.is_contiguous()):
        raise ValueError(f"qk_norm_rope_store_sum: fp32 rope_rows and int64 slot_mapping of {T} rows, contiguous")
    _check_cuda(q_out, "qk_norm_rope_store_sum")
    rc = _lib.lib().nsv_qk_norm_rope_store_sum(
        partials.data_ptr(), splits, q_norm_w.data_ptr(), k_norm_w.data_ptr(), rope_rows.data_ptr(),
        slot_mapping.data_ptr(), q_out.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), T, H, Hkv, D, eps,
        _lib.stream_ptr(q_out.device))
    _lib.check(rc, "qk_norm_rope_store_sum")


def silu_mul(gate_up: torch.Tensor, out: torch.Tensor) -> None:
    rc = _lib.lib().nsv_silu_mul(gate_up.data_ptr(), out.data_ptr(), gate_up.shape[0], out.shape[1],
                                 _lib.stream_ptr(gate_up.device))
    _lib.check(rc, "silu_mul")


# Verify rows up to which the forward runs on the fused few-row linear
# kernel.  Every workgroup of that kernel reads the whole activation block,
# so its cost grows with rows x hidden size, while hipBLASLt's wide tiles
# reuse the activations.  Measured on MI355X (each projection alone): at
# hidden 1024 the fused layer (4 launches) beats hipBLASLt + the separate
# norm / SiLU kernels up to 72 rows (38 vs 42 us per layer at 72; attention
# included and graph-replayed, 65 vs 72 at 72, 66 vs 72 at 80, 84 vs 73 at 96);
# at hidden 4096 it wins at 9 rows and loses from about 20 (graph-replayed
# against the weight-streaming kernel: 93 vs 108 at 13, 96 vs 109 at 16, 116 vs
# 116 at 20, 148 vs 124 at 36): the line, at the drafts + 1 rows of one request,
# is on the safe side of that.
FUSED_ROWS = 80
FUSED_ROWS_WIDE = 12  # hidden size above 2048


# Rows, past the fused kernel's, up to which the projections and the LM head
# run on the weight-streaming kernel (nsv_wide_linear): beyond, the activations
# each workgroup re-reads cost what the library GEMM's larger tiles save.
# Measured on MI355X at hidden 4096, graph-replayed over rotating weights, the
# library against it: 72 rows qkv 23.1 -> 17.0 us, o 16.2 -> 11.5, gate_up with
# SiLU 53.5 + 4 -> 46, down 42.9 -> 25.5, LM head 283 -> 239; 108 rows 23.7 ->
# 21.2, 16.4 -> 14.1, 55 + 4 -> 55, 43.1 -> 30.6, 291 -> 282.  A whole layer at
# 16, 36, 72, 96 and 128 rows: 126 -> 116, 146 -> 128, 178 -> 150, 198 -> 164,
# 225 -> 187 us (intermediate size 14336: 143 -> 127, 157 -> 141, 189 -> 163,
# 128 rows 244 -> 197; 16384: 54 rows 171 -> 163, 16 rows 146 -> 149).  The LM
# head alone at hidden 1024, 2048 and 4096: 80 rows 84 -> 66, 161 -> 121, 272 ->
# 241, 128 rows 90 -> 79, 167 -> 143, 279 -> 277.
WIDE_ROWS = 128
# Hidden size past which the layers do (the head at any): up to it the fused
# kernel serves 80 rows, and past those a layer takes, library against this
# kernel, at hidden 1024 72.7 -> 73.7 us (88 rows), 79.3 -> 84.7 (108), 81.5 ->
# 89.8 (128), at 2048 103.5 -> 101.2 (96), 109.3 -> 111.0 (108), 114 -> 117
# (128); at 2560 72 rows 132 -> 122, 128 rows 185 -> 154.
WIDE_HIDDEN = 2048


# Rows up to which the LM head runs on this library's kernels: nsv_linear
# streams a vocabulary-wide head's weight tiles while the activations fit its
# LDS (rows x (hidden + 8) bf16 within 160 KiB), hipBLASLt's large tiles
# beyond.  Measured on MI355X, graph-replayed, the 0.6B head alone: 58.6 vs
# 58.6 us at 9 rows, 59.9 vs 69.2 at 18, 70.5 vs 83.7 at 72; the 8B head
# (hidden 4096): 232 vs 248 us at 9 rows.
LM_HEAD_LDS = 160 * 1024


def lm_head_rows(hidden: int) -> int:
    return max(16, min(79, LM_HEAD_LDS // ((hidden + 8) * 2)))


def prefill_rows(token_lists, starts, tables, block_size: int):
    """Rows of one prefill forward over several sequences' new tokens, as
    numpy arrays: sequence i contributes its tokens starts[i] ..
    len(token_lists[i]) - 1 at their positions (the pages before starts[i]
    already hold their KV: a cached prefix).
    Returns (input_ids, positions, slot_mapping, last_rows, block_tables, new,
    lens): last_rows[i] is the row of sequence i's last token, block_tables
    has one row per sequence (-1 padded), and new / lens are the sequences'
    new and whole lengths."""
    import numpy as np

    if not len(token_lists) == len(starts) == len(tables):
        raise ValueError(f"{len(token_lists)} token lists, {len(starts)} starts and {len(tables)} block tables")
    lens = [len(t) for t in token_lists]
    for n, start in zip(lens, starts):
        if not 0 <= start < n:
            raise ValueError(f"prefill start {start} outside a {n}-token sequence")
    new = [n - start for n, start in zip(lens, starts)]
    pos = [np.arange(start, n, dtype=np.int64) for n, start in zip(lens, starts)]
    slots = [np.asarray(t, dtype=np.int64)[p // block_size] * block_size + p % block_size for t, p in zip(tables, pos)]
    ids = [np.asarray(t[start:], dtype=np.int64) for t, start in zip(token_lists, starts)]
    bt = np.full((len(tables), max(len(t) for t in tables)), -1, dtype=np.int32)
    for row, t in zip(bt, tables):
        row[:len(t)] = t
    last = np.cumsum(new, dtype=np.int64) - 1
    return np.concatenate(ids), np.concatenate(pos), np.concatenate(slots), last, bt, new, lens


def fused_rows(hidden_size: int) -> int:
    return FUSED_ROWS if hidden_size <= 2048 else FUSED_ROWS_WIDE


class Qwen3Verify:
    """Random-init Qwen3 weights plus the verify forward."""

    def __init__(self, cfg: Qwen3Config, device, dtype=torch.bfloat16, seed: int = 0, std: float = 0.02):
        self.cfg = cfg
        self.device = torch.device(device)
        self.dtype = dtype
        g = torch.Generator(device=self.device)
        g.manual_seed(seed)

        def w(*shape, scale=std):
            return (torch.randn(*shape, generator=g, device=self.device, dtype=torch.float32) * scale).to(dtype)

        H, Hkv, D, E = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.hidden_size
        self.embed = w(cfg.vocab_size, E, scale=1.0)
        self.layers = []
        for _ in range(cfg.num_layers):
            self.layers.append(dict(
                ln1=torch.ones(E, device=self.device, dtype=dtype),
                qkv=w((H + 2 * Hkv) * D, E, scale=1.0 / math.sqrt(E)),
                q_norm=torch.ones(D, device=self.device, dtype=dtype),
                k_norm=torch.ones(D, device=self.device, dtype=dtype),
                o=w(E, H * D, scale=1.0 / math.sqrt(H * D)),
                ln2=torch.ones(E, device=self.device, dtype=dtype),
                gate_up=w(2 * cfg.intermediate_size, E, scale=1.0 / math.sqrt(E)),
                down=w(E, cfg.intermediate_size, scale=1.0 / math.sqrt(cfg.intermediate_size)),
            ))
        self.norm = torch.ones(E, device=self.device, dtype=dtype)
        self.lm_head = self.embed if cfg.tie_word_embeddings else w(cfg.vocab_size, E, scale=1.0 / math.sqrt(E))
        self.pack_lm_head()
        self.rope = rope_cache(cfg, self.device)
        self.scale = 1.0 / math.sqrt(D)
        self.k_caches: list[torch.Tensor] = []
        self.v_caches: list[torch.Tensor] = []
        self.block_size = 0
        # forwards of one or two rows take the one-wave-per-column projections
        # (a drafter's steps; the target keeps one kernel family at every row
        # count, so its rows come out the same at every batch shape)
        self.decode_linears = False

    def pack_lm_head(self) -> None:
        """Repack the LM head's weight in the streaming kernel's load order
        (nsv_lm_head_pack) where this shape streams; it serves up to WIDE_ROWS
        rows, the row-major weight the embedding lookup and more rows.  Called
        once by the constructor; whoever replaces or edits self.lm_head
        afterwards calls it again."""
        self.lm_head_packed = None
        self.lm_head_packed_rows = 0
        if self.device.type != "cuda" or self.lm_head.dtype != torch.bfloat16:
            return
        V, E = self.lm_head.shape
        self.lm_head_packed_rows = _lib.lib().nsv_lm_head_rows(V, E)
        if self.lm_head_packed_rows > 0:
            self.lm_head_packed = torch.empty_like(self.lm_head)
            _lib.check(_lib.lib().nsv_lm_head_pack(self.lm_head.data_ptr(), self.lm_head_packed.data_ptr(), V, E,
                                                   _lib.stream_ptr(self.device)), "lm_head_pack")

    def _wide_splits(self, T: int) -> tuple[int, int, int] | None:
        """Splits of the qkv, o and down projections where T rows run on the
        weight-streaming kernel, else None."""
        cfg = self.cfg
        E, I, HD = cfg.hidden_size, cfg.intermediate_size, cfg.num_heads * cfg.head_dim
        # (its loads take weights on 16 bytes: a view at an odd offset stays on hipBLASLt)
        if T > WIDE_ROWS or E <= WIDE_HIDDEN or E % 4 or E > 4096 or not all(
                L[k].is_contiguous() and L[k].data_ptr() % 16 == 0
                for L in self.layers for k in ("qkv", "o", "gate_up", "down")):
            return None
        n = (wide_splits(T, HD + 2 * cfg.num_kv_heads * cfg.head_dim, E), wide_splits(T, E, HD), wide_splits(T, E, I))
        return n if min(*n, wide_splits(T, 2 * I, E, swiglu=True)) > 0 else None

    @torch.inference_mode()
    def prefill(self, token_lists, starts, tables) -> torch.Tensor:
        """One forward over the new tokens of several sequences (sequence i's
        from starts[i] on; the pages before hold their K/V: a cached prefix):
        their K/V land in the paged cache, and the logits of each sequence's
        last token come back, [len(token_lists), vocab]."""
        import numpy as np

        bs = self.block_size
        *per_row, last, bt, new, lens = prefill_rows(token_lists, starts, tables, bs)
        rows = _lib.upload(np.concatenate([*per_row, last]), self.device)
        T = sum(new)
        H, Hkv = self.cfg.num_heads, self.cfg.num_kv_heads
        args = (rows[:T], rows[T:2 * T], rows[2 * T:3 * T], _lib.upload(bt, self.device))
        if verify_serves_prefill(new, lens, H, Hkv, bs, bt.shape[1]):
            few = PrefillRows(new, lens, self.device)
            return self.forward(*args, few.context_lens, few.cu_seqlens_q, few.max_q_len, logits_rows=rows[3 * T:],
                                tile_references=True)
        plan = PrefillPlan(new, lens, H, Hkv, bs, self.device)
        return self.forward(*args, None, None, 0, logits_rows=rows[3 * T:], prefill=plan)

    def allocate_kv_cache(self, num_blocks: int, block_size: int) -> None:
        """One [num_blocks, block_size, Hkv, D] K and V pool per layer
        (engine/model_runner.py:244-279 keeps one [2, L, ...] tensor)."""
        cfg = self.cfg
        shape = (num_blocks, block_size, cfg.num_kv_heads, cfg.head_dim)
        self.k_caches = [torch.zeros(shape, device=self.device, dtype=self.dtype) for _ in range(cfg.num_layers)]
        self.v_caches = [torch.zeros(shape, device=self.device, dtype=self.dtype) for _ in range(cfg.num_layers)]
        self.block_size = block_size

    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor, slot_mapping: torch.Tensor,
                block_tables: torch.Tensor, context_lens: torch.Tensor, cu_seqlens_q: torch.Tensor,
                max_q_len: int, logits_out: torch.Tensor | None = None,
                logits_rows: torch.Tensor | None = None, prefill: PrefillPlan | None = None,
                tile_references: bool = False) -> torch.Tensor:
        """Verify forward over T = sum of per-sequence query rows.  Rows at
        position -1 are inert padding (no KV store, zero attention output).
        Returns logits [T, vocab] (written into logits_out when given), or
        only the rows ``logits_rows`` indexes (the prefill's last rows).
        prefill: the rows are whole prompts' (block_tables then one row per
        prompt; context_lens, cu_seqlens_q and max_q_len are not used).
        tile_references: as paged_attention_verify's."""
        if self.dtype != torch.bfloat16:
            raise ValueError("the fused forward kernels are bf16")
        cfg = self.cfg
        H, Hkv, D, E = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.hidden_size
        eps = cfg.rms_norm_eps
        T = input_ids.shape[0]
        I = cfg.intermediate_size
        resid = torch.empty(T, E, dtype=self.dtype, device=self.device)  # the residual stream
        h = torch.empty_like(resid)
        q = torch.empty(T, H, D, dtype=self.dtype, device=self.device)
        if prefill is not None:
            attn = lambda li: prefill_attention(  # noqa: E731
                q, self.k_caches[li], self.v_caches[li], prefill, self.scale, D, block_tables)
        else:
            block_m = max(16, 1 << (max_q_len - 1).bit_length())
            attn = lambda li: paged_attention_verify(  # noqa: E731
                q, self.k_caches[li], self.v_caches[li], block_tables, context_lens, cu_seqlens_q, positions,
                self.scale, H, Hkv, D, self.block_size, block_m, max_q_len=max_q_len, tile_references=tile_references)
        # embedding lookup, layer 0's input norm, and the rotary rows of the step's
        # positions (gathered once for every layer, so that each layer's epilogue
        # loads them without first loading the positions) in one launch
        rope_rows = torch.empty(T, D, dtype=torch.float32, device=self.device)
        embed_rms_norm(input_ids, self.embed, self.layers[0]["ln1"], eps, resid, h, positions, self.rope, rope_rows)
        if T <= fused_rows(E):
            # Every RMSNorm after layer 0's is the prologue of the projection
            # that consumes it and every residual add the epilogue of the
            # projection that produces it: 6 launches per layer.
            qkv = torch.empty(T, (H + 2 * Hkv) * D, dtype=self.dtype, device=self.device)
            act = torch.empty(T, I, dtype=self.dtype, device=self.device)
            # one or two rows on a drafter: the one-wave-per-column kernel
            dec = self.decode_linears and T <= 2 and decode_fits(E, H * D, I)
            # partial sums of resid^2 from o_proj and down (their tiles' count)
            ss_o = torch.empty(decode_ss_rows(T, E) if dec else ss_rows(T, E, H * D), T, dtype=torch.float32,
                               device=self.device)
            ss_d = torch.empty(decode_ss_rows(T, E) if dec else ss_rows(T, E, I), T, dtype=torch.float32,
                               device=self.device)
            for li, L in enumerate(self.layers):
                if li == 0:
                    linear(h, L["qkv"], qkv, decode=dec)
                else:
                    linear(resid, L["qkv"], qkv, norm_w=L["ln1"], ss_in=ss_d, eps=eps, decode=dec)
                qk_norm_rope_store(qkv, L["q_norm"], L["k_norm"], rope_rows, None, slot_mapping, q,
                                   self.k_caches[li], self.v_caches[li], H, Hkv, D, eps)
                linear(attn(li).view(T, H * D), L["o"], resid=resid, ss_out=ss_o, decode=dec)
                linear(resid, L["gate_up"], act, norm_w=L["ln2"], ss_in=ss_o, eps=eps, swiglu=True, decode=dec)
                linear(act, L["down"], resid=resid, ss_out=ss_d, decode=dec)
            rms_norm(resid, self.norm, eps, h)
        elif (splits := self._wide_splits(T)) is not None:
            # a few sequences' rows at wide hidden sizes: the weight-streaming
            # kernel, whose split reductions the next kernel sums (8 launches
            # per layer)
            s_qkv, s_o, s_d = splits
            nq = (H + 2 * Hkv) * D
            f32 = dict(dtype=torch.float32, device=self.device)
            part = torch.empty(max((s * n for s, n in ((s_qkv, nq), (s_o, E), (s_d, E)) if s > 1), default=0) * T, **f32)
            qkv = torch.empty(T, nq, dtype=self.dtype, device=self.device)
            act = torch.empty(T, I, dtype=self.dtype, device=self.device)
            x = torch.empty_like(resid)

            def add_norm(splits, weight, residual_out):  # h = rmsnorm(resid + the projection's output)
                if splits > 1:
                    rms_norm_sum(part, splits, weight, eps, h, resid, residual_out)
                else:
                    rms_norm(x, weight, eps, h, residual=resid, residual_out=residual_out)

            for li, L in enumerate(self.layers):
                wide_linear(h, L["qkv"], qkv, part)
                if s_qkv > 1:
                    qk_norm_rope_store_sum(part, s_qkv, L["q_norm"], L["k_norm"], rope_rows, slot_mapping, q,
                                           self.k_caches[li], self.v_caches[li], H, Hkv, D, eps)
                else:
                    qk_norm_rope_store(qkv, L["q_norm"], L["k_norm"], rope_rows, None, slot_mapping, q,
                                       self.k_caches[li], self.v_caches[li], H, Hkv, D, eps)
                wide_linear(attn(li).view(T, H * D), L["o"], x, part)
                add_norm(s_o, L["ln2"], resid)
                wide_linear(h, L["gate_up"], act, swiglu=True)
                wide_linear(act, L["down"], x, part)
                last = li + 1 == len(self.layers)
                add_norm(s_d, self.norm if last else self.layers[li + 1]["ln1"], None if last else resid)
        else:
            # wider batches: hipBLASLt projections between this library's
            # norm / epilogue / SiLU kernels (9 launches per layer)
            act = torch.empty(T, I, dtype=self.dtype, device=self.device)
            for li, L in enumerate(self.layers):
                if li > 0:
                    rms_norm(x, L["ln1"], eps, h, residual=resid, residual_out=resid)
                qkv = F.linear(h, L["qkv"])
                qk_norm_rope_store(qkv, L["q_norm"], L["k_norm"], rope_rows, None, slot_mapping, q,
                                   self.k_caches[li], self.v_caches[li], H, Hkv, D, eps)
                x = F.linear(attn(li).view(T, H * D), L["o"])
                rms_norm(x, L["ln2"], eps, h, residual=resid, residual_out=resid)
                silu_mul(F.linear(h, L["gate_up"]), act)
                x = F.linear(act, L["down"])
            rms_norm(x, self.norm, eps, h, residual=resid)
        if logits_rows is not None:
            h = h.index_select(0, logits_rows)
            T = h.shape[0]
        # the LM head: this library's streaming kernel up to lm_head_rows rows
        # (activations whole in LDS), the weight-streaming kernel on the same
        # packed copy up to WIDE_ROWS, hipBLASLt's large tiles beyond
        if T <= lm_head_rows(E):
            if logits_out is None:
                logits_out = torch.empty(T, self.lm_head.shape[0], dtype=self.dtype, device=self.device)
            if self.lm_head_packed is not None and T <= self.lm_head_packed_rows:
                lm_head(h, self.lm_head_packed, logits_out)
            else:
                linear(h, self.lm_head, logits_out)
            return logits_out
        # (a logits_out that the kernel cannot write, a strided view above all,
        # is left to matmul, which writes it or refuses it)
        V = self.lm_head.shape[0]
        if (self.lm_head_packed is not None and T <= WIDE_ROWS and wide_splits(T, V, E, packed=True)
                and (logits_out is None or dense_bf16(logits_out, T, V, h.device))):
            if logits_out is None:
                logits_out = torch.empty(T, V, dtype=self.dtype, device=self.device)
            wide_linear(h, self.lm_head_packed, logits_out, packed=True)
            return logits_out
        if logits_out is None:
            return F.linear(h, self.lm_head)
        torch.matmul(h, self.lm_head.t(), out=logits_out)
        return logits_out
