"""GPU parity of the verify-attention and KV-store kernels against the CPU
oracle, through the reference-signature wrappers (which call the C ABI)."""

import numpy as np
import pytest
import torch

from naivllm_amd.layers.attention import paged_attention_verify, store_kvcache, verify_attention_plan
from naivllm_amd.utils import synth
from oracle import attention as ora
from tests.gpu_util import assert_close, to_device

pytestmark = pytest.mark.gpu


def _gpu(vb, block_m=16, **kw):
    t = to_device(vb)
    out = paged_attention_verify(t["query"], t["k_cache"], t["v_cache"], t["block_tables"], t["context_lens"],
                                 t["cu_seqlens_q"], t["positions"], 1.0 / np.sqrt(vb.head_dim), vb.num_heads,
                                 vb.num_kv_heads, vb.head_dim, vb.block_size, block_m, **kw)
    torch.cuda.synchronize()
    return out


def _kernel(vb, max_q_len):
    """The kernel the plan runs for this batch on the current device."""
    dtype = torch.float32 if vb.dtype == "f32" else torch.bfloat16
    return verify_attention_plan(len(vb.context_lens), vb.num_heads, vb.num_kv_heads, vb.head_dim, vb.block_size,
                                 vb.block_tables.shape[1], max_q_len, dtype)[0]


def _oracle(vb):
    return ora.verify_attention(vb.q, vb.k_cache, vb.v_cache, vb.block_tables, vb.context_lens, vb.cu_seqlens_q,
                                vb.positions, 1.0 / np.sqrt(vb.head_dim), vb.num_heads, vb.num_kv_heads)


def _live_rows(vb):
    return vb.positions >= 0


def test_config1_fp32():
    print("case: config1 fp32 b1 L=1248", flush=True)
    vb = synth.config1_batch()
    out = _gpu(vb, max_q_len=9)
    assert_close(out, _oracle(vb), "f32", "config1")


def test_config2_bf16():
    print("case: config2 bf16 b8", flush=True)
    vb = synth.config2_batch()
    out = _gpu(vb, max_q_len=9)
    assert_close(out, _oracle(vb), "bf16", "config2")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("split", [128, 256, 1024])
def test_split_sizes_agree_with_oracle(dtype, split):
    print(f"case: splits dtype={dtype} split={split}", flush=True)
    vb = synth.verify_batch(21, [700, 129, 1], [9, 3, 1], dtype=dtype, block_size=64)
    out = _gpu(vb, max_q_len=9, kv_split_tokens=split)
    assert_close(out, _oracle(vb), dtype, f"split {split}")


@pytest.mark.parametrize("dtype,ctx,max_blocks,kernel", [("bf16", [1500], None, "d-sliced"), ("f32", [900, 1500], None, "fp32"),
                                                        ("bf16", [900, 1500], None, "key-split"),
                                                        ("bf16", [900, 1500], 24, "key-split")])
def test_gqa4_8b_shape(dtype, ctx, max_blocks, kernel):
    # 36 rows of the 4-head group: three 16-row m-tiles (one sequence's 8
    # pairs take the d-sliced kernel, two sequences the key-split kernel)
    print(f"case: 32Q/8KV dtype={dtype} ctx={ctx} max_blocks={max_blocks}", flush=True)
    vb = synth.verify_batch(22, ctx, [9] * len(ctx), num_heads=32, num_kv_heads=8, dtype=dtype, max_blocks=max_blocks)
    assert _kernel(vb, 9) == kernel
    out = _gpu(vb, max_q_len=9)
    assert_close(out, _oracle(vb), dtype, "gqa4")


@pytest.mark.parametrize("dtype,max_blocks,G,ql,Hkv,kernel",
                         [("bf16", None, 4, 17, 4, "d-sliced"), ("bf16", 24, 4, 17, 8, "key-split"),
                          ("f32", None, 4, 17, 8, "fp32"), ("bf16", None, 8, 9, 4, "d-sliced"),
                          ("bf16", 24, 8, 9, 8, "key-split"), ("f32", None, 8, 9, 8, "fp32")])
def test_groups_beyond_64_rows(dtype, max_blocks, G, ql, Hkv, kernel):
    # (H / Hkv) * max_q_len > 64 rows: GQA-4 with K = 16 drafts (68 rows)
    # and GQA-8 with K = 8 (72 rows) run as launches over subsets of each
    # kv head's query heads (2 of 4, 4 of 8), through the d-sliced kernel
    # (8 pairs), the key-split kernel and the fp32 kernel; the second
    # sequence is ragged and carries padding rows
    print(f"case: {G * Hkv}Q/{Hkv}KV {ql} rows per sequence, dtype={dtype} max_blocks={max_blocks}", flush=True)
    vb = synth.verify_batch(23, [1100, 1500], [ql, ql - 3], num_heads=G * Hkv, num_kv_heads=Hkv, dtype=dtype,
                            max_blocks=max_blocks, pad_rows=[0, 2])
    assert _kernel(vb, ql) == kernel
    out = _gpu(vb, max_q_len=ql)
    assert_close(out, _oracle(vb), dtype, f"{G} heads x {ql} rows")


@pytest.mark.parametrize("max_blocks,kernel", [(None, "d-sliced"), (16, "key-split")])
def test_small_batch_many_key_splits(max_blocks, kernel):
    # few (sequence, kv head) pairs (4 x 2): each context is cut into many
    # short splits (some sequences shorter than one split per CU share); a
    # 5-page table takes the d-sliced kernel and its merge kernel, a 16-page
    # table (4096 keys) the key-split kernel and its in-kernel merge
    print(f"case: b4 bf16 short and long contexts, max_blocks={max_blocks}", flush=True)
    vb = synth.verify_batch(27, [1, 17, 300, 1248], [1, 9, 9, 9], num_heads=4, num_kv_heads=2, dtype="bf16",
                            max_blocks=max_blocks)
    assert _kernel(vb, 9) == kernel
    out = _gpu(vb, max_q_len=9)
    assert_close(out, _oracle(vb), "bf16", "many splits")


def test_workspace_reuse_across_shapes():
    # calls of different batch sizes (different split plans and partial
    # layouts) share one workspace; the key-split merge's arrival counters
    # must come back to zero after each
    print("case: workspace reuse b8 -> b24 -> b2 -> b8", flush=True)
    batches = [(8, 30), (24, 31), (2, 32), (8, 30)]
    for batch, seed in batches:
        ctx = [int(x) for x in synth.randint(seed, 1, batch, 100, 900)]
        # 64-page tables (4096 keys): the key-split kernel
        vb = synth.verify_batch(seed, ctx, [9] * batch, dtype="bf16", block_size=64, max_blocks=64)
        out = _gpu(vb, max_q_len=9)
        assert_close(out, _oracle(vb), "bf16", f"reuse b{batch}")


@pytest.mark.parametrize("batch,bs,qlen,kernel", [(16, 256, 9, "key-split"), (32, 16, 9, "key-split"),
                                                 (20, 64, 5, "key-split"), (16, 8, 9, "d-sliced")])
def test_wide_batches(batch, bs, qlen, kernel):
    # >= 128 (sequence, kv head) pairs: the key-split kernel with one split
    # per pair; pages below 16 keys take the d-sliced kernel, which fills the
    # chip with two 64-dim slices per pair (the 32-dim slicing of smaller
    # batches is covered above)
    print(f"case: wide batch={batch} block_size={bs} q_len={qlen}", flush=True)
    ctx = [int(x) for x in synth.randint(26, batch, batch, 40, 700)]
    vb = synth.verify_batch(26 + batch, ctx, [qlen] * batch, block_size=bs, dtype="bf16")
    assert _kernel(vb, qlen) == kernel
    out = _gpu(vb, max_q_len=qlen)
    assert_close(out, _oracle(vb), "bf16", f"wide b{batch}")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_block_m_bound_without_max_q_len(dtype):
    # the reference only passes block_m (>= every q_len); rows are then laid
    # out with a 16-row stride per head, the result must not change
    print(f"case: block_m only dtype={dtype}", flush=True)
    vb = synth.verify_batch(23, [300, 260], [9, 6], num_heads=8, num_kv_heads=2, dtype=dtype)
    out = _gpu(vb, block_m=16)
    assert_close(out, _oracle(vb), dtype, "block_m")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_ragged_pad_rows_holes_and_empty_sequences(dtype):
    print(f"case: ragged dtype={dtype}", flush=True)
    vb = synth.verify_batch(24, [300, 0, 77, 513], [9, 9, 2, 9], num_heads=16, num_kv_heads=8, block_size=32,
                            dtype=dtype, pad_rows=[3, 9, 0, 0])
    vb.block_tables[3, 2] = -1  # unmapped page inside a context
    out = _gpu(vb, max_q_len=9, kv_split_tokens=128)
    want = _oracle(vb)
    assert_close(out, want, dtype, "ragged")
    pad = ~_live_rows(vb)
    assert torch.all(out[torch.from_numpy(pad).cuda()] == 0)


@pytest.mark.parametrize("num_heads", [2, 4, 8])
def test_key_split_head_dim_64(num_heads):
    # head_dim 64 through the key-split kernel (a fixed split length selects
    # it): GQA groups 1, 2 and 4 over 2 kv heads give 1, 2 and 3 query
    # m-tiles; a 64-dim row is 8 chunks of the LDS swizzle, not 16
    print(f"case: key-split head_dim=64 H={num_heads} Hkv=2", flush=True)
    vb = synth.verify_batch(29, [517, 33, 260], [9, 4, 9], num_heads=num_heads, num_kv_heads=2, head_dim=64,
                            block_size=32, dtype="bf16")
    out = _gpu(vb, max_q_len=9, kv_split_tokens=128)
    assert_close(out, _oracle(vb), "bf16", f"ks d64 H{num_heads}")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("bs", [4, 16])
def test_small_pages(dtype, bs):
    print(f"case: block_size={bs} dtype={dtype}", flush=True)
    vb = synth.verify_batch(25, [131, 40], [5, 9], num_heads=4, num_kv_heads=2, head_dim=64, block_size=bs,
                            dtype=dtype)
    out = _gpu(vb, max_q_len=9)
    assert_close(out, _oracle(vb), dtype, f"bs {bs}")


def test_golden_fixture_fp32():
    import json
    import os
    c = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "attention_tiny.json")))
    # the fixture's head_dim 4 is below the kernels' minimum; embed it in
    # head_dim 64 with zero padding, which leaves every dot product unchanged
    pad = lambda x: np.concatenate([np.array(x), np.zeros(np.array(x).shape[:-1] + (60,))], axis=-1)
    vb = synth.VerifyBatch(pad(c["q"]), pad(c["k_cache"]), pad(c["v_cache"]), np.array(c["block_tables"], np.int32),
                           np.array(c["context_lens"], np.int64), np.array(c["cu_seqlens_q"], np.int32),
                           np.array(c["positions"], np.int64), 4, 2, 64, 4, "f32")
    t = to_device(vb)
    out = paged_attention_verify(t["query"], t["k_cache"], t["v_cache"], t["block_tables"], t["context_lens"],
                                 t["cu_seqlens_q"], t["positions"], c["scale"], 4, 2, 64, 4, 16)
    want = pad(c["expected"])
    assert_close(out, want, "f32", "golden")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_store_kvcache_matches_oracle(dtype):
    print(f"case: store_kv dtype={dtype}", flush=True)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    T, Hkv, D, nb, bs = 20, 8, 128, 6, 16
    key = torch.randn(T, Hkv, D, dtype=dt, device="cuda")
    val = torch.randn(T, Hkv, D, dtype=dt, device="cuda")
    kc = torch.randn(nb, bs, Hkv, D, dtype=dt, device="cuda")
    vc = torch.randn(nb, bs, Hkv, D, dtype=dt, device="cuda")
    slots = torch.tensor(synth.randperm(3, 0, nb * bs)[:T], dtype=torch.int64)
    slots[::5] = -1
    kc_ref, vc_ref = kc.float().cpu().numpy(), vc.float().cpu().numpy()
    ora.store_kvcache(key.float().cpu().numpy(), val.float().cpu().numpy(), kc_ref, vc_ref, slots.numpy())
    store_kvcache(key, val, kc, vc, slots.cuda(), bs)
    torch.cuda.synchronize()
    assert np.array_equal(kc.float().cpu().numpy(), kc_ref)
    assert np.array_equal(vc.float().cpu().numpy(), vc_ref)


@pytest.mark.parametrize("split", [128, 384])
def test_repeated_calls_share_the_workspace(split):
    # calls reuse one partials workspace: repeat the call (eagerly and under
    # graph replay) and check each result
    print(f"case: repeated split={split}", flush=True)
    vb = synth.config2_batch()
    want = _oracle(vb)
    t = to_device(vb)
    args = (t["query"], t["k_cache"], t["v_cache"], t["block_tables"], t["context_lens"], t["cu_seqlens_q"],
            t["positions"], 1.0 / np.sqrt(128), 16, 8, 128, 256, 16)
    for _ in range(3):
        out = paged_attention_verify(*args, max_q_len=9, kv_split_tokens=split)
        torch.cuda.synchronize()
        assert_close(out, want, "bf16", f"eager split {split}")
    out = torch.empty_like(t["query"])
    paged_attention_verify(*args, max_q_len=9, kv_split_tokens=split, out=out)  # workspace allocated
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        paged_attention_verify(*args, max_q_len=9, kv_split_tokens=split, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert_close(out, want, "bf16", f"graph split {split}")


@pytest.mark.parametrize("G,ql,D,bs", [(1, 1, 128, 1), (2, 9, 128, 16), (4, 9, 64, 4), (4, 12, 128, 256), (4, 16, 64, 64),
                                       (4, 16, 128, 16)])
def test_fp32_tile_edges(G, ql, D, bs):
    # one to four row tiles of the fp32 kernel, contexts around a 16-key tile,
    # a 64-key split and a turn of its four waves, an unmapped page
    print(f"case: fp32 {G} heads x {ql} rows, D={D} page={bs}", flush=True)
    ctx = [max(ql, n) for n in (1, 15, 16, 17, 63, 64, 65, 129, 321)]
    vb = synth.verify_batch(41, ctx, [min(ql, n) for n in ctx], num_heads=2 * G, num_kv_heads=2, head_dim=D,
                            block_size=bs, dtype="f32")
    if bs <= 64:
        vb.block_tables[8, 2] = -1
    out = _gpu(vb, max_q_len=ql)
    assert_close(out, _oracle(vb), "f32", "fp32 edges")


@pytest.mark.parametrize("G,ql", [(2, 1), (2, 9), (4, 9)])
def test_split_counts_follow_the_context(G, ql):
    # a 10k-key table plans more than 8 splits; the kernel counts a context's
    # splits by its own length: the lengths around each change of the rule,
    # for one, two and three row tiles, short and long contexts in one call
    print(f"case: splits by context, {G} heads x {ql} rows", flush=True)
    ctx = [9, 100, 200, 201, 320, 321, 512, 513, 4607, 4608, 5121, 1250]
    vb = synth.verify_batch(43, ctx, [ql] * len(ctx), num_heads=2 * G, num_kv_heads=2, dtype="bf16", max_blocks=40)
    assert _kernel(vb, ql) == "key-split"
    out = _gpu(vb, max_q_len=ql)
    assert_close(out, _oracle(vb), "bf16", "splits by context")


@pytest.mark.parametrize("rows,ctx", [(9, 300), (2, 150), (9, 1250), (9, 4000)])
def test_fewer_splits_are_no_less_precise(rows, ctx):
    # a table much wider than the context: the splits are counted by the
    # context, and the error against 64 bits stays that of splits whose waves
    # take one 16-key tile each (every tile its own exponent reference).  The
    # same references give the same rounding up to the splits' merge order, a
    # few permille; one reference per wave gives 3 to 15 percent more.
    print(f"case: verify attention precision rows={rows} ctx={ctx}", flush=True)
    H, Hkv, D, page, width = 16, 8, 128, 64, 520
    g = torch.Generator(device="cuda").manual_seed(ctx + rows)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    B, npg = 1, -(-ctx // page)  # 8 pairs: the plan takes 32 splits of such a table
    q, k, v = rand(B * rows, H, D), rand(B * npg, page, Hkv, D), rand(B * npg, page, Hkv, D)
    bt = torch.full((B, width), -1, dtype=torch.int32)
    bt[:, :npg] = torch.arange(B * npg, dtype=torch.int32).view(B, npg)
    lens = torch.full((B,), ctx, dtype=torch.int64, device="cuda")
    cu = torch.arange(0, B * rows + 1, rows, dtype=torch.int32, device="cuda")
    pos = torch.arange(ctx - rows, ctx, device="cuda").repeat(B)
    run = lambda split: paged_attention_verify(  # noqa: E731
        q, k, v, bt.cuda(), lens, cu, pos, D ** -0.5, H, Hkv, D, page, 16, max_q_len=rows, kv_split_tokens=split).double()
    kd, vd = (t.double().view(B, npg * page, Hkv, D)[:, :ctx].permute(0, 2, 1, 3).repeat_interleave(H // Hkv, 1)
              for t in (k, v))
    s = torch.matmul(q.double().view(B, rows, H, D).permute(0, 2, 1, 3), kd.transpose(2, 3).contiguous()) * D ** -0.5
    s.masked_fill_(torch.arange(ctx, device="cuda")[None] > pos[:rows, None], -float("inf"))
    want = torch.matmul(s.softmax(-1), vd.contiguous()).permute(0, 2, 1, 3).reshape(B * rows, H, D)
    assert verify_attention_plan(B, H, Hkv, D, page, width, rows, torch.bfloat16)[0] == "key-split"
    err = [((run(split) - want).norm() / want.norm()).item() for split in (0, 128)]
    assert err[0] <= 1.01 * err[1], err
