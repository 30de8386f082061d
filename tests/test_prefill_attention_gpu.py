"""The prefill attention kernel against the fp64 oracle at the edges of its
tiles: rows around 1, a wave and a tile, keys around a key tile, every head
group form, both head sizes, pages from one token on, unmapped pages, and each
form of the kernel: 4 and 8 waves, whole tiles and tiles cut over keys, paged
and contiguous K/V, block tables longer than LDS holds (each case names the
form it takes)."""

import numpy as np
import pytest
import torch

from gpu_util import assert_close
from naivllm_amd.layers.attention import PrefillPlan, paged_attention_verify, prefill_attention, prefill_tiles
from naivllm_amd.utils import synth
from oracle import attention as ora

pytestmark = pytest.mark.gpu

CASES = [
    # heads, kv heads, head dim, new rows, keys, page
    (2, 1, 128, [1, 31, 33, 63], [1, 31, 64, 65], 16),
    (4, 1, 128, [64, 65, 129], [64, 65, 129], 64),
    (1, 1, 64, [127, 128, 2], [127, 200, 66], 1),
    (3, 1, 64, [40, 257], [90, 257], 32),
    (4, 2, 64, [70], [700], 256),         # cut over keys
    (2, 1, 128, [300, 5], [1800, 2100], 16),  # cut over keys, 8 waves
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_prefill_attention_matches_oracle(case):
    H, Hkv, D, ql, kl, page = CASES[case]
    print(f"case: prefill attention {CASES[case]}", flush=True)
    vb = synth.verify_batch(70 + case, kl, ql, num_heads=H, num_kv_heads=Hkv, head_dim=D, block_size=page)
    bt = vb.block_tables.copy()
    if case == 3:  # an unmapped page inside the context: its keys are not attended
        bt[1, 3] = -1
    f = lambda x: torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda().bfloat16()  # noqa: E731
    plan = PrefillPlan(ql, kl, H, Hkv, page, torch.device("cuda"))
    out = prefill_attention(f(vb.q), f(vb.k_cache), f(vb.v_cache), plan, 1 / np.sqrt(D), D, torch.from_numpy(bt).cuda())
    torch.cuda.synchronize()
    want = ora.verify_attention(vb.q, vb.k_cache, vb.v_cache, bt, vb.context_lens, vb.cu_seqlens_q, vb.positions,
                                1 / np.sqrt(D), H, Hkv)
    assert_close(out, want, "bf16", f"paged {CASES[case]}")
    if ql != kl or case == 3:
        return
    # the same rows from contiguous K/V
    rows = [np.concatenate([c[p] for p in bt[b] if p >= 0])[:n] for c in (vb.k_cache, vb.v_cache)
            for b, n in enumerate(kl)]
    k, v = np.concatenate(rows[:len(kl)]), np.concatenate(rows[len(kl):])
    plan = PrefillPlan(ql, kl, H, Hkv, None, torch.device("cuda"))
    got = prefill_attention(f(vb.q), f(k), f(v), plan, 1 / np.sqrt(D), D)
    torch.cuda.synchronize()
    assert torch.equal(got, out)


def test_both_workgroup_sizes_and_cuts_are_reached():
    rows = {prefill_tiles(ql, kl, H, Hkv, page, 256)[2] * (2 if H // Hkv % 2 == 0 else 1)
            for H, Hkv, _, ql, kl, page in CASES}
    assert rows == {128, 256}
    assert [prefill_tiles(ql, kl, H, Hkv, page, 256)[3] > 0 for H, Hkv, _, ql, kl, page in CASES][-2:] == [True, True]


def make_plan(ql, kl, H, Hkv, page, cus):
    """A plan for a device of ``cus`` compute units (1: no tile is cut)."""
    plan = PrefillPlan(ql, kl, H, Hkv, page, torch.device("cuda"))
    tiles, merges, plan.tile_rows, plan.slots = prefill_tiles(ql, kl, H, Hkv, page, cus)
    plan.ntiles, plan.nmerges = len(tiles), len(merges)
    plan.work = torch.from_numpy(np.concatenate([tiles.ravel(), merges.ravel()])).cuda()
    return plan


FORMS = [
    # waves, heads per workgroup, cut, heads, kv heads, head dim, new rows, keys, page (None: contiguous), unmapped pages
    (8, 2, False, 2, 1, 128, [300, 5], [1800, 2100], 16, []),
    (8, 2, True, 2, 1, 128, [300, 5], [1800, 2100], 16, [(0, 0), (1, 77)]),
    (8, 2, False, 4, 1, 64, [129, 2], [2000, 1537], 32, [(0, 5), (1, 48)]),
    (8, 2, True, 2, 1, 64, [40], [4136], 64, []),
    (8, 1, False, 3, 1, 128, [257], [1900], 16, [(0, 0), (0, 118)]),
    (8, 1, True, 3, 1, 64, [31], [1600], 16, []),
    (8, 2, False, 2, 1, 128, [3150], [3150], None, []),
    (8, 1, False, 1, 1, 64, [3300], [3300], None, []),
    (8, 2, True, 2, 1, 64, [3200], [3200], None, []),
    (4, 2, True, 2, 1, 128, [700], [700], None, []),
    (4, 1, False, 3, 1, 64, [129, 70], [129, 70], None, []),
    # block tables of more entries than LDS holds: two and more turns of the ring
    (8, 2, False, 2, 1, 64, [70], [4700], 1, [(0, 10), (0, 3000), (0, 4699)]),
    (8, 1, False, 1, 1, 128, [33], [3200], 1, [(0, n) for n in range(2100)]),  # the first mapped page past the first turn
    (8, 2, True, 2, 1, 128, [5], [5001], 1, [(0, 4000)]),
    (8, 2, False, 2, 1, 128, [70], [9001], 2, []),
    (4, 2, False, 2, 1, 64, [1, 1, 1], [3000, 64, 65], 1, [(0, 2500)]),
    (4, 1, False, 1, 1, 128, [3, 1, 1], [2600, 64, 65], 1, []),
]


@pytest.mark.parametrize("form", range(len(FORMS)))
def test_every_form_matches_oracle(form):
    waves, hw, cut, H, Hkv, D, ql, kl, page, unmapped = FORMS[form]
    print(f"case: prefill attention form {FORMS[form][:9]}", flush=True)
    plan = make_plan(ql, kl, H, Hkv, page, 256 if cut else 1)
    assert (plan.tile_rows * hw // 32, 2 if H // Hkv % 2 == 0 else 1, plan.slots > 0) == (waves, hw, cut)
    vb = synth.verify_batch(90 + form, kl, ql, num_heads=H, num_kv_heads=Hkv, head_dim=D, block_size=page or 16)
    bt = vb.block_tables.copy()
    for b, i in unmapped:
        bt[b, i] = -1
    f = lambda x: torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda().bfloat16()  # noqa: E731
    k, v = vb.k_cache, vb.v_cache
    if page is None:
        k, v = (np.concatenate([c[[p for p in bt[b] if p >= 0]].reshape(-1, Hkv, D)[:n] for b, n in enumerate(kl)])
                for c in (k, v))
    out = prefill_attention(f(vb.q), f(k), f(v), plan, 1 / np.sqrt(D), D,
                            None if page is None else torch.from_numpy(bt).cuda())
    torch.cuda.synchronize()
    want = ora.verify_attention(vb.q, vb.k_cache, vb.v_cache, bt, vb.context_lens, vb.cu_seqlens_q, vb.positions,
                                1 / np.sqrt(D), H, Hkv)
    assert_close(out, want, "bf16", f"form {FORMS[form][:9]}")


def test_prefill_attention_refuses_bad_shapes():
    plan = PrefillPlan([4], [4], 2, 1, None, torch.device("cuda"))
    q = torch.zeros(4, 2, 128, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(4, 1, 128, device="cuda", dtype=torch.bfloat16)
    for bad in ((q[:3], k, k), (q, k[:3], k[:3]), (q.float(), k, k), (q, k, k[:, :, :64])):
        with pytest.raises(ValueError):
            prefill_attention(*bad, plan, 1.0, 128)


def test_a_plan_serves_other_streams_and_captures():
    # built on one stream while work is queued there, used at once on another,
    # then inside a capture (its own stream), replayed twice
    print("case: prefill plan on other streams", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(200, 2, 128, generator=g, device="cuda").bfloat16()
    k, v = (torch.randn(200, 1, 128, generator=g, device="cuda").bfloat16() for _ in range(2))
    want = prefill_attention(q, k, v, PrefillPlan([200], [200], 2, 1, None, q.device), 0.1, 128)
    busy = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for _ in range(8):
        busy.add_(1)
    plan = PrefillPlan([200], [200], 2, 1, None, q.device)
    with torch.cuda.stream(side):
        got = prefill_attention(q, k, v, plan, 0.1, 128)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = prefill_attention(q, k, v, plan, 0.1, 128)
    for _ in range(2):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_rows_at_odd_offsets():
    # contiguous views that start 2 bytes into an allocation give the aligned rows' output
    print("case: prefill attention from views at odd offsets", flush=True)
    g = torch.Generator(device="cuda").manual_seed(4)
    base = torch.randn(3, 150 * 2 * 128 + 1, generator=g, device="cuda").bfloat16()
    q, k, v = (b[1:].view(150, -1, 128)[:, :n].contiguous() for b, n in zip(base, (2, 1, 1)))
    plan = PrefillPlan([150], [150], 2, 1, None, q.device)
    want = prefill_attention(q, k, v, plan, 0.1, 128)
    odd = []
    for t in (q, k, v):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        flat[1:].copy_(t.reshape(-1))
        odd.append(flat[1:].view(t.shape))
        assert odd[-1].data_ptr() % 16 == 2
    assert torch.equal(prefill_attention(*odd, plan, 0.1, 128), want)


@pytest.mark.parametrize("new,keys", [(40, 296), (270, 526), (300, 1324), (1000, 1000)])
def test_prefill_is_no_less_precise_than_verify(new, keys):
    # error against 64 bits beside that of the verify kernel over causal blocks
    # of 64 / G rows: both round each weight to bf16 once, and a weight at its
    # exponent reference not at all, so the kernel with fewer references per
    # row is further off (one lazily moved reference: 5 to 12 percent); a
    # permille is the spread of equal counts
    print(f"case: prefill precision, {new} rows of {keys} keys", flush=True)
    H, Hkv, D, page = 16, 8, 128, 64
    g = torch.Generator(device="cuda").manual_seed(keys)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    npg, block = -(-keys // page), 64 // (H // Hkv)
    q, k, v = rand(new, H, D), rand(npg, page, Hkv, D), rand(npg, page, Hkv, D)
    bt = torch.arange(npg, dtype=torch.int32, device="cuda")[None]
    first = list(range(keys - new, keys, block))
    ends = [min(keys, b + block) for b in first]
    pos = torch.arange(keys - new, keys, device="cuda")
    blocks = paged_attention_verify(
        q, k, v, bt.repeat(len(ends), 1), torch.tensor(ends, device="cuda"),
        torch.tensor([0] + [e - keys + new for e in ends], dtype=torch.int32, device="cuda"), pos, D ** -0.5, H, Hkv, D,
        page, block, max_q_len=block)
    got = prefill_attention(q, k, v, PrefillPlan([new], [keys], H, Hkv, page, q.device), D ** -0.5, D, bt)
    kd, vd = (t.double().view(npg * page, Hkv, D)[:keys].permute(1, 0, 2).repeat_interleave(H // Hkv, 0) for t in (k, v))
    s = torch.matmul(q.double().permute(1, 0, 2), kd.transpose(1, 2).contiguous()) * D ** -0.5
    s.masked_fill_(torch.arange(keys, device="cuda")[None] > pos[:, None], -float("inf"))
    want = torch.matmul(s.softmax(-1), vd.contiguous()).permute(1, 0, 2)
    err = [((x.double() - want).norm() / want.norm()).item() for x in (got, blocks)]
    assert err[0] <= 1.005 * err[1], err
