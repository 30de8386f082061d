"""The prefill attention kernel against the fp64 oracle at the edges of its
tiles: rows around 1, a wave and a tile, keys around a key tile, every head
group form, both head sizes, pages from one token on, unmapped pages, tiles
cut over keys, and both workgroup sizes."""

import numpy as np
import pytest
import torch

from gpu_util import assert_close
from naivllm_amd.layers.attention import PrefillPlan, prefill_attention, prefill_tiles
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
