"""The weight-streaming projections (nsv_wide_linear) and the kernels that sum
their split reductions, against fp32/fp64 torch references at the edges of
their dispatch: row tiles, column remainders, odd and even chunk counts, every
workgroup form."""

import pytest
import torch
import torch.nn.functional as F

import naivllm_amd.layers.qwen3 as qm
from naivllm_amd import _lib

pytestmark = pytest.mark.gpu

# one bf16 rounding of the output, and sums of up to K products in fp32
BF16 = dict(rtol=1e-2, atol=2e-2)


def randn(seed, *shape, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(torch.bfloat16)


def product(x, w):
    return x.double() @ w.double().t().contiguous()


# N, K: 64 columns unsplit (odd chunks), split with a column remainder, 128
# columns split (odd ranges) and unsplit
@pytest.mark.parametrize("M", [1, 13, 17, 33, 49, 65, 80, 81, 97, 113, 128])
@pytest.mark.parametrize("N,K", [(1040, 256), (16400, 768), (1040, 2048), (8208, 2560), (33024, 1280)])
def test_wide_linear_plain(M, N, K):
    splits = qm.wide_splits(M, N, K)
    print(f"case: wide linear M={M} N={N} K={K} splits={splits}", flush=True)
    x, w = randn(M + N, M, K), randn(K + 1, N, K, scale=K ** -0.5)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    part = torch.full((max(splits, 1), M, N), float("nan"), device="cuda")
    qm.wide_linear(x, w, y, part)
    got = part.double().sum(0) if splits > 1 else y.double()
    torch.testing.assert_close(got, product(x, w), **BF16)
    if splits > 1:
        assert y.isnan().all()  # the consumer sums the partials; y is not touched


# reductions of 11 and 38 chunks, which no even split cuts finely enough: 64
# columns (ranges of 2 and 3 chunks) and 128 columns (3 and 4)
@pytest.mark.parametrize("M", [1, 17, 128])
@pytest.mark.parametrize("N,K,splits", [(1040, 2816, 5), (2560, 9728, 12)])
def test_wide_linear_uneven_splits(M, N, K, splits):
    assert qm.wide_splits(M, N, K) == splits
    print(f"case: wide linear M={M} N={N} K={K} uneven splits={splits}", flush=True)
    x, w = randn(M + N, M, K), randn(K + 1, N, K, scale=K ** -0.5)
    part = torch.full((splits, M, N), float("nan"), device="cuda")
    qm.wide_linear(x, w, None, part)
    torch.testing.assert_close(part.double().sum(0), product(x, w), **BF16)


def test_wide_linear_plan_covers_its_forms():
    assert [qm.wide_splits(72, N, K) for N, K in ((1040, 256), (1040, 2048), (8208, 2560), (33024, 1280))] == [1, 4, 2, 1]
    assert qm.wide_splits(129, 1024, 1024) == qm.wide_splits(8, 1024, 1000) == qm.wide_splits(8, 1000, 1024) == 0


# gate columns per workgroup: 16 (up to one slot per CU), 48 and 64 (rows past 80), with remainders
@pytest.mark.parametrize("M", [1, 17, 80, 81, 128])
@pytest.mark.parametrize("I,K", [(16, 256), (1040, 768), (4112, 512), (4176, 1024)])
def test_wide_linear_swiglu(M, I, K):
    print(f"case: wide linear swiglu M={M} I={I} K={K}", flush=True)
    x, w = randn(M + I, M, K), randn(K + 2, 2 * I, K, scale=K ** -0.5)
    y = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    qm.wide_linear(x, w, y, swiglu=True)
    gu = product(x, w).to(torch.bfloat16).float()
    torch.testing.assert_close(y.float(), F.silu(gu[:, :I]) * gu[:, I:], **BF16)


# 48 columns would take a second turn of workgroups and 64 do not (769 and 1024
# slots of 16), or both do (1025)
@pytest.mark.parametrize("M", [1, 80])
@pytest.mark.parametrize("I", [12304, 16384, 16400])
def test_wide_linear_swiglu_turns(M, I):
    print(f"case: wide linear swiglu M={M} I={I}", flush=True)
    x, w = randn(M + I, M, 256), randn(3, 2 * I, 256, scale=1 / 16)
    y = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    qm.wide_linear(x, w, y, swiglu=True)
    gu = product(x, w).to(torch.bfloat16).float()
    torch.testing.assert_close(y.float(), F.silu(gu[:, :I]) * gu[:, I:], **BF16)


@pytest.mark.parametrize("M", [2, 20, 72, 100, 128])
@pytest.mark.parametrize("N,K", [(160, 1024), (32976, 1024), (33088, 2048)])
def test_wide_linear_packed(M, N, K):
    # fewer column groups than CUs, and several groups per workgroup with a partial last one
    print(f"case: wide linear packed M={M} N={N} K={K}", flush=True)
    x, w = randn(M + N, M, K), randn(K + 3, N, K, scale=K ** -0.5)
    packed = torch.empty_like(w)
    assert _lib.lib().nsv_lm_head_pack(w.data_ptr(), packed.data_ptr(), N, K, _lib.stream_ptr(w.device)) == 0
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    qm.wide_linear(x, packed, y, packed=True)
    torch.testing.assert_close(y.double(), product(x, w), **BF16)


@pytest.mark.parametrize("splits", [2, 4, 5, 12])
@pytest.mark.parametrize("T,E", [(3, 1024), (17, 2056), (2, 4096)])
def test_rms_norm_of_a_sum(splits, T, E):
    print(f"case: rms_norm_sum T={T} E={E} splits={splits}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(splits + E)
    part = torch.randn(splits, T, E, generator=g, device="cuda")
    res, w = randn(5, T, E), randn(6, E)
    out, res_out = torch.empty_like(res), torch.empty_like(res)
    qm.rms_norm_sum(part, splits, w, 1e-6, out, res, res_out)
    x = part[0].clone()
    for s in range(1, splits):
        x += part[s]  # split order
    want, want_res = torch.empty_like(res), torch.empty_like(res)
    qm.rms_norm(x.to(torch.bfloat16), w, 1e-6, want, residual=res, residual_out=want_res)
    assert torch.equal(res_out, want_res)
    torch.testing.assert_close(out.float(), want.float(), **BF16)  # the row sum's order differs


@pytest.mark.parametrize("splits", [2, 8, 9])
def test_qk_norm_rope_store_of_a_sum(splits):
    print(f"case: qk_norm_rope_store_sum splits={splits}", flush=True)
    T, H, Hkv, D = 5, 4, 2, 128
    g = torch.Generator(device="cuda").manual_seed(splits)
    part = torch.randn(splits, T, (H + 2 * Hkv) * D, generator=g, device="cuda")
    x = part[0].clone()
    for s in range(1, splits):
        x += part[s]
    qw, kw = randn(1, D), randn(2, D)
    rope = torch.randn(T, D, generator=g, device="cuda")
    slots = torch.tensor([3, -1, 0, 17, 9], dtype=torch.int64, device="cuda")
    got = [torch.zeros(T, H, D, dtype=torch.bfloat16, device="cuda")] + [
        torch.zeros(2, 16, Hkv, D, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    want = [t.clone() for t in got]
    qm.qk_norm_rope_store_sum(part, splits, qw, kw, rope, slots, *got, H, Hkv, D, 1e-6)
    qm.qk_norm_rope_store(x.to(torch.bfloat16), qw, kw, rope, None, slots, *want, H, Hkv, D, 1e-6)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_head_writes_or_refuses_the_callers_logits():
    # 96 rows at hidden 1024: past the streaming head's rows, on the packed copy
    print("case: logits_out of the wide head", flush=True)
    cfg = qm.Qwen3Config(vocab_size=131072, hidden_size=1024, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=64,
                         intermediate_size=512, max_position=256)
    model = qm.Qwen3Verify(cfg, "cuda", seed=3)
    model.allocate_kv_cache(8, 16)
    T, V = 96, cfg.vocab_size
    assert qm.lm_head_rows(1024) < T and model.lm_head_packed is not None
    i64 = dict(dtype=torch.int64, device="cuda")
    pos = torch.arange(T, **i64)
    bt = torch.arange(8, dtype=torch.int32, device="cuda")[None]
    plan = qm.PrefillPlan([T], [T], 4, 2, 16, torch.device("cuda"))
    run = lambda out: model.forward(pos % 50, pos, pos, bt, None, None, 0, logits_out=out, prefill=plan)  # noqa: E731
    want = run(None)
    dense = torch.empty(T, V, dtype=torch.bfloat16, device="cuda")
    assert run(dense) is dense and torch.equal(dense, want)
    wide = torch.full((T, V + 64), 7.0, dtype=torch.bfloat16, device="cuda")
    got = run(wide[:, :V])  # rows V + 64 apart
    torch.testing.assert_close(got.float(), want.float(), **BF16)
    torch.testing.assert_close(wide[:, :V].float(), want.float(), **BF16)
    assert (wide[:, V:] == 7.0).all()
    with pytest.raises(RuntimeError):
        run(torch.empty(T, V, device="cuda"))  # fp32
