"""The work a user of this framework has it do, as measurable cases.

A case is a dict of plain values.  ``prepare`` makes what a serving program
holds before a call (models with their weights, paged caches, plans and
captured graphs, inputs drawn from the seed), ``run`` makes one pass through
the public entry points and returns what they return, ``exact`` computes the
same values in 64 bits with plain torch.

Kinds of cases and what each stands for:
  verify_attention   the paged attention of a verify round (drafts + 1 query
                     rows per sequence; drafts 0 is a plain decode step), over
                     the distinct caches of several layers, captured in a
                     hipGraph as the engine's rounds are
  prefill_attention  an Attention layer of a prefill step: the step's K/V
                     stored, then every new row attends causally, from the
                     step's own keys (prefix 0) or from paged keys behind a
                     cached prefix
  verify             ModelRunner.run_spec_verify: host sequences with their
                     drafts in, the target's logits of every verify row out
  prefill            Qwen3Verify.prefill: token lists in, last-row logits out
  accept             acceptance of a round's drafts over the full vocabulary,
                     greedy or stochastic
  ngram              prompt-lookup drafting over token histories
"""

from __future__ import annotations

import math
import random

import torch

from naivllm_amd.engine.model_runner import ModelRunner
from naivllm_amd.engine.sequence import Sequence
from naivllm_amd.layers.attention import Attention, paged_attention_verify
from naivllm_amd.layers.qwen3 import Qwen3Config, Qwen3Verify
from naivllm_amd.spec_engine.drafters import ngram_draft
from naivllm_amd.spec_engine.rejection_sampler import accept_greedy, accept_stochastic
from naivllm_amd.utils.context import reset_context, set_context

DEVICE = "cuda"
VOCAB = 151936
HEAD_DIM = 128
KV_HEADS = 8
# query heads, hidden size and intermediate size of the two Qwen3 shapes
SHAPES = {"0.6b": (16, 1024, 3072), "8b": (32, 4096, 12288)}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed() -> list[dict]:
    return [
        # one layer kind of the 0.6B verify round at 8 sequences, ~1.25k keys (a RAG document's round)
        dict(name="verify_attention_b8", kind="verify_attention", model="0.6b", batch=8, drafts=8, ctx_lo=1200,
             ctx_hi=1300, page=256, layers=28, dtype="bf16"),
        # long-context serving of the 8B model: 16 sequences of 16k to 32k keys
        dict(name="verify_attention_8b_long", kind="verify_attention", model="8b", batch=16, drafts=8, ctx_lo=16384,
             ctx_hi=32768, page=256, layers=2, dtype="bf16"),
        # the fp32 parity path at one sequence
        dict(name="verify_attention_b1_f32", kind="verify_attention", model="0.6b", batch=1, drafts=8, ctx_lo=1248,
             ctx_hi=1248, page=256, layers=8, dtype="f32"),
        # eight uneven prompts prefilled together, nothing cached
        dict(name="prefill_attention_b8", kind="prefill_attention", model="0.6b", batch=8, new_lo=700, new_hi=1300,
             prefix=0, page=256, layers=4),
        # two long 8B prompts behind a cached prefix
        dict(name="prefill_attention_8b_prefix", kind="prefill_attention", model="8b", batch=2, new_lo=2900,
             new_hi=4100, prefix=4096, page=256, layers=2),
        # the whole 0.6B verify forward for one request, the round's latency case
        dict(name="verify_b1", kind="verify", model="0.6b", batch=1, drafts=8, ctx_lo=1206, ctx_hi=1254, page=256,
             layers=28),
        # the same forward at eight requests, four of its layers and the head
        dict(name="verify_b8", kind="verify", model="0.6b", batch=8, drafts=8, ctx_lo=1200, ctx_hi=1300, page=256,
             layers=4),
        # the 8B target of a cascade at eight requests, two layers and the head
        dict(name="verify_8b_b8", kind="verify", model="8b", batch=8, drafts=8, ctx_lo=1200, ctx_hi=1300, page=256,
             layers=2),
        # time to first token of one RAG prompt, four layers and the head
        dict(name="prefill_b1", kind="prefill", model="0.6b", batch=1, new_lo=1206, new_hi=1206, prefix=0, page=256,
             layers=4),
        # rejection sampling of eight model drafts in each of eight sequences
        dict(name="accept_stochastic_b8", kind="accept", batch=8, drafts=8, mode="model", dtype="bf16"),
        # the smallest call: one sequence's drafts against its argmax rows
        dict(name="accept_greedy_b1", kind="accept", batch=1, drafts=8, mode="greedy", dtype="bf16"),
        # drafts for eight sequences with histories up to the longest contexts served
        dict(name="ngram_b8_long", kind="ngram", batch=8, drafts=8, min_n=2, max_n=8, ctx_lo=1200, ctx_hi=32768),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    """One more case of the listed cases' ranges."""
    kind = rng.choice(["verify_attention", "verify_attention", "prefill_attention", "prefill_attention", "verify",
                       "prefill", "accept", "ngram"])
    model = rng.choice(["0.6b", "8b"])
    if kind == "verify_attention":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        batch = rng.choice([1, 2, 3, 5, 8, 13, 16])
        hi = _log_int(rng, 120, 32768 if dtype == "bf16" else 4096)
        return dict(kind=kind, model=model, batch=batch, drafts=rng.choice([0, 1, 3, 5, 8, 11]),
                    ctx_lo=max(100, int(hi * rng.uniform(0.4, 1.0))), ctx_hi=hi, page=rng.choice([16, 64, 256]),
                    layers=2, dtype=dtype)
    if kind == "prefill_attention":
        batch = rng.choice([1, 2, 3, 5, 8])
        hi = _log_int(rng, 40, 8192 // batch)
        page = rng.choice([16, 256])
        prefix = page * rng.choice([0, 0, 1, _log_int(rng, 1, 4096 // page)])
        return dict(kind=kind, model=model, batch=batch, new_lo=max(1, int(hi * rng.uniform(0.3, 1.0))), new_hi=hi,
                    prefix=prefix, page=page, layers=2)
    if kind == "verify":
        hi = _log_int(rng, 120, 4096)
        return dict(kind=kind, model=model, batch=rng.choice([1, 2, 3, 4, 6, 8, 12]), drafts=rng.choice([3, 5, 8]),
                    ctx_lo=max(100, int(hi * rng.uniform(0.6, 1.0))), ctx_hi=hi, page=256, layers=2)
    if kind == "prefill":
        batch = rng.choice([1, 2, 4, 8])
        hi = _log_int(rng, 24, 2480 // batch)
        return dict(kind=kind, model=model, batch=batch, new_lo=max(1, int(hi * rng.uniform(0.4, 1.0))), new_hi=hi,
                    prefix=256 * rng.choice([0, 0, 1, 4]), page=256, layers=2)
    if kind == "accept":
        return dict(kind=kind, batch=rng.choice([1, 2, 3, 4, 6, 8]), drafts=rng.randint(1, 11),
                    mode=rng.choice(["greedy", "model", "ngram"]), dtype=rng.choice(["bf16", "bf16", "f32"]))
    hi = _log_int(rng, 200, 32768)
    return dict(kind=kind, batch=rng.choice([1, 2, 4, 8]), drafts=rng.choice([4, 5, 8]), min_n=2,
                max_n=rng.randint(3, 8), ctx_lo=max(100, int(hi * rng.uniform(0.1, 1.0))), ctx_hi=hi)


# ------------------------------------------------------------------ shapes
def _lens(case: dict, lo: str, hi: str) -> list[int]:
    """Uneven lengths of the case's sequences (the case alone decides them)."""
    rng = random.Random(f"{case['batch']} {case[lo]} {case[hi]}")
    return [rng.randint(case[lo], case[hi]) for _ in range(case["batch"])]


def _tables(lens: list[int], page: int, gen: torch.Generator) -> tuple[int, list[list[int]]]:
    """Disjoint pages scattered over a pool a little larger than needed."""
    need = [-(-n // page) for n in lens]
    pool = sum(need) + 3
    order = torch.randperm(pool, generator=gen, device=DEVICE).tolist()
    tables, off = [], 0
    for n in need:
        tables.append(order[off:off + n])
        off += n
    return pool, tables


def _padded(tables: list[list[int]]) -> torch.Tensor:
    width = max(len(t) for t in tables)
    return torch.tensor([t + [-1] * (width - len(t)) for t in tables], dtype=torch.int32, device=DEVICE)


def _slots(table: list[int], first: int, last: int, page: int) -> list[int]:
    return [table[p // page] * page + p % page for p in range(first, last)]


def _normal(gen: torch.Generator, *shape: int, dtype: torch.dtype = torch.bfloat16, scale: float = 1.0):
    """N(0, scale^2) values, drawn in 32 bits."""
    return (torch.randn(*shape, generator=gen, device=DEVICE) * scale).to(dtype)


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _captured(step) -> torch.cuda.CUDAGraph:
    """The step in a hipGraph, run once before, as the engine captures its rounds."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    torch.cuda.synchronize()
    return graph


# ----------------------------------------------------------- the six kinds' inputs
def _verify_attention_inputs(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    heads, rows, page = SHAPES[case["model"]][0], case["drafts"] + 1, case["page"]
    dtype = DTYPES[case["dtype"]]
    ctx = _lens(case, "ctx_lo", "ctx_hi")
    pool, tables = _tables(ctx, page, gen)
    layers = range(case["layers"])
    return dict(
        heads=heads, ctx=ctx, tables=tables, rows=rows,
        q=[_normal(gen, len(ctx) * rows, heads, HEAD_DIM, dtype=dtype) for _ in layers],
        k=[_normal(gen, pool, page, KV_HEADS, HEAD_DIM, dtype=dtype) for _ in layers],
        v=[_normal(gen, pool, page, KV_HEADS, HEAD_DIM, dtype=dtype) for _ in layers])


def _prefill_attention_inputs(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    heads, page, prefix = SHAPES[case["model"]][0], case["page"], case["prefix"]
    new = _lens(case, "new_lo", "new_hi")
    keys = [prefix + n for n in new]
    pool, tables = _tables(keys, page, gen)
    total, layers = sum(new), range(case["layers"])
    return dict(
        heads=heads, new=new, keys=keys, tables=tables,
        q=[_normal(gen, total, heads, HEAD_DIM) for _ in layers],
        k=[_normal(gen, total, KV_HEADS, HEAD_DIM) for _ in layers],
        v=[_normal(gen, total, KV_HEADS, HEAD_DIM) for _ in layers],
        k_cache=[_normal(gen, pool, page, KV_HEADS, HEAD_DIM) for _ in layers],
        v_cache=[_normal(gen, pool, page, KV_HEADS, HEAD_DIM) for _ in layers])


def _config(case: dict) -> Qwen3Config:
    make = Qwen3Config.qwen3_0_6b if case["model"] == "0.6b" else Qwen3Config.qwen3_8b
    return make(num_layers=case["layers"])


def _weights(case: dict, gen: torch.Generator) -> dict:
    """Random weights of the case's layers and its embedding and head."""
    heads, hidden, inter = SHAPES[case["model"]]
    near_one = lambda n: (1 + 0.1 * torch.randn(n, generator=gen, device=DEVICE)).to(torch.bfloat16)  # noqa: E731
    mat = lambda n, k: _normal(gen, n, k, scale=1 / math.sqrt(k))  # noqa: E731
    layers = [dict(ln1=near_one(hidden), qkv=mat((heads + 2 * KV_HEADS) * HEAD_DIM, hidden), q_norm=near_one(HEAD_DIM),
                   k_norm=near_one(HEAD_DIM), o=mat(hidden, heads * HEAD_DIM), ln2=near_one(hidden),
                   gate_up=mat(2 * inter, hidden), down=mat(hidden, inter)) for _ in range(case["layers"])]
    embed = _normal(gen, VOCAB, hidden)
    return dict(layers=layers, embed=embed, norm=near_one(hidden),
                head=embed if case["model"] == "0.6b" else mat(VOCAB, hidden))


def _model_inputs(case: dict, seed: int) -> dict:
    """Weights, filled caches and token lists of a verify or prefill forward;
    rows[i] new rows of sequence i end its tokens."""
    gen = _generator(seed)
    weights = _weights(case, gen)
    if case["kind"] == "verify":
        lens = [n + case["drafts"] for n in _lens(case, "ctx_lo", "ctx_hi")]
        rows = [case["drafts"] + 1] * len(lens)
    else:
        rows = _lens(case, "new_lo", "new_hi")
        lens = [case["prefix"] + n for n in rows]
    pool, tables = _tables(lens, case["page"], gen)
    shape = (pool, case["page"], KV_HEADS, HEAD_DIM)
    k_cache = [_normal(gen, *shape) for _ in range(case["layers"])]
    v_cache = [_normal(gen, *shape) for _ in range(case["layers"])]
    tokens = [torch.randint(VOCAB, (n,), generator=gen, device=DEVICE).tolist() for n in lens]
    return dict(weights=weights, tables=tables, k_cache=k_cache, v_cache=v_cache, tokens=tokens, rows=rows)


def _accept_inputs(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    B, K = case["batch"], case["drafts"]
    dtype = DTYPES[case["dtype"]]
    draft = torch.randn(B, K, VOCAB, generator=gen, device=DEVICE) * 2.0
    target = torch.randn(B, K + 1, VOCAB, generator=gen, device=DEVICE) * 2.0
    target[:, :K] = draft + 0.25 * target[:, :K]
    if case["mode"] == "model":
        drafts = torch.multinomial(torch.softmax(draft, -1).view(-1, VOCAB), 1, generator=gen).view(B, K)
    else:  # drafts that the target's argmax mostly confirms
        drafts = target[:, :K].argmax(-1)
        miss = torch.rand(B, K, generator=gen, device=DEVICE) < 0.2
        drafts = torch.where(miss, torch.randint(VOCAB, (B, K), generator=gen, device=DEVICE), drafts)
    noise_rows = 1 if case["mode"] == "model" else K + 1
    state = dict(
        target=target.to(dtype).view(B * (K + 1), VOCAB), drafts=drafts.to(torch.int32),
        num_drafts=torch.full((B,), K, dtype=torch.int32, device=DEVICE))
    if case["mode"] != "greedy":
        noise = torch.empty(B, noise_rows, VOCAB, device=DEVICE).exponential_(1, generator=gen).to(dtype)
        state.update(draft=draft.to(dtype).view(B * K, VOCAB), uniforms=torch.rand(B, K, generator=gen, device=DEVICE),
                     noise=noise.view(B, VOCAB) if noise_rows == 1 else noise,
                     temperature=torch.ones(B, device=DEVICE))
    return state


def _ngram_inputs(case: dict, seed: int) -> dict:
    """Histories with token frequencies like a text's (few frequent, many
    rare); every second sequence ends quoting a span of its document."""
    gen = _generator(seed)
    lens = _lens(case, "ctx_lo", "ctx_hi")
    history = torch.zeros(len(lens), max(lens) + case["drafts"] + 1, dtype=torch.int32, device=DEVICE)
    for b, n in enumerate(lens):
        u = torch.rand(n, generator=gen, device=DEVICE)
        history[b, :n] = (VOCAB ** u).to(torch.int32).clamp_(max=VOCAB - 1)
        if b % 2:
            at = int(torch.randint(0, n // 2, (1,), generator=gen, device=DEVICE))
            history[b, n - 10:n] = history[b, at:at + 10].clone()
    return dict(history=history, lens=torch.tensor(lens, dtype=torch.int32, device=DEVICE))


# ----------------------------------------------------------------- prepare
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "verify_attention":
        x = _verify_attention_inputs(case, seed)
        rows, ctx = x["rows"], x["ctx"]
        outs = [torch.empty_like(q) for q in x["q"]]
        tables = _padded(x["tables"])
        lens = torch.tensor(ctx, dtype=torch.int64, device=DEVICE)
        cu = torch.arange(0, len(ctx) * rows + 1, rows, dtype=torch.int32, device=DEVICE)
        positions = torch.tensor([p for n in ctx for p in range(n - rows, n)], dtype=torch.int64, device=DEVICE)

        def step():
            for q, k, v, out in zip(x["q"], x["k"], x["v"], outs):
                paged_attention_verify(q, k, v, tables, lens, cu, positions, 1 / math.sqrt(HEAD_DIM), x["heads"],
                                       KV_HEADS, HEAD_DIM, case["page"], 16, max_q_len=rows, out=out)

        return dict(case=case, graph=_captured(step), outs=outs, keep=(x, tables, lens, cu, positions))
    if kind == "prefill_attention":
        x = _prefill_attention_inputs(case, seed)
        layers = []
        for k, v in zip(x["k_cache"], x["v_cache"]):
            layer = Attention(x["heads"], HEAD_DIM, 1.0, KV_HEADS, case["page"])
            layer.k_cache, layer.v_cache = k, v
            layers.append(layer)
        offsets = lambda n: torch.tensor([sum(n[:i]) for i in range(len(n) + 1)], dtype=torch.int32,  # noqa: E731
                                         device=DEVICE)
        slots = [s for t, k, n in zip(x["tables"], x["keys"], x["new"]) for s in _slots(t, k - n, k, case["page"])]
        step = dict(cu_seqlens_q=offsets(x["new"]), cu_seqlens_k=offsets(x["keys"]), max_seqlen_q=max(x["new"]),
                    max_seqlen_k=max(x["keys"]), slot_mapping=torch.tensor(slots, dtype=torch.int64, device=DEVICE),
                    block_tables=_padded(x["tables"]) if case["prefix"] else None, seqlens_q=x["new"],
                    seqlens_k=x["keys"])
        return dict(case=case, x=x, layers=layers, step=step)
    if kind in ("verify", "prefill"):
        x = _model_inputs(case, seed)
        w = x["weights"]
        model = Qwen3Verify(_config(case), DEVICE, seed=seed)
        model.layers, model.embed, model.norm, model.lm_head = w["layers"], w["embed"], w["norm"], w["head"]
        model.pack_lm_head()
        model.k_caches, model.v_caches, model.block_size = x["k_cache"], x["v_cache"], case["page"]
        state = dict(case=case, model=model)
        if kind == "prefill":
            state.update(tokens=x["tokens"], starts=[case["prefix"]] * case["batch"], tables=x["tables"])
            return state
        seqs = []
        for tokens, table in zip(x["tokens"], x["tables"]):
            seq = Sequence(tokens[:len(tokens) - case["drafts"]])
            seq.draft_tokens = tokens[len(tokens) - case["drafts"]:]
            for t in seq.draft_tokens:
                seq.append_token(t)
            seq.block_table = table
            seqs.append(seq)
        longest = max(len(s) for s in seqs)
        runner = ModelRunner(model, case["batch"], case["drafts"], max(4096, longest))
        state.update(runner=runner, seqs=seqs)
        return state
    if kind == "accept":
        x = _accept_inputs(case, seed)
        state = dict(case=case, x=x)
        if case["mode"] != "greedy":  # part of a captured round; the greedy call is made directly
            outs = (torch.empty(case["batch"], case["drafts"] + 1, dtype=torch.int32, device=DEVICE),
                    torch.empty(case["batch"], dtype=torch.int32, device=DEVICE))
            rows = dict(uniforms=x["uniforms"], draft_logits=x["draft"], draft_seq_stride=case["drafts"],
                        draft_row_stride=1) if case["mode"] == "model" else {}
            outs[0].fill_(-1)  # entries past a sequence's accepted tokens are never written

            def step():
                accept_stochastic(x["target"], x["drafts"], x["num_drafts"], x["temperature"], x["noise"],
                                  target_seq_stride=case["drafts"] + 1, out_tokens=outs[0], out_len=outs[1], **rows)

            state.update(graph=_captured(step), outs=outs)
        else:
            state["out"] = torch.full((case["batch"], case["drafts"] + 1), -1, dtype=torch.int32, device=DEVICE)
        return state
    x = _ngram_inputs(case, seed)
    drafts = torch.full((case["batch"], case["drafts"]), -1, dtype=torch.int32, device=DEVICE)
    return dict(case=case, x=x, drafts=drafts, found=torch.zeros(case["batch"], dtype=torch.int32, device=DEVICE))


# --------------------------------------------------------------------- run
def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "verify_attention":
        state["graph"].replay()
        return state["outs"]
    if kind == "prefill_attention":
        x = state["x"]
        set_context(True, **state["step"])
        outs = [layer(q, k, v) for layer, q, k, v in zip(state["layers"], x["q"], x["k"], x["v"])]
        reset_context()
        return dict(out=outs, k_cache=x["k_cache"], v_cache=x["v_cache"])
    if kind == "verify":
        logits = state["runner"].run_spec_verify(state["seqs"])
        return dict(logits=logits, k_cache=state["model"].k_caches, v_cache=state["model"].v_caches)
    if kind == "prefill":
        model = state["model"]
        logits = model.prefill(state["tokens"], state["starts"], state["tables"])
        return dict(logits=logits, k_cache=model.k_caches, v_cache=model.v_caches)
    if kind == "accept":
        if case["mode"] == "greedy":
            x = state["x"]
            return accept_greedy(x["target"], x["drafts"], x["num_drafts"], case["drafts"] + 1,
                                 out_tokens=state["out"])
        state["graph"].replay()
        return state["outs"]
    x = state["x"]
    return ngram_draft(x["history"], x["lens"], case["drafts"], case["min_n"], case["max_n"],
                       out_drafts=state["drafts"], out_len=state["found"])


# -------------------------------------------------------------------- work
def _causal_pairs(new: list[int], keys: list[int]) -> int:
    """(query row, key) pairs of causal rows that end each sequence."""
    return sum(n * k - n * (n - 1) // 2 for n, k in zip(new, keys))


def _param_count(case: dict) -> int:
    heads, hidden, inter = SHAPES[case["model"]]
    return case["layers"] * hidden * ((2 * heads + 2 * KV_HEADS) * HEAD_DIM + 3 * inter)


def work(case: dict) -> dict:
    kind = case["kind"]
    kv_row = KV_HEADS * HEAD_DIM  # elements of one token's K (or V)
    if kind == "verify_attention":
        heads, rows = SHAPES[case["model"]][0], case["drafts"] + 1
        ctx = _lens(case, "ctx_lo", "ctx_hi")
        size = DTYPES[case["dtype"]].itemsize
        qo = 2 * len(ctx) * rows * heads * HEAD_DIM
        return dict(bytes=case["layers"] * size * (2 * sum(ctx) * kv_row + qo),
                    flops=case["layers"] * 4 * heads * HEAD_DIM * _causal_pairs([rows] * len(ctx), ctx))
    if kind == "prefill_attention":
        heads = SHAPES[case["model"]][0]
        new = _lens(case, "new_lo", "new_hi")
        keys = [case["prefix"] + n for n in new]
        moved = 2 * sum(new) * heads * HEAD_DIM + 2 * kv_row * (2 * sum(new) + sum(keys) - sum(new))
        return dict(bytes=case["layers"] * 2 * moved,
                    flops=case["layers"] * 4 * heads * HEAD_DIM * _causal_pairs(new, keys))
    if kind in ("verify", "prefill"):
        heads, hidden, _ = SHAPES[case["model"]]
        if kind == "verify":
            keys = [n + case["drafts"] for n in _lens(case, "ctx_lo", "ctx_hi")]
            new = [case["drafts"] + 1] * len(keys)
            head_rows = sum(new)
        else:
            new = _lens(case, "new_lo", "new_hi")
            keys = [case["prefix"] + n for n in new]
            head_rows = len(new)
        params = _param_count(case)
        head = VOCAB * hidden
        return dict(bytes=2 * (params + head + head_rows * VOCAB + case["layers"] * 2 * kv_row * sum(keys)),
                    flops=2 * sum(new) * params + 2 * head_rows * head
                    + case["layers"] * 4 * heads * HEAD_DIM * _causal_pairs(new, keys))
    if kind == "accept":
        B, K = case["batch"], case["drafts"]
        size = DTYPES[case["dtype"]].itemsize
        rows = {"greedy": K + 1, "model": 2 * K + 2, "ngram": 2 * (K + 1)}[case["mode"]]
        return dict(bytes=B * rows * VOCAB * size, flops=0)
    return dict(bytes=4 * sum(_lens(case, "ctx_lo", "ctx_hi")), flops=0)


# --------------------------------------------------------------- tolerance
def tolerance(case: dict):
    """Largest difference of a correct implementation at the same precision,
    about four times the measured distance from the 64-bit values: attention
    2.2e-3 (bf16 probabilities and outputs) and 5e-7 (32-bit sums), the
    logits of up to four layers 5.5e-3 to 8e-3; deeper models sum more
    rounded layers."""
    kind = case["kind"]
    if kind == "verify_attention":
        return {"rel": 5e-6} if case["dtype"] == "f32" else {"rel": 1e-2}
    if kind == "prefill_attention":
        return {"rel": 1e-2}
    if kind in ("verify", "prefill"):
        return {"rel": 2e-2 if case["layers"] <= 4 else 3e-2}
    return "exact"


# ------------------------------------------------------------------- exact
def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
    """Causal attention in 64 bits: row t of q [T, H, D] at position first + t
    over k, v [L, Hkv, D]."""
    T, H, D = q.shape
    group = H // KV_HEADS
    out = torch.empty(T, H, D, dtype=torch.float64, device=q.device)
    for hk in range(KV_HEADS):
        kt, vh = k[:, hk].t().contiguous(), v[:, hk].contiguous()
        for t0 in range(0, T, 1024):
            t1 = min(T, t0 + 1024)
            hide = torch.arange(k.shape[0], device=q.device)[None] > torch.arange(first + t0, first + t1,
                                                                                  device=q.device)[:, None]
            for h in range(hk * group, (hk + 1) * group):
                s = (q[t0:t1, h] @ kt) / math.sqrt(D)
                out[t0:t1, h] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ vh
    return out


def _keys(cache: torch.Tensor, table: list[int], n: int) -> torch.Tensor:
    """The first n rows of a paged sequence, in 64 bits."""
    return cache[table].reshape(-1, KV_HEADS, HEAD_DIM)[:n].double()


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.double()


def _rotate(x: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    half = HEAD_DIM // 2
    inv = 1_000_000.0 ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    angle = (pos.double()[:, None] * inv)[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)


def _exact_model(case: dict, seed: int) -> dict:
    x = _model_inputs(case, seed)
    w = x["weights"]
    heads, _, inter = SHAPES[case["model"]]
    ids, pos, slots = [], [], []
    for tokens, table, n in zip(x["tokens"], x["tables"], x["rows"]):
        ids += tokens[len(tokens) - n:]
        pos += range(len(tokens) - n, len(tokens))
        slots += _slots(table, len(tokens) - n, len(tokens), case["page"])
    pos, slots = torch.tensor(pos, device=DEVICE), torch.tensor(slots, device=DEVICE)
    r = w["embed"][ids].double()
    k_caches, v_caches = [], []
    for li, L in enumerate(w["layers"]):
        qkv = (_rms(r, L["ln1"]) @ L["qkv"].double().t()).view(len(ids), -1, HEAD_DIM)
        q = _rotate(_rms(qkv[:, :heads], L["q_norm"]), pos)
        k = _rotate(_rms(qkv[:, heads:heads + KV_HEADS], L["k_norm"]), pos)
        k_cache, v_cache = x["k_cache"][li].double(), x["v_cache"][li].double()
        k_cache.view(-1, KV_HEADS, HEAD_DIM)[slots] = k
        v_cache.view(-1, KV_HEADS, HEAD_DIM)[slots] = qkv[:, heads + KV_HEADS:]
        k_caches.append(k_cache)
        v_caches.append(v_cache)
        outs, at = [], 0
        for tokens, table, n in zip(x["tokens"], x["tables"], x["rows"]):
            outs.append(_attend(q[at:at + n], _keys(k_cache, table, len(tokens)), _keys(v_cache, table, len(tokens)),
                                len(tokens) - n))
            at += n
        r = r + torch.cat(outs).reshape(len(ids), -1) @ L["o"].double().t()
        gate_up = _rms(r, L["ln2"]) @ L["gate_up"].double().t()
        r = r + (torch.nn.functional.silu(gate_up[:, :inter]) * gate_up[:, inter:]) @ L["down"].double().t()
    if case["kind"] == "prefill":
        last, at = [], 0
        for n in x["rows"]:
            at += n
            last.append(at - 1)
        r = r[last]
    return dict(logits=_rms(r, w["norm"]) @ w["head"].double().t(), k_cache=k_caches, v_cache=v_caches)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "verify_attention":
        x = _verify_attention_inputs(case, seed)
        rows, outs = x["rows"], []
        for q, k, v in zip(x["q"], x["k"], x["v"]):
            outs.append(torch.cat([_attend(q[b * rows:(b + 1) * rows].double(), _keys(k, t, n), _keys(v, t, n), n - rows)
                                   for b, (t, n) in enumerate(zip(x["tables"], x["ctx"]))]))
        return outs
    if kind == "prefill_attention":
        x = _prefill_attention_inputs(case, seed)
        outs = []
        for li, q in enumerate(x["q"]):
            k_cache, v_cache = x["k_cache"][li], x["v_cache"][li]
            rows, at = [], 0
            for table, n, keys in zip(x["tables"], x["new"], x["keys"]):
                slots = torch.tensor(_slots(table, keys - n, keys, case["page"]), device=DEVICE)
                k_cache.view(-1, KV_HEADS, HEAD_DIM)[slots] = x["k"][li][at:at + n]
                v_cache.view(-1, KV_HEADS, HEAD_DIM)[slots] = x["v"][li][at:at + n]
                rows.append(_attend(q[at:at + n].double(), _keys(k_cache, table, keys), _keys(v_cache, table, keys),
                                    keys - n))
                at += n
            outs.append(torch.cat(rows).reshape(at, -1))
        return dict(out=outs, k_cache=[t.double() for t in x["k_cache"]], v_cache=[t.double() for t in x["v_cache"]])
    if kind in ("verify", "prefill"):
        return _exact_model(case, seed)
    return None
