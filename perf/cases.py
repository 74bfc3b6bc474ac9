"""The work that users of this package have it do, as cases that can be timed
and compared: whole decode steps and prompt prefills of the hybrid model, and
the layers' own entry points over the sizes that serving meets.

Every kind names a public entry point.  ``listed()`` holds representative
cases, ``draw`` gives others of the same ranges, ``prepare`` makes what a
program has in hand before the call, ``run`` is one pass, ``work`` the bytes
and operations that a pass cannot do without, ``exact`` the same outputs in
float64 from plain torch, and ``tolerance`` how far two correct
implementations at the same precision may be apart.

Sizes: the 4B-shaped model of ``runtime.ModelConfig`` (hidden 2560, 32 heads of
128, 8 KV / memory groups, 1024-slot window, 256 anchor slots in chunks of 64,
vocabulary 151936), the batches and prompt lengths of the benchmark workloads
and of the tests.  Whole-model cases keep its widths and take one period of the
layer pattern (4 of 36 layers), so that several models fit one GPU and the
rounding of one layer does not travel through many others.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from yanchor_amd import gdn, layers, runtime
from yanchor_amd import independent_memory as im
from yanchor_amd import inference_kernels as ik

BF16 = torch.bfloat16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
D = 128                      # head dim of every layer
HEADS, GROUPS = 32, 8        # query heads, KV / memory groups
WINDOW = 1024                # SWA ring slots
CHUNK = 64                   # tokens per anchor-memory commit
CHANNELS = 3 * HEADS * D     # conv channels of a GDN layer (q | k | v)
PROJ = CHANNELS + HEADS * D + 2 * HEADS   # its packed projection row (qkv | z | b | a)
VOCAB = 151936


def listed():
    return [
        # one interactive session: every weight read for one token, launches back to back
        {"name": "decode_b1", "kind": "decode", "batch": 1, "layers": 4},
        # the serving batch of the benchmark: one captured step of 128 slots
        {"name": "decode_b128", "kind": "decode", "batch": 128, "layers": 4},
        # a refill: ragged prompts packed into one prefill, logits and caches out
        {"name": "prefill_ragged", "kind": "prefill", "n": 12, "lo": 33, "hi": 1200, "lengths": 5, "layers": 4},
        # one GDN layer of a large packed prefill (the benchmark's prefill workload)
        {"name": "gdn_prefill_packed", "kind": "gdn_prefill", "n": 32, "lo": 512, "hi": 8192, "lengths": 1, "h": 32,
         "h0": False},
        # the same layer for a single long prompt that continues a state: the latency of one request
        {"name": "gdn_prefill_single", "kind": "gdn_prefill", "n": 1, "lo": 3001, "hi": 3001, "lengths": 1, "h": 32,
         "h0": True},
        # the decode core of a GDN layer with the throughput profile's float16 state
        {"name": "gdn_core_fp16", "kind": "gdn_core", "batch": 128, "state": "fp16"},
        # the drop-in recurrence on the live slots of a pool (the vLLM / SGLang layout)
        {"name": "gdn_update_pool", "kind": "gdn_update", "batch": 61, "pool": 96, "h": 32, "dtype": "bf16"},
        # the causal conv over a packed refill
        {"name": "conv_prefill", "kind": "conv", "n": 64, "lo": 1, "hi": 511, "lengths": 2},
        # window attention of prompt pieces that continue full rings, and the rings they leave
        {"name": "window_prefill", "kind": "window_prefill", "n": 16, "lo": 65, "hi": 2048, "lengths": 3,
         "context": True, "dtype": "bf16"},
        # the anchor memory's side of a prefill that continues a state
        {"name": "memory_prefill", "kind": "memory_prefill", "batch": 32, "length": 2048, "capacity": 256,
         "ragged": False},
        # an attention layer's reads for one token per slot: full rings, live memories, the commit
        {"name": "attention_decode", "kind": "attention_decode", "batch": 128, "capacity": 256},
        # the step's sampler over the vocabulary with the presence penalty
        {"name": "sample_top20", "kind": "sample", "batch": 128, "dtype": "bf16", "mode": "fused", "top_k": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "prefill", "gdn_prefill", "gdn_prefill", "gdn_core", "gdn_update", "conv",
                       "window_prefill", "memory_prefill", "attention_decode", "sample"])
    lengths = rng.randrange(1, 1 << 20)
    if kind == "decode":
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "layers": 4}
    if kind == "prefill":
        hi = _log_int(rng, 40, 1200)
        return {"kind": kind, "n": _log_int(rng, 1, min(48, 18000 // hi)), "lo": rng.randint(1, hi), "hi": hi,
                "lengths": lengths, "layers": 4}
    if kind == "gdn_prefill":
        hi = _log_int(rng, 50, 8192)
        return {"kind": kind, "n": _log_int(rng, 1, min(96, 130000 // hi)), "lo": rng.randint(1, hi), "hi": hi,
                "lengths": lengths, "h": rng.choice([16, 32]), "h0": rng.random() < 0.5}
    if kind == "gdn_core":
        return {"kind": kind, "batch": _log_int(rng, 1, 160), "state": rng.choice(["fp32", "fp16"])}
    if kind == "gdn_update":
        batch = _log_int(rng, 1, 160)
        return {"kind": kind, "batch": batch, "pool": batch + rng.randint(0, 64), "h": rng.choice([16, 32]),
                "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "conv":
        hi = _log_int(rng, 2, 2048)
        return {"kind": kind, "n": _log_int(rng, 1, min(128, max(1, 18000 // hi))), "lo": rng.randint(1, hi),
                "hi": hi, "lengths": lengths}
    if kind == "window_prefill":
        hi = _log_int(rng, 20, 4096)
        return {"kind": kind, "n": _log_int(rng, 1, min(64, 18000 // hi)), "lo": rng.randint(1, hi), "hi": hi,
                "lengths": lengths, "context": rng.random() < 0.5, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "memory_prefill":
        length = _log_int(rng, 40, 4096)
        return {"kind": kind, "batch": _log_int(rng, 1, min(64, 65536 // length)), "length": length,
                "capacity": rng.choice([16, 256]), "ragged": rng.random() < 0.5}
    if kind == "attention_decode":
        return {"kind": kind, "batch": _log_int(rng, 1, 160), "capacity": rng.choice([16, 256])}
    mode = rng.choice(["fused", "fused", "torch"])
    return {"kind": "sample", "batch": _log_int(rng, 1, 160), "dtype": rng.choice(["bf16", "fp32"]), "mode": mode,
            "top_k": 20 if mode == "fused" else rng.choice([0, 1, 20, 50])}


# ---------------------------------------------------------------------------
# inputs

def _lengths(case):
    """The sequence lengths of a packed case, uniform in [lo, hi]."""
    gen = torch.Generator().manual_seed(int(case["lengths"]))
    return torch.randint(case["lo"], case["hi"] + 1, (case["n"],), generator=gen).tolist()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape, dtype=BF16, std=1.0):
    return (torch.randn(*shape, device="cuda", generator=gen) * std).to(dtype)


def _cu(lengths):
    return torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device="cuda")


def _gates(gen, *shape):
    """(g, beta) float32: log decays near 0, mixing rates in (0, 1)."""
    g = F.logsigmoid(torch.randn(*shape, device="cuda", generator=gen) + 3.0)
    return g, torch.sigmoid(torch.randn(*shape, device="cuda", generator=gen))


def _gdn_params(gen):
    a_log = torch.log(torch.empty(HEADS, device="cuda").uniform_(1.0, 16.0, generator=gen))
    return {"conv_w": _randn(gen, CHANNELS, 4, std=0.3), "a_log": a_log,
            "dt_bias": torch.ones(HEADS, device="cuda"), "norm_w": 1.0 + _randn(gen, D, std=0.1)}


def _memory(gen, positions, groups, capacity, dtype=BF16):
    """An anchor memory at the given sequence positions ([B] int64): whole
    chunks committed in rank order, the rest pending."""
    b = positions.shape[0]
    st = im.IndependentMemoryState.empty(b, groups, capacity, CHUNK, D, "cuda", dtype)
    committed = positions // CHUNK * CHUNK
    for rows in (st.keys, st.values, st.pending_keys, st.pending_values):
        rows.copy_(torch.randn(rows.shape, device="cuda", generator=gen))
    # capacity distinct earlier positions per group; slots past the committed tokens are empty
    at = torch.rand(b, groups, capacity, device="cuda", generator=gen)
    at = ((torch.arange(capacity, device="cuda") + at) / capacity * committed[:, None, None]).long()
    live = torch.arange(capacity, device="cuda") < committed[:, None, None]
    at = torch.where(committed[:, None, None] <= capacity, torch.arange(capacity, device="cuda"), at)
    sc = torch.randn(b, groups, capacity, device="cuda", generator=gen).sort(-1, descending=True).values
    st.positions.copy_(torch.where(live, at, torch.full_like(at, -1)))
    st.scores.copy_(sc.masked_fill(~live, -math.inf))
    for rows in (st.keys, st.values):
        rows.masked_fill_(~live[..., None], 0)
    held = torch.arange(CHUNK, device="cuda") < (positions % CHUNK)[:, None, None]
    ps = torch.randn(b, groups, CHUNK, device="cuda", generator=gen)
    st.pending_scores.copy_(ps.masked_fill(~held, -math.inf))
    st.count.copy_(positions % CHUNK)
    st.total.copy_(positions)
    return st


MEMORY_FIELDS = ("keys", "values", "scores", "positions", "pending_keys", "pending_values", "pending_scores", "count",
                 "total")


def _memory_outputs(st):
    return {f: getattr(st, f) for f in MEMORY_FIELDS}


def _rings(gen, positions, dtype=BF16):
    """Window rings of rows that have seen ``positions`` tokens each."""
    b = positions.shape[0]
    k, v = _randn(gen, b, GROUPS, WINDOW, D, dtype=dtype), _randn(gen, b, GROUPS, WINDOW, D, dtype=dtype)
    last = positions[:, None] - 1
    slots = torch.arange(WINDOW, device="cuda")[None]
    pos = last - (last - slots) % WINDOW              # the newest position <= last in each slot
    pos = torch.where((pos >= 0) & (last >= 0), pos, torch.full_like(pos, -1)).to(torch.int32)
    return k, v, pos[:, None].expand(b, GROUPS, WINDOW).contiguous()


def _config(case):
    return runtime.ModelConfig(layers=case["layers"])


def _prepare_decode(case, seed):
    cfg, b = _config(case), case["batch"]
    model = runtime.Model(cfg, b, "cuda", seed=seed)
    tokens = torch.zeros(b, dtype=torch.long, device="cuda")
    positions = torch.zeros(b, dtype=torch.long, device="cuda")
    valid = torch.ones(b, dtype=torch.bool, device="cuda")
    for _ in range(2):                                # warm the allocator outside the capture
        model.decode_step(tokens, positions, valid, float_logits=False)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = model.decode_step(tokens, positions, valid, float_logits=False)
    torch.cuda.synchronize()
    # the sequences in the slots: up to 4000 tokens so far, caches in place
    gen = _gen(seed + 1)
    tokens.copy_(torch.randint(0, cfg.vocab, (b,), device="cuda", generator=gen))
    positions.copy_(torch.randint(64, 4000, (b,), device="cuda", generator=gen))
    for i in model.gdn_state:
        model.gdn_state[i].copy_(_randn(gen, *model.gdn_state[i].shape, dtype=torch.float32, std=0.02))
        model.conv_state[i].copy_(_randn(gen, *model.conv_state[i].shape))
    for i in model.ring_k:
        for dst, src in zip((model.ring_k[i], model.ring_v[i], model.ring_pos[i]), _rings(gen, positions)):
            dst.copy_(src)
        st = _memory(gen, positions, GROUPS, cfg.memory_capacity)
        for f in MEMORY_FIELDS:
            getattr(model.memory[i], f).copy_(getattr(st, f))
    return {"model": model, "tokens": tokens, "positions": positions, "valid": valid, "graph": graph,
            "logits": logits}


def _prepare_prefill(case, seed):
    gen = torch.Generator().manual_seed(seed)
    model = runtime.Model(_config(case), 1, "cuda", seed=seed)
    return {"model": model, "prompts": [torch.randint(0, VOCAB, (n,), generator=gen) for n in _lengths(case)]}


def _prepare_gdn_prefill(case, seed):
    gen, lens = _gen(seed), _lengths(case)
    n, h = sum(lens), case["h"]
    q, k = _randn(gen, 1, n, h, D), _randn(gen, 1, n, h, D)
    g, beta = _gates(gen, 1, n, HEADS)
    h0 = _randn(gen, len(lens), HEADS, D, D, dtype=torch.float32, std=0.02) if case["h0"] else None
    return {"q": q, "k": k, "v": _randn(gen, 1, n, HEADS, D), "g": g, "beta": beta, "h0": h0, "cu": _cu(lens),
            "lengths": lens}


def _prepare_gdn_core(case, seed):
    gen, b = _gen(seed), case["batch"]
    return {**_gdn_params(gen), "proj": _randn(gen, b, PROJ), "conv": _randn(gen, b, 3, CHANNELS),
            "state": _randn(gen, b, HEADS, D, D, dtype=DTYPES[case["state"]], std=0.02)}


def _prepare_gdn_update(case, seed):
    gen, b, h, dtype = _gen(seed), case["batch"], case["h"], DTYPES[case["dtype"]]
    g, beta = _gates(gen, b, 1, HEADS)
    slots = torch.randperm(case["pool"], device="cuda", generator=gen)[:b].to(torch.int32)
    return {"q": _randn(gen, b, 1, h, D, dtype=dtype), "k": _randn(gen, b, 1, h, D, dtype=dtype),
            "v": _randn(gen, b, 1, HEADS, D, dtype=dtype), "g": g, "beta": beta, "slots": slots,
            "state": _randn(gen, case["pool"], HEADS, D, D, dtype=torch.float32, std=0.02)}


def _prepare_conv(case, seed):
    gen, lens = _gen(seed), _lengths(case)
    return {"proj": _randn(gen, sum(lens), PROJ), "window": _randn(gen, len(lens), 3, CHANNELS),
            "w": _randn(gen, CHANNELS, 4, std=0.3), "cu": _cu(lens)}


def _prepare_window_prefill(case, seed):
    gen, lens, dtype = _gen(seed), _lengths(case), DTYPES[case["dtype"]]
    n, r = sum(lens), len(lens)
    starts = torch.zeros(r, dtype=torch.long, device="cuda")
    if case["context"]:                               # pieces of longer prompts: earlier tokens in the rings
        starts.copy_(torch.randint(1, 3 * WINDOW, (r,), device="cuda", generator=gen))
    ring_k, ring_v, ring_pos = _rings(gen, starts, dtype)
    # the attention projection row: (q | gate) per head, then k and v of every group
    proj = _randn(gen, n, 2 * HEADS * D + 2 * GROUPS * D, dtype=dtype)
    qg = proj[:, : 2 * HEADS * D].view(n, HEADS, 2 * D)
    return {"q": _randn(gen, n, HEADS, D, dtype=dtype), "gate": qg[..., D:], "k": _randn(gen, n, GROUPS, D, dtype=dtype),
            "v": proj[:, 2 * HEADS * D + GROUPS * D:].view(n, GROUPS, D), "cu": _cu(lens), "starts": starts,
            "rows": torch.arange(r, device="cuda"), "lengths": lens, "ring_k": ring_k, "ring_v": ring_v,
            "ring_pos": ring_pos}


def _prepare_memory_prefill(case, seed):
    gen, b, n = _gen(seed), case["batch"], case["length"]
    positions = torch.randint(0, 1024, (b,), device="cuda", generator=gen)
    valid = None
    if case["ragged"]:                                # right-padded rows, the longest one whole
        lens = torch.randint(1, n + 1, (b,), device="cuda", generator=gen)
        lens[0] = n
        valid = torch.arange(n, device="cuda")[None] < lens[:, None]
    return {"q": _randn(gen, b, n, HEADS, D), "k": _randn(gen, b, n, GROUPS, D), "v": _randn(gen, b, n, GROUPS, D),
            "scores": torch.randn(b, n, GROUPS, device="cuda", generator=gen), "valid": valid,
            "state": _memory(gen, positions, GROUPS, case["capacity"])}


def _prepare_attention_decode(case, seed):
    gen, b = _gen(seed), case["batch"]
    positions = torch.randint(WINDOW, 4 * WINDOW, (b,), device="cuda", generator=gen)
    ring_k, ring_v, ring_pos = _rings(gen, positions)
    proj = _randn(gen, b, 2 * HEADS * D)              # (q | gate) per head
    return {"q": _randn(gen, b, 1, HEADS, D), "gate": proj.view(b, HEADS, 2 * D)[..., D:], "ring_k": ring_k,
            "ring_v": ring_v, "ring_pos": ring_pos, "mq": _randn(gen, b, 1, HEADS, D),
            "head_gate": torch.rand(b, HEADS, device="cuda", generator=gen) * 2,
            "valid": torch.rand(b, device="cuda", generator=gen) < 0.97,
            "key": _randn(gen, b, 1, GROUPS, D), "value": _randn(gen, b, 1, GROUPS, D),
            "scores": torch.randn(b, 1, GROUPS, device="cuda", generator=gen),
            "state": _memory(gen, positions, GROUPS, case["capacity"])}


def _prepare_sample(case, seed):
    gen, b = _gen(seed), case["batch"]
    return {"logits": _randn(gen, b, VOCAB, dtype=DTYPES[case["dtype"]], std=2.0),
            "seen": torch.rand(b, VOCAB, device="cuda", generator=gen) < 0.007,
            "ids": torch.randperm(4096, device="cuda", generator=gen)[:b],
            "steps": torch.randint(1, 4096, (b,), device="cuda", generator=gen)}


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, int(seed))
    return {"case": dict(case), **state}


# ---------------------------------------------------------------------------
# one pass

def _model_caches(model, caches=None):
    """The caches that a step or a prefill leaves, except the anchor memories'
    committed slots: those stand in rank order of the admission scores, and
    which of two nearly tied scores is the higher one turns on the last bit of
    the layers before (the ``memory_prefill`` and ``attention_decode`` cases,
    whose scores are inputs, compare them)."""
    per = {}
    if caches is None:
        caches = model.cache_tensors()
    it = iter(caches)
    for i in model.gdn_state:
        per[f"gdn{i}"], per[f"conv{i}"] = next(it), next(it)
    for i in model.ring_k:
        per[f"ring_k{i}"], per[f"ring_v{i}"], per[f"ring_pos{i}"] = next(it), next(it), next(it)
        fields = {f: next(it) for f in MEMORY_FIELDS}
        per[f"count{i}"], per[f"total{i}"] = fields["count"], fields["total"]
    return per


def _run_decode(s):
    s["graph"].replay()
    return {"logits": s["logits"], **_model_caches(s["model"])}


def _run_prefill(s):
    logits, caches = s["model"].prefill(s["prompts"])
    return {"logits": logits, **_model_caches(s["model"], caches)}


def _run_gdn_prefill(s):
    o, state = gdn.chunk_gated_delta_rule(s["q"], s["k"], s["v"], g=s["g"], beta=s["beta"], initial_state=s["h0"],
                                          output_final_state=True, use_qk_l2norm_in_kernel=True, cu_seqlens=s["cu"],
                                          lengths=s["lengths"])
    return {"o": o, "state": state}


def _run_gdn_core(s):
    y = layers.gdn_decode_fused(s["proj"], s["conv"], s["conv_w"], s["a_log"], s["dt_bias"], s["state"], s["norm_w"],
                                1e-6, heads=HEADS, head_dim=D, z_offset=CHANNELS, b_offset=CHANNELS + HEADS * D,
                                a_offset=CHANNELS + HEADS * D + HEADS)
    return {"y": y, "state": s["state"], "conv": s["conv"]}


def _run_gdn_update(s):
    o, state = gdn.recurrent_gated_delta_rule(s["q"], s["k"], s["v"], g=s["g"], beta=s["beta"],
                                              initial_state=s["state"], state_indices=s["slots"])
    return {"o": o, "state": state}


def _run_conv(s):
    y = layers.conv_prefill(s["proj"], s["window"], s["w"], s["cu"], CHANNELS)
    return {"y": y, "window": s["window"]}


def _run_window_prefill(s):
    out = layers.swa_prefill(s["q"], s["k"], s["v"], s["cu"], s["starts"], s["ring_k"], s["ring_v"], s["rows"],
                             gate=s["gate"], lengths=s["lengths"])
    layers.ring_fill(s["k"], s["v"], s["cu"], s["starts"], s["rows"], s["ring_k"], s["ring_v"], s["ring_pos"])
    return {"out": out, "ring_k": s["ring_k"], "ring_v": s["ring_v"], "ring_pos": s["ring_pos"]}


def _run_memory_prefill(s):
    out = im.sequence(s["q"], s["k"], s["v"], s["scores"], s["valid"], CHUNK, s["state"])
    return {"out": out, **_memory_outputs(s["state"])}


def _run_attention_decode(s):
    att = im.ring_decode_attention(s["q"], s["ring_k"], s["ring_v"], s["ring_pos"], gate=s["gate"])
    read = im.committed_gqa_gated(s["mq"], s["state"], None, s["valid"], s["head_gate"])
    im.commit_decode(s["key"], s["value"], s["scores"], s["valid"], CHUNK, s["state"])
    return {"att": att, "read": read, **_memory_outputs(s["state"])}


def _run_sample(s):
    c = s["case"]
    mode = ik.SAMPLE_FUSED if c["mode"] == "fused" else ik.SAMPLE_TORCH
    return ik.topk_sample(s["logits"], s["ids"], s["steps"], seed=20260923, temperature=0.6, top_k=c["top_k"],
                          top_p=0.95, mode=mode, seen=s["seen"], presence_penalty=1.5)


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _model_weights(case):
    """(weights of the layers, weights of the lm_head), in elements."""
    c = _config(case)
    mlp = 3 * c.intermediate * c.hidden
    att = c.hidden * (2 * HEADS * D + 2 * GROUPS * D) + HEADS * D * c.hidden
    mem = c.hidden * (HEADS * D + c.admission_rank + 2 * c.writer_intermediate) + c.writer_intermediate * c.hidden \
        + c.hidden * 2 * GROUPS * D + HEADS * D * c.hidden
    rec = c.hidden * PROJ + HEADS * D * c.hidden + CHANNELS * 4
    n_att = sum(c.is_memory_layer(i) for i in range(c.layers))
    return c.layers * mlp + n_att * (att + mem) + (c.layers - n_att) * rec, c.vocab * c.hidden


def _gdn_chunk_flops(tokens, heads):
    """The chunked form of the recurrence, C = 64 (products only)."""
    return tokens / 64 * heads * (10 * 64 * 64 * D + 6 * 64 * D * D + 2 / 3 * 64 ** 3)


def _window_pairs(lens, starts=None):
    """(query, key) pairs of sliding-window causal attention."""
    total = 0
    for n in lens:
        if starts:                                    # a full window before the piece
            total += n * WINDOW
        else:
            m = min(n, WINDOW)
            total += m * (m + 1) // 2 + (n - m) * WINDOW
    return total


def work(case):
    kind = case["kind"]
    if kind == "decode":
        c, b = _config(case), case["batch"]
        w, head = _model_weights(case)
        n_att = sum(c.is_memory_layer(i) for i in range(c.layers))
        n_rec = c.layers - n_att
        state = n_rec * (2 * b * HEADS * D * D * 4 + 2 * b * 3 * CHANNELS * 2)
        reads = n_att * b * GROUPS * D * 2 * 2 * (WINDOW + c.memory_capacity)
        return {"bytes": 2 * (w + head) + state + reads + b * c.vocab * 2,
                "flops": 2 * b * (w + head) + n_rec * b * HEADS * D * D * 6 + n_att * b * HEADS * D * 4 *
                (WINDOW + c.memory_capacity)}
    if kind == "prefill":
        c, lens = _config(case), _lengths(case)
        n, r = sum(lens), len(lens)
        w, head = _model_weights(case)
        n_att = sum(c.is_memory_layer(i) for i in range(c.layers))
        n_rec = c.layers - n_att
        caches = n_rec * r * (HEADS * D * D * 4 + 3 * CHANNELS * 2) + \
            n_att * r * GROUPS * D * 2 * 2 * (WINDOW + c.memory_capacity + CHUNK)
        return {"bytes": 2 * (w + head) + n * c.hidden * 2 + caches + r * c.vocab * 4,
                "flops": 2 * n * w + 2 * r * head + n_rec * _gdn_chunk_flops(n, HEADS) +
                n_att * HEADS * D * 4 * (_window_pairs(lens) + n * c.memory_capacity)}
    if kind == "gdn_prefill":
        lens = _lengths(case)
        n, h = sum(lens), case["h"]
        state = len(lens) * HEADS * D * D * 4 * (2 if case["h0"] else 1)
        return {"bytes": n * (2 * h * D + 2 * HEADS * D) * 2 + n * HEADS * 8 + state,
                "flops": _gdn_chunk_flops(n, HEADS)}
    if kind == "gdn_core":
        b, size = case["batch"], SIZES[case["state"]]
        return {"bytes": 2 * b * HEADS * D * D * size + b * PROJ * 2 + 2 * b * 3 * CHANNELS * 2 + CHANNELS * 8 +
                b * HEADS * D * 2, "flops": b * HEADS * D * D * 6}
    if kind == "gdn_update":
        b, size = case["batch"], SIZES[case["dtype"]]
        return {"bytes": 2 * b * HEADS * D * D * 4 + b * (2 * case["h"] + 2 * HEADS) * D * size + b * HEADS * 8,
                "flops": b * HEADS * D * D * 6}
    if kind == "conv":
        lens = _lengths(case)
        n = sum(lens)
        return {"bytes": 2 * n * CHANNELS * 2 + 2 * len(lens) * 3 * CHANNELS * 2 + CHANNELS * 8,
                "flops": n * CHANNELS * 8}
    if kind == "window_prefill":
        lens = _lengths(case)
        n, r = sum(lens), len(lens)
        context = r * GROUPS * WINDOW * D * 4 if case["context"] else 0
        filled = sum(min(x, WINDOW) for x in lens) * GROUPS * D * 4
        return {"bytes": n * (3 * HEADS * D + 2 * GROUPS * D) * 2 + context + filled,
                "flops": HEADS * D * 4 * _window_pairs(lens, case["context"])}
    if kind == "memory_prefill":
        b, n, cap = case["batch"], case["length"], case["capacity"]
        n_valid = b * n * (0.5 if case["ragged"] else 1.0)
        state = b * GROUPS * (2 * cap + CHUNK) * D * 4
        return {"bytes": n_valid * (2 * HEADS + 2 * GROUPS) * D * 2 + n_valid * GROUPS * 4 + state,
                "flops": n_valid * HEADS * cap * D * 4}
    if kind == "attention_decode":
        b, slots = case["batch"], WINDOW + case["capacity"]
        return {"bytes": b * GROUPS * slots * (D * 4 + 4) + b * (5 * HEADS + 4 * GROUPS) * D * 2,
                "flops": b * HEADS * slots * D * 4}
    return {"bytes": case["batch"] * VOCAB * (SIZES[case["dtype"]] + 1), "flops": case["batch"] * VOCAB}


# ---------------------------------------------------------------------------
# how far two correct implementations may be apart

def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "gdn_update" and case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if kind in ("decode", "prefill"):                 # 4 layers of bf16 activations and the head
        return {"rel": 3e-2}
    return {"rel": 1e-2}                              # one layer with bf16 / fp16 outputs


# ---------------------------------------------------------------------------
# the same outputs in float64

def _norm64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1.0 + w.double())


def _unit64(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _silu64(x):
    return x * torch.sigmoid(x)


def _delta64(state, q, k, v, g, beta):
    """One token of the gated delta rule: state [B, HV, K, V] -> (o, state);
    q, k [B, H, K] raw (normalised here), HV a multiple of H."""
    rep = v.shape[1] // q.shape[1]
    q = (_unit64(q) * D ** -0.5).repeat_interleave(rep, 1)
    k = _unit64(k).repeat_interleave(rep, 1)
    state = state * g.exp()[..., None, None]
    delta = beta[..., None] * (v - (state * k[..., None]).sum(-2))
    state = state + k[..., None] * delta[..., None, :]
    return (state * q[..., None]).sum(-2), state


def _core64(proj, conv, conv_w, a_log, dt_bias, state, norm_w):
    """One token of a GDN layer between its projections: (y, conv window, state)."""
    b = proj.shape[0]
    window = torch.cat((conv, proj[:, None, :CHANNELS]), 1)
    mixed = _silu64((window * conv_w.double().t()[None]).sum(1)).view(b, 3, HEADS, D)
    z, rest = proj[:, CHANNELS: CHANNELS + HEADS * D].view(b, HEADS, D), proj[:, CHANNELS + HEADS * D:]
    g = -a_log.double().exp() * F.softplus(rest[:, HEADS:] + dt_bias.double())
    o, state = _delta64(state, mixed[:, 0], mixed[:, 1], mixed[:, 2], g, torch.sigmoid(rest[:, :HEADS]))
    y = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-6) * norm_w.double() * _silu64(z)
    return y.reshape(b, -1), window[:, 1:], state


def _attend64(q, keys, values, live, sink):
    """q [B, H, D] over keys / values [B, G, S, D] of the live [B, G, S] slots."""
    b, h, _ = q.shape
    g = keys.shape[1]
    logits = (q.view(b, g, h // g, D) @ keys.transpose(-1, -2).contiguous()) / math.sqrt(D)
    logits = logits.masked_fill(~live[:, :, None], -math.inf)
    if sink:
        logits = F.pad(logits, (0, 1))
    w = logits.softmax(-1)
    return (w[..., : keys.shape[2]] @ values).reshape(b, h, D)


def _rank(scores, positions):
    """Order of candidates: score descending, position ascending with empty
    slots last."""
    key = torch.where(positions < 0, torch.full_like(positions, 1 << 30), positions)
    by_pos = key.argsort(dim=-1, stable=True)
    return by_pos.gather(-1, scores.gather(-1, by_pos).argsort(dim=-1, descending=True, stable=True))


def _commit64(st, key, value, scores, active):
    """One token per active row into the pending chunk; full chunks committed.
    ``st``: dict of the memory's fields."""
    rows = torch.arange(key.shape[0], device=key.device)[active]
    at = st["count"][rows]
    for f, x in (("pending_keys", key), ("pending_values", value), ("pending_scores", scores)):
        st[f][rows, :, at] = x[rows].to(st[f].dtype)
    st["total"][rows] += 1
    st["count"][rows] = at + 1
    full = rows[at + 1 == CHUNK]
    if full.numel():
        cap = st["keys"].shape[2]
        pend = (st["total"][full] - CHUNK)[:, None, None] + torch.arange(CHUNK, device=key.device)
        pos = torch.cat((st["positions"][full].long(), pend.expand(-1, st["keys"].shape[1], -1)), -1)
        sc = torch.cat((st["scores"][full], st["pending_scores"][full]), -1)
        take = _rank(sc, pos)[..., :cap]
        for f in ("keys", "values"):
            src = torch.cat((st[f][full], st["pending_" + f][full]), 2)
            st[f][full] = src.gather(2, take[..., None].expand(-1, -1, -1, D))
        st["scores"][full] = sc.gather(-1, take)
        st["positions"][full] = pos.gather(-1, take).to(st["positions"].dtype)
        st["count"][full] = 0


class _Model64:
    """The model's decode step in float64 on its raw weights."""

    def __init__(self, model):
        self.c, self.kinds = model.cfg, [L["kind"] for L in model.layers]
        self.layers = [{k: v.double() for k, v in L.items() if torch.is_tensor(v) and "@" not in k}
                       for L in model.layers]
        self.embed, self.head = model.embed, model.lm_head
        self.final_norm = model.final_norm

    def rope(self, x, positions):
        c = self.c
        half = c.rotary_dim // 2
        inv = c.rope_theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
        ang = positions.double()[:, None, None] * inv
        a, b = x[..., :half], x[..., half: 2 * half]
        return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), x[..., 2 * half:]), -1)

    def step(self, tokens, positions, caches, active):
        """The residual stream of one token per row; ``caches``: per layer, a
        dict of float64 tensors that the rows of ``active`` [B] update."""
        c, b = self.c, tokens.shape[0]
        h = self.embed[tokens].double()
        rows = torch.arange(b, device=h.device)
        keep = active
        for L, kind, st in zip(self.layers, self.kinds, caches):
            xn = _norm64(h, L["in_norm"])
            if kind == "gdn":
                y, conv, state = _core64(xn @ L["w_in"].t(), st["conv"], L["conv_w"], L["a_log"], L["dt_bias"],
                                         st["gdn"], L["gnorm"])
                st["conv"] = torch.where(keep[:, None, None], conv, st["conv"])
                st["gdn"] = torch.where(keep[:, None, None, None], state, st["gdn"])
                delta = y @ L["w_out"].t()
            else:
                proj = xn @ L["w_qkv"].t()
                qg = proj[:, : 2 * HEADS * D].view(b, HEADS, 2 * D)
                kv = proj[:, 2 * HEADS * D:].view(b, 2, GROUPS, D)
                q = self.rope(_norm64(qg[..., :D], L["q_norm"]), positions)
                k = self.rope(_norm64(kv[:, 0], L["k_norm"]), positions)
                live, slot = rows[keep], (positions % WINDOW)[keep]
                st["ring_k"][live, :, slot], st["ring_v"][live, :, slot] = k[keep], kv[:, 1][keep]
                st["ring_pos"][live, :, slot] = positions[keep].to(st["ring_pos"].dtype)[:, None]
                att = _attend64(q, st["ring_k"], st["ring_v"], st["ring_pos"] >= 0, sink=False)
                delta = (att * torch.sigmoid(qg[..., D:])).reshape(b, -1) @ L["w_o"].t()
                delta = delta + self.memory(L, st, h, positions, keep)
            h = h + delta
            gate, up = (_norm64(h, L["post_norm"]) @ L["mlp_gate_up"].t()).chunk(2, -1)
            h = h + (_silu64(gate) * up) @ L["mlp_down"].t()
        return h

    def memory(self, L, st, h, positions, keep):
        c, b = self.c, h.shape[0]
        u = _norm64(h, L["m_in_norm"])
        proj = u @ L["m_in"].t()
        qn = _norm64(proj[:, : HEADS * D].view(b, HEADS, D), L["m_q_norm"])
        gate = torch.tanh(L["read_scale"]) * 2 * torch.sigmoid(
            (qn * L["read_gate_w"]).sum(-1) / math.sqrt(D) + L["read_gate_b"])
        feats, wg, wu = proj[:, HEADS * D:].split((c.admission_rank, c.writer_intermediate, c.writer_intermediate), -1)
        read = _attend64(self.rope(qn, positions), st["keys"], st["values"], st["positions"] >= 0, sink=True)
        kv = ((u + (_silu64(wg) * wu) @ L["writer_down"].t()) @ L["m_kv"].t()).view(b, 2, GROUPS, D)
        key = self.rope(_norm64(kv[:, 0], L["m_k_norm"]), positions)
        _commit64(st, key, kv[:, 1], _silu64(feats) @ L["adm_up"].t(), keep)
        return (read * gate[..., None]).reshape(b, -1) @ L["m_o"].t()

    def logits(self, h):
        return _norm64(h, self.final_norm) @ self.head.double().t()

    def outputs(self, h, caches):
        out = {"logits": self.logits(h)}
        for i, (kind, st) in enumerate(zip(self.kinds, caches)):
            if kind == "gdn":
                out[f"gdn{i}"], out[f"conv{i}"] = st["gdn"], st["conv"]
            else:
                for f in ("ring_k", "ring_v", "ring_pos", "count", "total"):
                    out[f"{f}{i}"] = st[f]
        return out


def _wide(x):
    return x.double() if x.is_floating_point() else x.clone()


def _exact_decode(case, s):
    m = s["model"]
    caches = []
    for i, L in enumerate(m.layers):
        if L["kind"] == "gdn":
            caches.append({"gdn": m.gdn_state[i].double(), "conv": m.conv_state[i].double()})
        else:
            st = {f: _wide(getattr(m.memory[i], f)) for f in MEMORY_FIELDS}
            caches.append({**st, "ring_k": m.ring_k[i].double(), "ring_v": m.ring_v[i].double(),
                           "ring_pos": m.ring_pos[i].clone()})
    ref = _Model64(m)
    return ref.outputs(ref.step(s["tokens"], s["positions"], caches, s["valid"]), caches)


def _exact_prefill(case, s):
    lens = _lengths(case)
    if max(lens) > 1200:                               # token by token: about 15 s at this length
        return None
    m, r, cap = s["model"], len(lens), s["model"].cfg.memory_capacity
    caches = []
    for kind in (L["kind"] for L in m.layers):
        z = dict(device="cuda", dtype=torch.float64)
        if kind == "gdn":
            caches.append({"gdn": torch.zeros(r, HEADS, D, D, **z), "conv": torch.zeros(r, 3, CHANNELS, **z)})
        else:
            st = im.IndependentMemoryState.empty(r, GROUPS, cap, CHUNK, D, "cuda", torch.float64)
            caches.append({**{f: _wide(getattr(st, f)) for f in MEMORY_FIELDS},
                           "ring_k": torch.zeros(r, GROUPS, WINDOW, D, **z),
                           "ring_v": torch.zeros(r, GROUPS, WINDOW, D, **z),
                           "ring_pos": torch.full((r, GROUPS, WINDOW), -1, device="cuda", dtype=torch.int32)})
    ref = _Model64(m)
    tokens = torch.zeros(r, max(lens), dtype=torch.long)
    for i, p in enumerate(s["prompts"]):
        tokens[i, : lens[i]] = p
    tokens, n = tokens.cuda(), torch.tensor(lens, device="cuda")
    last = torch.zeros(r, m.cfg.hidden, device="cuda", dtype=torch.float64)
    for t in range(max(lens)):
        h = ref.step(tokens[:, t], torch.full_like(n, t), caches, t < n)
        last = torch.where((t == n - 1)[:, None], h, last)
    return ref.outputs(last, caches)


def _exact_gdn_prefill(case, s):
    lens = s["lengths"]
    order = sorted(range(len(lens)), key=lambda i: -lens[i])
    at = s["cu"][:-1].long()[order]
    state = torch.zeros(len(lens), HEADS, D, D, device="cuda", dtype=torch.float64)
    if s["h0"] is not None:
        state.copy_(s["h0"][order])
    out = torch.empty(1, sum(lens), HEADS, D, device="cuda", dtype=torch.float64)
    for t in range(max(lens)):
        n = sum(lens[i] > t for i in order)           # the first n rows are still running
        rows = at[:n] + t
        x = (s[f][0, rows].double() for f in ("q", "k", "v", "g", "beta"))
        out[0, rows], state[:n] = _delta64(state[:n], *x)
    final = torch.empty_like(state)
    final[order] = state
    return {"o": out, "state": final}


def _exact_gdn_core(case, s):
    y, conv, state = _core64(s["proj"].double(), s["conv"].double(), s["conv_w"], s["a_log"], s["dt_bias"],
                             s["state"].double(), s["norm_w"])
    return {"y": y, "state": state, "conv": conv}


def _exact_gdn_update(case, s):
    state, slots = s["state"].double(), s["slots"].long()
    o, new = _delta64(state[slots], *(s[f][:, 0].double() for f in ("q", "k", "v", "g", "beta")))
    state[slots] = new
    return {"o": o[:, None], "state": state}


def _exact_conv(case, s):
    w, ys, windows, off = s["w"].double(), [], [], 0
    for r, n in enumerate(_lengths(case)):
        ext = torch.cat((s["window"][r].double(), s["proj"][off: off + n, :CHANNELS].double()), 0)
        ys.append(_silu64(sum(ext[j: j + n] * w[:, j] for j in range(4))))
        windows.append(ext[n:])
        off += n
    return {"y": torch.cat(ys), "window": torch.stack(windows)}


def _exact_window_prefill(case, s):
    lens, outs, off = s["lengths"], [], 0
    ring = {f: _wide(s[f]) for f in ("ring_k", "ring_v", "ring_pos")}
    rep = HEADS // GROUPS
    for r, n in enumerate(lens):
        start = int(s["starts"][r])
        held = min(start, WINDOW - 1)
        slots = torch.arange(start - held, start, device="cuda") % WINDOW
        k = torch.cat((s["ring_k"][r][:, slots].transpose(0, 1), s["k"][off: off + n]), 0).double()
        v = torch.cat((s["ring_v"][r][:, slots].transpose(0, 1), s["v"][off: off + n]), 0).double()
        q = s["q"][off: off + n].double()
        for b0 in range(0, n, 512):
            b1 = min(n, b0 + 512)
            lo, hi = max(0, held + b0 - WINDOW + 1), held + b1
            qp = torch.arange(held + b0, held + b1, device="cuda")[:, None]
            kp = torch.arange(lo, hi, device="cuda")[None]
            mask = (kp <= qp) & (kp > qp - WINDOW)
            kb = k[lo:hi].transpose(0, 1).repeat_interleave(rep, 0)          # [H, S, D]
            vb = v[lo:hi].transpose(0, 1).repeat_interleave(rep, 0)
            logits = q[b0:b1].transpose(0, 1).contiguous() @ kb.transpose(1, 2).contiguous() / math.sqrt(D)
            outs.append((logits.masked_fill(~mask, -math.inf).softmax(-1) @ vb).transpose(0, 1))
        t = torch.arange(max(0, n - WINDOW), n, device="cuda")
        slot = (start + t) % WINDOW
        ring["ring_k"][r][:, slot] = s["k"][off + t].transpose(0, 1).double()
        ring["ring_v"][r][:, slot] = s["v"][off + t].transpose(0, 1).double()
        ring["ring_pos"][r][:, slot] = (start + t).to(torch.int32)[None]
        off += n
    return {"out": torch.cat(outs) * torch.sigmoid(s["gate"].double()), **ring}


def _exact_memory_prefill(case, s):
    st = {f: _wide(getattr(s["state"], f)) for f in MEMORY_FIELDS}
    b, n, cap = case["batch"], case["length"], case["capacity"]
    rep = HEADS // GROUPS
    out = torch.zeros(b, n, HEADS, D, device="cuda", dtype=torch.float64)
    for r in range(b):
        count = n if s["valid"] is None else int(s["valid"][r].sum())
        old, base = int(st["count"][r]), int(st["total"][r]) - int(st["count"][r])
        k = torch.cat((st["pending_keys"][r, :, :old], s["k"][r, :count].double().transpose(0, 1)), 1)
        v = torch.cat((st["pending_values"][r, :, :old], s["v"][r, :count].double().transpose(0, 1)), 1)
        sc = torch.cat((st["pending_scores"][r, :, :old], s["scores"][r, :count].double().t()), 1)
        mem = {f: st[f][r] for f in ("keys", "values", "scores")}
        mem["positions"] = st["positions"][r].long()
        take = _rank(mem["scores"], mem["positions"])

        def gather(m, take):
            return {f: x.gather(1, take[..., None].expand(-1, -1, D) if x.ndim == 3 else take) for f, x in m.items()}

        mem, total = gather(mem, take), old + count
        for c0 in range(0, max(total, 1), CHUNK):
            c1 = min(total, c0 + CHUNK)
            t0, t1 = max(c0 - old, 0), c1 - old       # the block's new tokens
            if t1 > t0:
                q = s["q"][r, t0:t1].double().view(t1 - t0, GROUPS, rep * D).transpose(0, 1)
                q = q.reshape(GROUPS, (t1 - t0) * rep, D)
                logits = q @ mem["keys"].transpose(1, 2).contiguous() / math.sqrt(D)
                w = F.pad(logits.masked_fill((mem["positions"] < 0)[:, None], -math.inf), (0, 1)).softmax(-1)
                got = (w[..., :cap] @ mem["values"]).view(GROUPS, t1 - t0, rep * D).transpose(0, 1)
                out[r, t0:t1] = got.reshape(t1 - t0, HEADS, D)
            if c1 - c0 == CHUNK:
                pos = torch.arange(base + c0, base + c1, device="cuda").expand(GROUPS, -1)
                new = {"keys": k[:, c0:c1], "values": v[:, c0:c1], "scores": sc[:, c0:c1], "positions": pos}
                both = {f: torch.cat((mem[f], new[f]), 1) for f in mem}
                mem = gather(both, _rank(both["scores"], both["positions"])[:, :cap])
        for f in mem:
            st[f][r] = mem[f].to(st[f].dtype)
        gone = st["positions"][r] < 0
        st["keys"][r][gone], st["values"][r][gone] = 0, 0
        left, full = total % CHUNK, total // CHUNK * CHUNK
        for f, x, fill in (("pending_keys", k, 0), ("pending_values", v, 0), ("pending_scores", sc, -math.inf)):
            st[f][r].fill_(fill)
            st[f][r][:, :left] = x[:, full:]
        st["count"][r], st["total"][r] = left, st["total"][r] + count
    return {"out": out, **st}


def _exact_attention_decode(case, s):
    st = {f: _wide(getattr(s["state"], f)) for f in MEMORY_FIELDS}
    att = _attend64(s["q"][:, 0].double(), s["ring_k"].double(), s["ring_v"].double(), s["ring_pos"] >= 0, sink=False)
    read = _attend64(s["mq"][:, 0].double(), st["keys"], st["values"], st["positions"] >= 0, sink=True)
    read = read * s["valid"][:, None, None] * s["head_gate"].double()[..., None]
    _commit64(st, s["key"][:, 0].double(), s["value"][:, 0].double(), s["scores"][:, 0].double(), s["valid"])
    return {"att": (att * torch.sigmoid(s["gate"].double()))[:, None], "read": read[:, None], **st}


def exact(case, seed):
    if case["kind"] == "sample":                      # whole numbers: compared as they are
        return None
    return globals()["_exact_" + case["kind"]](case, prepare(case, seed))
