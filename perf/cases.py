"""What the performance of this framework is measured on: the calls that serving spends its time in, with their inputs, the work each
cannot do without, and what plain float64 arithmetic gives for the same inputs.

Decode steps run through ``ModelRunner`` (staged metadata, captured graph, logits), the kernels of the single layers through ``ops`` and
``hybrid_ops`` as the models' layers call them, on what a layer has in hand: packed projections, pages in shuffled order, per-sequence
state.  Everything is bfloat16, the type that models are served in (float32 runs for comparisons).  Sizes are those of layers
like Qwen3-0.6B's and Qwen3-8B's; sequences of a batch have different lengths, most of them multiples of nothing."""
from __future__ import annotations

import math

import numpy as np
import torch

DEV, BF16, F64 = "cuda", torch.bfloat16, torch.float64
BLOCK = 256
# hidden size, feed-forward, query heads, layers of a published model
LIKE = {"0.6b": (1024, 3072, 16, 28), "8b": (4096, 12288, 32, 36)}
VOCAB, KV_HEADS, DIM, ROPE_BASE, EPS = 151936, 8, 128, 1e6, 1e-6


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one user, one model of 0.6B: every step is as long as its launches take
        {"name": "step_single", "kind": "step", "like": "0.6b", "layers": 28, "batch": 1, "lo": 700, "hi": 700},
        # a loaded server: four of the 36 layers of an 8B model and its head, 64 sequences of the engine's usual lengths
        {"name": "step_batch", "kind": "step", "like": "8b", "layers": 4, "batch": 64, "lo": 128, "hi": 1280},
        # decode attention of one layer: a few short sequences, and a batch of long ones
        {"name": "decode_small", "kind": "decode", "heads": 16, "batch": 4, "lo": 37, "hi": 1023},
        {"name": "decode_ragged", "kind": "decode", "heads": 32, "batch": 64, "lo": 512, "hi": 4096},
        # new prompts: norms, rotary positions and append in front of causal attention over the packed rows
        {"name": "prefill_ragged", "kind": "prefill", "heads": 32, "seqs": 16, "lo": 64, "hi": 2048},
        # prompts of the other designs: attention of two maps within chunks, over gathered pages
        {"name": "masked_prefill", "kind": "masked", "heads": 32, "maps": 2, "mask": "chunk", "size": 2048, "bias": False, "seqs": 6,
         "lo": 1100, "hi": 3000, "prefix": 0},
        # talking heads over tiled pages
        {"name": "talking_prefill", "kind": "talking", "heads": 16, "seqs": 8, "lo": 700, "hi": 2300, "prefix": 0},
        # the recurrences over prompts: gated delta rule, constant decay, selective state space
        {"name": "delta_prefill", "kind": "delta", "heads": 32, "seqs": 8, "lo": 500, "hi": 2600},
        {"name": "decay_prefill", "kind": "decay", "heads": 32, "form": "lightning", "seqs": 6, "lo": 900, "hi": 3700},
        {"name": "state_space_prefill", "kind": "state_space", "heads": 64, "seqs": 6, "lo": 900, "hi": 3700},
        # mixture of experts and the residual step that sums its rows: a decode batch, and a step of prompts
        {"name": "experts_decode", "kind": "experts", "width": 4096, "ff": 3072, "rows": 64},
        {"name": "experts_prefill", "kind": "experts", "width": 4096, "ff": 3072, "rows": 8000},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def ragged(tokens, longest):
        """A few to many sequences, in all about ``tokens`` tokens."""
        hi = size(64, longest)
        lo = max(2, int(hi * rng.uniform(0.1, 1.0)))
        return {"seqs": max(1, min(64, int(tokens / ((lo + hi) / 2)))), "lo": lo, "hi": hi}

    kind = rng.choice(["step", "decode", "decode", "prefill", "masked", "talking", "delta", "decay", "state_space", "experts"])
    heads = rng.choice([16, 32])
    if kind == "step":
        like, lo = rng.choice(["0.6b", "8b"]), size(100, 1000)
        return {"kind": kind, "like": like, "layers": 14 if like == "0.6b" else 3, "batch": size(1, 64), "lo": lo, "hi": lo + size(1, 900)}
    if kind == "decode":
        batch, lo = size(1, 128), size(16, 4096)
        return {"kind": kind, "heads": heads, "batch": batch, "lo": lo, "hi": lo + size(1, max(2, min(8000, 200000 // batch)))}
    if kind == "prefill":
        return {"kind": kind, "heads": heads, **ragged(size(500, 16000), 8192)}
    if kind == "masked":
        mask, maps = rng.choice(["window", "chunk"]), rng.choice([1, 2])
        case = {"kind": kind, "heads": heads, "maps": maps, "mask": mask, "size": rng.choice([512, 1024, 2048]),
                "bias": mask == "chunk" and maps == 1, **ragged(size(500, 12000), 6000)}
        return {**case, "prefix": rng.choice([0, size(100, 3000)]) if case["seqs"] < 9 else 0}
    if kind == "talking":
        case = {"kind": kind, "heads": 16, **ragged(size(500, 12000), 6000)}
        return {**case, "prefix": rng.choice([0, size(100, 2000)]) if case["seqs"] < 9 else 0}
    if kind in ("delta", "decay", "state_space"):
        case = {"kind": kind, "heads": 2 * heads if kind == "state_space" else heads, **ragged(size(300, 14000), 14000)}
        return {**case, "form": rng.choice(["lightning", "retention"])} if kind == "decay" else case
    width, ff = rng.choice([(1024, 768), (4096, 3072)])
    return {"kind": kind, "width": width, "ff": ff, "rows": size(1, 8000)}


def lengths(case):
    """The lengths of the batch's sequences: spread over the range, in an order of no meaning."""
    n, lo, hi = case.get("batch", case.get("seqs")), case["lo"], case["hi"]
    return [lo + int((hi - lo + 1) * (((i + 1) * 0.6180339887) % 1.0)) if hi > lo else lo for i in range(n)]


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)


def _rnd(gen, *shape, dtype=BF16, std=1.0):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _pages(lens, gen):
    """(block table with -1 behind a sequence's blocks, number of blocks): every block is somewhere else."""
    per = [-(-n // BLOCK) for n in lens]
    blocks = sum(per) + 3
    order = torch.randperm(blocks, generator=gen, device=DEV).tolist()
    table, at = np.full((len(lens), max(per)), -1, np.int32), 0
    for i, n in enumerate(per):
        table[i, :n] = order[at:at + n]
        at += n
    return torch.from_numpy(table).to(DEV), blocks


def _slots(table, lens):
    """The cache row of every token of every sequence, one after the other."""
    out = []
    for row, n in zip(table.cpu().numpy(), lens):
        p = np.arange(n)
        out.append(row[p // BLOCK].astype(np.int64) * BLOCK + p % BLOCK)
    return np.concatenate(out)


def _cu(lens):
    return _ints(np.concatenate(([0], np.cumsum(lens))).tolist())


def _spans(lens):
    first = np.concatenate(([0], np.cumsum(lens)))[:-1]
    spans = _ints([(int(r), n, i, 0) for i, (r, n) in enumerate(zip(first, lens))])
    ring = np.concatenate([np.stack((np.full(n, i), np.arange(n - 1, -1, -1)), 1) for i, n in enumerate(lens)]).astype(np.int32)
    positions = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(DEV)
    return spans, torch.from_numpy(ring).to(DEV), positions


def _rope_table(positions, dim=DIM, base=ROPE_BASE):
    """Cosines and sines of the rotary embedding in the precision of the model that the framework serves: bfloat16 throughout."""
    inv = 1.0 / (base ** (torch.arange(0, dim, 2, dtype=BF16, device=DEV) / dim))
    freqs = torch.arange(positions, dtype=BF16, device=DEV)[:, None] * inv
    return torch.cat((freqs.cos(), freqs.sin()), -1).contiguous()


def _angles(dims, positions, base=1e4):
    """[positions, dims / 2, 2] float32 cosines and sines."""
    freq = base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=DEV) / dims)
    a = torch.arange(positions, dtype=F64, device=DEV)[:, None] * freq
    return torch.stack((a.cos(), a.sin()), -1).float().contiguous()


def _step_weights(case, seed):
    """Name -> tensor of a Qwen3 model's weights."""
    width, ff, heads, _ = LIKE[case["like"]]
    gen, w = _gen(seed), {}
    w["model.embed_tokens.weight"] = _rnd(gen, VOCAB, width)       # layers add to it what is small beside it, as in trained models
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        w[p + "self_attn.qkv_proj.weight"] = _rnd(gen, (heads + 2 * KV_HEADS) * DIM, width, std=0.02)
        w[p + "self_attn.o_proj.weight"] = _rnd(gen, width, heads * DIM, std=0.02)
        w[p + "mlp.gate_up_proj.weight"] = _rnd(gen, 2 * ff, width, std=0.02)
        w[p + "mlp.down_proj.weight"] = _rnd(gen, width, ff, std=0.02)
        for name, size in (("self_attn.q_norm", DIM), ("self_attn.k_norm", DIM), ("input_layernorm", width), ("post_attention_layernorm", width)):
            w[p + name + ".weight"] = (1.0 + _rnd(gen, size, dtype=torch.float32, std=0.1)).to(BF16)
    w["model.norm.weight"] = (1.0 + _rnd(gen, width, dtype=torch.float32, std=0.1)).to(BF16)
    if case["like"] == "8b":
        w["lm_head.weight"] = _rnd(gen, VOCAB, width, std=0.02)
    return w


def _step_inputs(case, seed):
    """Tokens of every sequence (the last one is the step's), its blocks, and what fills the cache."""
    lens, gen, rng = lengths(case), _gen(seed + 1), np.random.default_rng(seed)
    table, blocks = _pages(lens, gen)
    tokens = [[int(t) for t in rng.integers(0, VOCAB, size=n)] for n in lens]
    cache = _rnd(gen, 2, case["layers"], blocks, BLOCK, KV_HEADS, DIM)
    return lens, tokens, table, blocks, cache


def _prepare_step(case, seed):
    from infer_amd.config import Config, ModelConfig
    from infer_amd.model_runner import ModelRunner
    from infer_amd.sequence import Sequence
    width, ff, heads, _ = LIKE[case["like"]]
    lens, tokens, table, blocks, cache = _step_inputs(case, seed)
    batch = case["batch"]
    slots = next(b for b in [1, 2, 4, 8] + list(range(16, 1024, 16)) if b >= batch)
    hf = ModelConfig(hidden_size=width, intermediate_size=ff, num_hidden_layers=case["layers"], num_attention_heads=heads,
                     tie_word_embeddings=case["like"] == "0.6b", rope_theta=ROPE_BASE, rms_norm_eps=EPS)
    longest = max(2048, max(lens) + 1)
    runner = ModelRunner(Config(hf_config=hf, max_num_seqs=slots, max_model_len=longest, max_num_batched_tokens=longest,
                                num_kvcache_blocks=blocks, decode_position_offset=0, kvcache_block_size=BLOCK, seed=seed))
    weights = _step_weights(case, seed)
    for name, p in runner.model.named_parameters():
        p.data.copy_(weights[name])
    runner.kv_cache.copy_(cache)
    seqs = []
    for ids, row in zip(tokens, table.tolist()):
        seq = Sequence(ids)
        seq.block_table = [b for b in row if b >= 0]
        seqs.append(seq)
    return {"runner": runner, "seqs": seqs}


def _decode_inputs(case, seed):
    lens, gen = lengths(case), _gen(seed)
    table, blocks = _pages(lens, gen)
    return {"lens": lens, "q": _rnd(gen, case["batch"], 1, case["heads"], DIM), "table": table,
            "k": _rnd(gen, blocks, BLOCK, KV_HEADS, DIM), "v": _rnd(gen, blocks, BLOCK, KV_HEADS, DIM), "ctx": _ints(lens)}


def _prefill_inputs(case, seed):
    lens, gen, heads = lengths(case), _gen(seed), case["heads"]
    table, blocks = _pages(lens, gen)
    return {"lens": lens, "cu": _cu(lens), "max": max(lens), "heads": heads,
            "qkv": _rnd(gen, sum(lens), (heads + 2 * KV_HEADS) * DIM), "slots": torch.from_numpy(_slots(table, lens).astype(np.int32)).to(DEV),
            "positions": torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(DEV),
            "q_norm": (1.0 + _rnd(gen, DIM, std=0.1)), "k_norm": (1.0 + _rnd(gen, DIM, std=0.1)), "table": _rope_table(max(lens)),
            "k_cache": torch.zeros(blocks, BLOCK, KV_HEADS, DIM, dtype=BF16, device=DEV),
            "v_cache": torch.zeros(blocks, BLOCK, KV_HEADS, DIM, dtype=BF16, device=DEV)}


def _masked_inputs(case, seed):
    lens, gen, heads, maps = lengths(case), _gen(seed), case["heads"], case["maps"]
    keys = [n + case["prefix"] for n in lens]
    table, blocks = _pages(keys, gen)
    return {"lens": lens, "keys": keys, "tables": table, "cache": _rnd(gen, blocks, KV_HEADS, BLOCK, 2 * DIM),
            "q": _rnd(gen, sum(lens), heads * DIM), "gate": _rnd(gen, sum(lens), heads) if maps == 2 else None,
            "sink": _rnd(gen, heads, dtype=torch.float32) if case["bias"] else None,
            "seqs": _ints(range(len(lens))), "cu_q": _cu(lens), "cu_k": _cu(keys)}


def _masked_shape(case):
    from infer_amd.hybrid_ops import MaskedShape
    maps = case["maps"]
    return MaskedShape(case["heads"], KV_HEADS, DIM // maps, DIM, (DIM // maps) ** -0.5, maps=maps, mask=case["mask"], mask_size=case["size"],
                       distance_bias=case["bias"], lam=0.4, out_scale=0.5 if maps == 2 else 1.0, eps=EPS, rot_dims=64)


def _talking_inputs(case, seed):
    lens, gen, heads = lengths(case), _gen(seed), case["heads"]
    keys = [n + case["prefix"] for n in lens]
    table, blocks = _pages(keys, gen)
    talk = (torch.eye(heads, device=DEV) + _rnd(gen, heads, heads, dtype=torch.float32, std=0.2)).to(BF16)
    # packed projections of every token, those of the prefixes too
    return {"lens": lens, "keys": keys, "tables": table, "blocks": blocks, "talk": talk, "proj": _rnd(gen, sum(keys), (heads + 2 * KV_HEADS) * DIM),
            "seqs": _ints(range(len(lens))), "cu_q": _cu(lens), "cu_k": _cu(keys)}


def _fill_tiles(case, s):
    """Pages with the keys and values of all tokens, and the queries of the new ones."""
    from infer_amd import hybrid_ops
    from infer_amd.cache import TilePages
    heads, shape, keys = case["heads"], s["shape"], s["keys"]
    pages = TilePages(KV_HEADS, DIM, DIM, BF16).allocate(s["blocks"], 0, BLOCK, DEV)
    proj, n = s.pop("proj"), sum(keys)
    hybrid_ops.unit_head_front(shape, proj, [0, heads * DIM, (heads + KV_HEADS) * DIM], torch.arange(n, device=DEV),
                               torch.from_numpy(_slots(s["tables"], keys).astype(np.int32)).to(DEV), pages["keys"], pages["values"],
                               torch.empty(1, heads, DIM, dtype=BF16, device=DEV), 0)
    s["q"] = proj[:, :heads * DIM] if not case["prefix"] else torch.cat([x[-m:, :heads * DIM] for x, m in zip(proj.split(keys), s["lens"])])
    s["k_pages"], s["v_pages"] = pages["keys"], pages["values"]
    s["out"] = torch.zeros(sum(s["lens"]), heads * DIM, dtype=BF16, device=DEV)


def _delta_inputs(case, seed):
    lens, gen, heads = lengths(case), _gen(seed), case["heads"]
    t, channels = sum(lens), 3 * heads * DIM
    first = np.concatenate(([0], np.cumsum(lens)))
    portions, chunks = [], []
    for i, n in enumerate(lens):
        portions.append((len(chunks), -(-n // 16), i, 0))
        chunks += [(int(first[i]) + c, min(16, n - c), c, 0, i, 0) for c in range(0, n, 16)]
    _, ring, positions = _spans(lens)
    return {"lens": lens, "proj": _rnd(gen, t, -(-(channels + heads) // 64) * 64), "decay": _rnd(gen, t, heads * DIM), "gate": _rnd(gen, t, heads * DIM),
            "conv": _rnd(gen, channels, 4, dtype=torch.float32, std=0.5), "a_log": _rnd(gen, heads, dtype=torch.float32, std=0.5),
            "dt_bias": _rnd(gen, heads * DIM, dtype=torch.float32) - 4.0, "norm": 1.0 + _rnd(gen, DIM, dtype=torch.float32, std=0.1),
            "ring": torch.zeros(len(lens), 4, channels, dtype=BF16, device=DEV), "state": torch.zeros(len(lens), heads, DIM, DIM, device=DEV),
            "portions": _ints(portions), "chunks": _ints(chunks), "ring_slot": ring, "positions": positions,
            "out": torch.zeros(t, heads * DIM, dtype=BF16, device=DEV)}


def _decay_of(heads):
    return [1.0 - 2.0 ** (-4.0 - 7.0 * h / heads) for h in range(heads)]


def _decay_inputs(case, seed):
    lens, gen, heads = lengths(case), _gen(seed), case["heads"]
    spans, _, _ = _spans(lens)
    light = case["form"] == "lightning"
    return {"lens": lens, "proj": _rnd(gen, sum(lens), 4 * heads * DIM), "spans": spans,
            "table": None if light else _angles(DIM, max(lens)),
            "norm": 1.0 + _rnd(gen, heads * DIM, dtype=torch.float32, std=0.1) if light else None,
            "state": torch.zeros(len(lens), heads, DIM, DIM, device=DEV), "out": torch.zeros(sum(lens), heads * DIM, dtype=BF16, device=DEV)}


def _state_space_inputs(case, seed):
    lens, gen, heads = lengths(case), _gen(seed), case["heads"]
    inner, channels = heads * 64, heads * 64 + 2 * 2 * DIM
    spans, ring, positions = _spans(lens)
    t = sum(lens)
    return {"lens": lens, "proj": _rnd(gen, t, -(-(inner + channels + heads) // 64) * 64), "spans": spans, "ring_slot": ring, "positions": positions,
            "conv": _rnd(gen, channels, 4, dtype=torch.float32, std=0.5), "conv_bias": _rnd(gen, channels, dtype=torch.float32, std=0.1),
            "dt_bias": _rnd(gen, heads, dtype=torch.float32) - 3.0, "a_log": _rnd(gen, heads, dtype=torch.float32, std=0.5),
            "d": 1.0 + _rnd(gen, heads, dtype=torch.float32, std=0.1), "norm": 1.0 + _rnd(gen, inner, dtype=torch.float32, std=0.1),
            "ring": torch.zeros(len(lens), 4, channels, dtype=BF16, device=DEV),
            "state": torch.zeros(len(lens), heads, DIM, 64, device=DEV), "out": torch.zeros(t, inner, dtype=BF16, device=DEV)}


EXPERTS, IDENTITY, TOP, GROUPS, KEEP = 14, 2, 3, 4, 2


def _experts_inputs(case, seed):
    gen, width, ff, n = _gen(seed), case["width"], case["ff"], case["rows"]
    return {"h": _rnd(gen, n, width), "router": _rnd(gen, EXPERTS + IDENTITY, width, std=0.02),
            "correction": _rnd(gen, EXPERTS + IDENTITY, dtype=torch.float32, std=0.01),
            "gate_up": _rnd(gen, EXPERTS, 2 * ff, width, std=0.02), "down": _rnd(gen, EXPERTS, width, ff, std=0.02),
            "counts": torch.zeros(EXPERTS, dtype=torch.int32, device=DEV), "x": _rnd(gen, n, width, dtype=torch.float32),
            "scale": 1.0 + _rnd(gen, width, dtype=torch.float32, std=0.1), "w": 1.0 + _rnd(gen, width, dtype=torch.float32, std=0.1)}


INPUTS = {"decode": _decode_inputs, "prefill": _prefill_inputs, "masked": _masked_inputs, "talking": _talking_inputs, "delta": _delta_inputs,
          "decay": _decay_inputs, "state_space": _state_space_inputs, "experts": _experts_inputs}


def prepare(case, seed):
    if case["kind"] == "step":
        return {"kind": "step", **_prepare_step(case, seed)}
    from infer_amd import hybrid_ops
    state = {"kind": case["kind"], **INPUTS[case["kind"]](case, seed)}
    heads = case.get("heads", 0)
    if case["kind"] == "masked":
        state["shape"] = _masked_shape(case)
        state["out"] = torch.zeros(sum(state["lens"]), heads * DIM, dtype=BF16, device=DEV)
    elif case["kind"] == "talking":
        state["shape"] = hybrid_ops.TalkShape(heads, KV_HEADS, DIM, DIM, DIM ** -0.5, EPS)
        _fill_tiles(case, state)
    elif case["kind"] == "delta":
        state["shape"] = hybrid_ops.DeltaShape(heads, heads, DIM, DIM, 4, EPS)
    elif case["kind"] == "decay":
        light = case["form"] == "lightning"
        state["shape"] = hybrid_ops.DecayShape(heads, DIM, DIM, EPS, light, 0 if light else DIM, 1.0 if light else DIM ** -0.5, not light, not light)
        state["constants"] = hybrid_ops.decay_constants(_decay_of(heads), DEV)
    elif case["kind"] == "state_space":
        state["shape"] = hybrid_ops.StateSpaceShape(heads, 64, DIM, 2, 4, 2, EPS)
    elif case["kind"] == "experts":
        state["shape"] = hybrid_ops.MoeShape(case["width"], case["ff"], EXPERTS, TOP, IDENTITY, GROUPS, KEEP, 2.0)
    return state


# ------------------------------------------------------------------ one pass
def run(s):
    from infer_amd import hybrid_ops as ho, ops
    kind = s["kind"]
    if kind == "step":
        return s["runner"].run_model(s["seqs"], False)
    if kind == "decode":
        return ops.flash_attn_with_kvcache(s["q"], s["k"], s["v"], cache_seqlens=s["ctx"], block_table=s["table"], softmax_scale=DIM ** -0.5,
                                           causal=True)
    if kind == "prefill":
        q, k, v = (x.view(x.shape[0], -1, DIM) for x in s["qkv"].split([s["heads"] * DIM, KV_HEADS * DIM, KV_HEADS * DIM], dim=-1))
        ops.qk_norm_rope_store_kvcache(q, k, v, s["positions"], s["q_norm"], s["k_norm"], EPS, s["table"], s["k_cache"], s["v_cache"], s["slots"],
                                       write_key=True)
        o = ops.flash_attn_varlen_func(q, k, v, max_seqlen_q=s["max"], cu_seqlens_q=s["cu"], max_seqlen_k=s["max"], cu_seqlens_k=s["cu"],
                                       softmax_scale=DIM ** -0.5, causal=True)
        return {"out": o, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "masked":
        rows = ho.masked_gather(s["shape"], s["cache"], s["tables"], s["seqs"], s["cu_q"], s["cu_k"], sum(s["keys"]), max(s["keys"]))
        ho.masked_prefill(s["shape"], s["q"], rows, s["out"], s["cu_q"], s["cu_k"], max(s["lens"]), s["sink"], s["gate"])
        return s["out"]
    if kind == "talking":
        ho.talking_prefill(s["shape"], s["q"], s["k_pages"], s["v_pages"], s["talk"], s["tables"], s["seqs"], s["cu_q"], s["cu_k"],
                           max(s["lens"]), max(s["keys"]), s["out"], max_score=s["shape"].max_score(max(s["keys"])))
        return s["out"]
    if kind == "delta":
        ho.delta_chunks(s["shape"], s["proj"], s["shape"].channels, s["decay"], s["gate"], s["conv"], s["a_log"], s["dt_bias"], s["norm"], s["ring"],
                        s["state"], s["portions"], s["chunks"], s["ring_slot"], s["positions"], 0, s["out"])
        return {"out": s["out"], "state": s["state"], "ring": s["ring"]}
    if kind == "decay":
        hd = s["shape"].heads * DIM
        ho.decay_attention(s["shape"], s["proj"], [0, hd, 2 * hd, 3 * hd], s["constants"], s["table"], s["norm"], s["state"], None, None, 0, s["spans"],
                           max(s["lens"]), s["out"])
        return {"out": s["out"], "state": s["state"]}
    if kind == "state_space":
        inner, channels = s["shape"].inner, s["shape"].channels
        ho.state_space(s["shape"], s["proj"], (0, inner, inner + channels), s["conv"], s["conv_bias"], s["dt_bias"], s["a_log"], s["d"], s["norm"], s["ring"],
                       s["state"], None, s["positions"], 0, s["spans"], max(s["lens"]), s["ring_slot"], s["out"])
        return {"out": s["out"], "state": s["state"], "ring": s["ring"]}
    y = ho.moe(s["shape"], s["h"], s["router"], s["correction"], s["gate_up"], s["down"], s["counts"])
    h = ho.pre_norm(s["x"], s["w"], EPS, y=y, scale=s["scale"])
    return {"h": h, "x": s["x"]}


# ------------------------------------------------------------------ the work of a pass
def _visible(case):
    """(query, key) pairs that the mask shows, over all sequences."""
    pairs, p = 0, case.get("prefix", 0)
    for n in lengths(case):
        at = np.arange(p, p + n, dtype=np.int64)
        seen = at + 1
        if case.get("mask") == "window":
            seen = np.minimum(seen, case["size"])
        elif case.get("mask") == "chunk":
            seen = at % case["size"] + 1
        pairs += int(seen.sum())
    return pairs


def work(case):
    kind = case["kind"]
    if kind == "experts":
        width, ff, n = case["width"], case["ff"], case["rows"]
        share = EXPERTS / (EXPERTS + IDENTITY) * TOP * n            # rows that meet an expert
        used = EXPERTS * (1.0 - (1.0 - TOP / (EXPERTS + IDENTITY)) ** n)
        return {"bytes": used * 3 * width * ff * 2 + n * width * (2 + 4 + 4 + 2), "flops": 2 * share * 3 * width * ff}
    if kind == "step":
        width, ff, heads, _ = LIKE[case["like"]]
        layer = width * ((2 * heads + 2 * KV_HEADS) * DIM + 3 * ff)
        weights = case["layers"] * layer + VOCAB * width
        cached = sum(lengths(case)) * case["layers"] * 2 * KV_HEADS * DIM
        return {"bytes": 2 * (weights + cached + case["batch"] * VOCAB), "flops": 2 * case["batch"] * weights + 2 * cached * heads // KV_HEADS}
    heads, lens = case["heads"], lengths(case)
    t = sum(lens)
    if kind == "decode":
        return {"bytes": 2 * (t * 2 * KV_HEADS * DIM + 2 * len(lens) * heads * DIM), "flops": 4 * t * heads * DIM}
    if kind == "prefill":
        return {"bytes": 2 * t * DIM * (2 * heads + 4 * KV_HEADS), "flops": 4 * heads * DIM * _visible(case)}
    if kind in ("masked", "talking"):
        keys = t + len(lens) * case["prefix"]
        mix = 2 * heads * heads if kind == "talking" else 0
        maps = case.get("maps", 1)
        return {"bytes": 2 * DIM * (2 * t * heads + 2 * keys * KV_HEADS), "flops": (2 * heads * DIM * (1 + maps) + mix) * _visible(case)}
    state = 4 * len(lens) * heads * DIM * (64 if kind == "state_space" else DIM)
    if kind == "delta":
        return {"bytes": 2 * t * 6 * heads * DIM + state, "flops": t * heads * 6 * DIM * DIM}
    if kind == "decay":
        return {"bytes": 2 * t * 5 * heads * DIM + state, "flops": t * heads * 4 * DIM * DIM}
    return {"bytes": 2 * t * (3 * heads * 64 + 4 * DIM + heads) + state, "flops": t * heads * 4 * DIM * 64}


def tolerance(case):
    # a step passes a dozen to two hundred roundings to bfloat16 one after the other (0.01 to 0.016 off float64), the others one to four (0.002 to 0.004)
    return {"rel": 0.03, "max": 0.5} if case["kind"] == "step" else {"rel": 0.01, "max": 0.2}


# ------------------------------------------------------------------ the same in float64
def _rms(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope(x, table, positions):
    """Rotates entry i with entry i + half; ``x`` [tokens, heads, dim]."""
    half = x.shape[-1] // 2
    c, s = table[positions].double()[:, None].split(half, -1)
    u, v = x.split(half, -1)
    return torch.cat((u * c - v * s, v * c + u * s), -1)


def _softmax_attention(q, k, v, scale, visible, sink=None, bias=None):
    """``q`` [queries, heads, n], ``k``/``v`` [keys, kv heads, n]; a block of queries at a time."""
    group = q.shape[1] // k.shape[1]
    kh, vh = (x.repeat_interleave(group, 1).transpose(0, 1) for x in (k, v))
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=F64, device=DEV)
    for lo in range(0, q.shape[0], 512):
        hi = min(lo + 512, q.shape[0])
        s = q[lo:hi].transpose(0, 1) @ kh.transpose(1, 2) * scale
        if bias is not None:
            s = s + bias(lo, hi)
        if visible is not None:
            s = s.masked_fill(~visible(lo, hi), -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink.double()[:, None, None])
        p = torch.exp(s - top)
        z = p.sum(-1, keepdim=True)
        if sink is not None:
            z = z + torch.exp(sink.double()[:, None, None] - top)
        out[lo:hi] = ((p / z) @ vh).transpose(0, 1)
    return out


def _exact_step(case, seed):
    width, ff, heads, _ = LIKE[case["like"]]
    lens, tokens, table, _, cache = _step_inputs(case, seed)
    w = _step_weights(case, seed)
    rope, b = _rope_table(max(lens)), len(lens)
    pos = torch.tensor([n - 1 for n in lens], device=DEV)
    x = w["model.embed_tokens.weight"][[t[-1] for t in tokens]].double()
    for i in range(case["layers"]):
        def p(name):
            return w[f"model.layers.{i}.{name}.weight"].double()
        qkv = _rms(x, p("input_layernorm")) @ p("self_attn.qkv_proj").T
        q, k, v = (y.view(b, -1, DIM) for y in qkv.split([heads * DIM, KV_HEADS * DIM, KV_HEADS * DIM], -1))
        q, k = _rope(_rms(q, p("self_attn.q_norm")), rope, pos), _rope(_rms(k, p("self_attn.k_norm")), rope, pos)
        o = torch.empty(b, heads, DIM, dtype=F64, device=DEV)
        for j, n in enumerate(lens):
            rows = torch.from_numpy(_slots(table[j:j + 1], [n])).to(DEV)
            kj, vj = (cache[c, i].view(-1, KV_HEADS, DIM)[rows].double() for c in range(2))
            kj[-1], vj[-1] = k[j], v[j]
            o[j] = _softmax_attention(q[j:j + 1], kj, vj, DIM ** -0.5, None)[0]
        x = x + o.view(b, -1) @ p("self_attn.o_proj").T
        g, u = (_rms(x, p("post_attention_layernorm")) @ p("mlp.gate_up_proj").T).split(ff, -1)
        x = x + (torch.nn.functional.silu(g) * u) @ p("mlp.down_proj").T
    head = w["lm_head.weight"] if "lm_head.weight" in w else w["model.embed_tokens.weight"]
    return _rms(x, w["model.norm.weight"].double()) @ head.double().T


def _exact_decode(case, s):
    out = torch.empty(s["q"].shape, dtype=F64, device=DEV)
    for j, n in enumerate(s["lens"]):
        rows = torch.from_numpy(_slots(s["table"][j:j + 1], [n])).to(DEV)
        k, v = (s[c].view(-1, KV_HEADS, DIM)[rows].double() for c in ("k", "v"))
        out[j] = _softmax_attention(s["q"][j].double(), k, v, DIM ** -0.5, None)
    return out


def _exact_prefill(case, s):
    heads = s["heads"]
    q, k, v = (x.view(x.shape[0], -1, DIM) for x in s["qkv"].double().split([heads * DIM, KV_HEADS * DIM, KV_HEADS * DIM], -1))
    q, k = (_rope(_rms(x, n.double()), s["table"], s["positions"]) for x, n in ((q, s["q_norm"]), (k, s["k_norm"])))
    out, at, caches = [], 0, []
    for n in s["lens"]:
        def visible(lo, hi, n=n):
            return torch.arange(n, device=DEV)[None] <= torch.arange(lo, hi, device=DEV)[:, None]
        out.append(_softmax_attention(q[at:at + n], k[at:at + n], v[at:at + n], DIM ** -0.5, visible))
        at += n
    for cache, x in ((s["k_cache"], k), (s["v_cache"], v)):
        cache = cache.double()
        cache.view(-1, KV_HEADS, DIM)[s["slots"].long()] = x
        caches.append(cache)
    return {"out": torch.cat(out), "k_cache": caches[0], "v_cache": caches[1]}


def _exact_masked(case, s):
    heads, maps, size, p = case["heads"], case["maps"], case["size"], case["prefix"]
    rows, out, at = s["cache"].transpose(1, 2).reshape(-1, KV_HEADS, 2 * DIM), [], 0
    slopes = 2.0 ** (-8.0 * torch.arange(1, heads + 1, dtype=F64, device=DEV) / heads)
    for j, n in enumerate(s["lens"]):
        kv = rows[torch.from_numpy(_slots(s["tables"][j:j + 1], [n + p])).to(DEV)].double()
        q = s["q"][at:at + n].double().view(n, heads, maps, DIM // maps)

        def back(lo, hi, n=n):
            return torch.arange(p + lo, p + hi, device=DEV)[:, None] - torch.arange(n + p, device=DEV)[None]

        def visible(lo, hi, n=n):
            i, key = torch.arange(p + lo, p + hi, device=DEV)[:, None], torch.arange(n + p, device=DEV)[None]
            return (key <= i) & ((i - key < size) if case["mask"] == "window" else (i // size == key // size))

        def bias(lo, hi):
            return -slopes[:, None, None] * back(lo, hi)
        a = [_softmax_attention(q[:, :, m], kv[:, :, DIM + m * (DIM // maps):DIM + (m + 1) * (DIM // maps)], kv[:, :, :DIM], (DIM // maps) ** -0.5,
                                visible, s["sink"], bias if case["bias"] else None) for m in range(maps)]
        o = a[0]
        if maps == 2:
            o = _rms(a[0] - 0.4 * a[1], 1.0) * 0.5 * torch.sigmoid(s["gate"][at:at + n].double())[..., None]
        out.append(o.reshape(n, -1))
        at += n
    return torch.cat(out)


def _exact_talking(case, s):
    heads, p, out = case["heads"], case["prefix"], []
    group, talk = heads // KV_HEADS, s["talk"].double()
    for rows, n in zip(s["proj"].split(s["keys"]), s["lens"]):
        x = rows.float().view(n + p, -1, DIM)
        x = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)).to(BF16).double().transpose(0, 1)      # as the pages hold them
        q, (k, v) = x[:heads, p:], (y.repeat_interleave(group, 0) for y in x[heads:].split(KV_HEADS))
        for lo in range(0, n, 256):
            hi = min(lo + 256, n)
            hidden = torch.arange(n + p, device=DEV)[None] > torch.arange(p + lo, p + hi, device=DEV)[:, None]
            e = (q[:, lo:hi] @ k.transpose(1, 2) * DIM ** -0.5).masked_fill(hidden, -math.inf).exp()
            w = e / (1.0 + e.sum(-1, keepdim=True))
            mixed = (talk @ w.reshape(heads, -1)).view_as(w)
            out.append((mixed @ v).transpose(0, 1).reshape(hi - lo, -1))
    return torch.cat(out)


def _padded(x, lens):
    """Packed rows [tokens, ...] -> [longest, sequences, ...], zeros behind a sequence."""
    out, at = torch.zeros(max(lens), len(lens), *x.shape[1:], dtype=x.dtype, device=DEV), 0
    for i, n in enumerate(lens):
        out[:n, i] = x[at:at + n]
        at += n
    return out


def _packed(x, lens):
    return torch.cat([x[:n, i] for i, n in enumerate(lens)])


def _conv_silu(x, taps, bias, lens, kept):
    """Causal convolution per channel and silu, and the ring that keeps the last ``kept`` inputs of every sequence."""
    n = taps.shape[1]
    out, ring, at = [], torch.zeros(len(lens), n, x.shape[1], dtype=F64, device=DEV), 0
    for i, length in enumerate(lens):
        y = torch.cat((torch.zeros(n - 1, x.shape[1], dtype=F64, device=DEV), x[at:at + length].double()))
        z = sum(y[j:j + length] * taps[:, j].double() for j in range(n))
        out.append(torch.nn.functional.silu(z + bias.double() if bias is not None else z))
        for pos in range(max(0, length - kept), length):
            ring[i, pos % n] = x[at + pos].double()
        at += length
    return torch.cat(out), ring


def _exact_delta(case, s):
    heads, lens = case["heads"], s["lens"]
    hd, t = heads * DIM, sum(s["lens"])
    y, ring = _conv_silu(s["proj"][:, :3 * hd], s["conv"], None, lens, 4)
    q, k, v = (x.view(t, heads, DIM) for x in y.split(hd, -1))
    q, k = (x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    beta = torch.sigmoid(s["proj"][:, 3 * hd:3 * hd + heads].double())
    step = torch.nn.functional.softplus(s["decay"].double() + s["dt_bias"].double()).view(t, heads, DIM)
    keep = torch.exp(-torch.exp(s["a_log"].double())[:, None] * step)
    q, k, v, beta = (_padded(x, lens) for x in (q * DIM ** -0.5, k, v, beta))
    keep = 1.0 - _padded(1.0 - keep, lens)                     # behind a sequence's end the state stays as it is
    state, o = torch.zeros(len(lens), heads, DIM, DIM, dtype=F64, device=DEV), torch.empty_like(v)
    for i in range(max(lens)):
        state.mul_(keep[i][..., None])
        u = beta[i][..., None] * (v[i] - (k[i][..., None, :] @ state)[..., 0, :])
        state.addcmul_(k[i][..., None], u[..., None, :])
        o[i] = (q[i][..., None, :] @ state)[..., 0, :]
    out = _rms(_packed(o, lens), s["norm"].double()) * torch.sigmoid(s["gate"].double()).view(t, heads, DIM)
    return {"out": out.view(t, hd), "state": state, "ring": ring}


def _linear_scan(q, k, v, keep, lens):
    """S = keep S + k v^T, o = S^T q, for all sequences side by side; ``keep`` [tokens, heads]."""
    keep, q, k, v = 1.0 - _padded(1.0 - keep, lens), *(_padded(x, lens) for x in (q, k, v))
    state, o = torch.zeros(*k.shape[1:], v.shape[-1], dtype=F64, device=DEV), torch.empty_like(v)
    for i in range(max(lens)):
        state.mul_(keep[i][..., None, None]).addcmul_(k[i][..., None], v[i][..., None, :])
        o[i] = (q[i][..., None, :] @ state)[..., 0, :]
    return _packed(o, lens), state


def _exact_decay(case, s):
    heads, lens, light = case["heads"], s["lens"], case["form"] == "lightning"
    t, hd = sum(lens), heads * DIM
    q, k, v, g = (x.view(t, heads, DIM) for x in s["proj"].double().split(hd, -1))
    if light:
        q, k, v = (torch.nn.functional.silu(x) for x in (q, k, v))
    else:
        table = torch.cat((s["table"][..., 0], s["table"][..., 1]), -1)
        at = torch.cat([torch.arange(n, device=DEV) for n in lens])
        q, k = _rope(q, table, at), _rope(k, table, at)
    keep = torch.tensor(_decay_of(heads), dtype=F64, device=DEV).expand(t, heads)
    o, state = _linear_scan(q, k, v, keep, lens)
    o = o * (1.0 if light else DIM ** -0.5)
    out = _rms(o.reshape(t, hd), s["norm"].double()) * torch.sigmoid(g.reshape(t, hd)) if light else (_rms(o, 1.0) * torch.nn.functional.silu(g)).view(t, hd)
    return {"out": out, "state": state}


def _exact_state_space(case, s):
    heads, lens = case["heads"], s["lens"]
    t, inner = sum(lens), heads * 64
    channels = inner + 4 * DIM
    y, ring = _conv_silu(s["proj"][:, inner:inner + channels], s["conv"], s["conv_bias"], lens, 3)
    x = y[:, :inner].view(t, heads, 64)
    b, c = (z.reshape(t, 2, DIM).repeat_interleave(heads // 2, 1) for z in y[:, inner:].split(2 * DIM, -1))
    dt = torch.nn.functional.softplus(s["proj"][:, inner + channels:inner + channels + heads].double() + s["dt_bias"].double())
    keep = torch.exp(-torch.exp(s["a_log"].double()) * dt)
    o, state = _linear_scan(c, b, x * dt[..., None], keep, lens)
    o = (o + s["d"].double()[:, None] * x).reshape(t, inner) * torch.nn.functional.silu(s["proj"][:, :inner].double())
    return {"out": _rms(o.view(t, 2, inner // 2), 1.0).reshape(t, inner) * s["norm"].double(), "state": state, "ring": ring}


def _exact_experts(case, s):
    h, n, ff = s["h"].double(), case["rows"], case["ff"]
    p = torch.softmax(h @ s["router"].double().T, -1)
    choice = p + s["correction"].double()
    best = choice.view(n, GROUPS, -1).amax(-1).topk(KEEP, -1).indices
    shut = torch.ones(n, GROUPS, dtype=torch.bool, device=DEV).scatter_(1, best, False)
    chosen = choice.masked_fill(shut.repeat_interleave((EXPERTS + IDENTITY) // GROUPS, 1), -math.inf).topk(TOP, -1).indices
    weight, y = 2.0 * p.gather(1, chosen), torch.zeros_like(h)
    for e in range(EXPERTS + IDENTITY):
        rows, place = torch.nonzero(chosen == e, as_tuple=True)
        z = h[rows]
        if e < EXPERTS and len(rows):
            g, u = (z @ s["gate_up"][e].double().T).split(ff, -1)
            z = (torch.nn.functional.silu(g) * u) @ s["down"][e].double().T
        y.index_add_(0, rows, weight[rows, place][:, None] * z)
    x = s["x"].double() + y * s["scale"].double()
    return {"h": _rms(x, s["w"].double()), "x": x}


EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "masked": _exact_masked, "talking": _exact_talking, "delta": _exact_delta,
         "decay": _exact_decay, "state_space": _exact_state_space, "experts": _exact_experts}


def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    return EXACT[case["kind"]](case, INPUTS[case["kind"]](case, seed))
