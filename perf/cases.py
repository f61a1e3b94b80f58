"""Workloads of the paged KV-cache attention path, as a serving program runs it.

A case is a dict of plain values; `prepare` fills a cache (or a page pool) the way a server that has been
running for a while has it, `run` is one step of that server: begin_forward, the attention call of every
layer, end_forward.  Sequence lengths come from the case alone (`lengths` seeds them), tensor values from
`seed` alone.  A step that appended tokens takes them back with popn, so that a state can be run again; a
sequence-window cache needs none of that: its windows slide.
"""
import math
import random

import torch

from tvm_amd import get_global_func
from tvm_amd import kernels

MHA, MLA, MHA_SLIDING = 0, 1, 3
ROPE_NORMAL, ROPE_INLINE = 1, 2

_create = get_global_func("vm.builtin.paged_attention_kv_cache_create")
_add = get_global_func("vm.builtin.kv_state_add_sequence")
_fork = get_global_func("vm.builtin.kv_state_fork_sequence")
_popn = get_global_func("vm.builtin.kv_state_popn")
_begin = get_global_func("vm.builtin.kv_state_begin_forward")
_end = get_global_func("vm.builtin.kv_state_end_forward")
_set_window = get_global_func("vm.builtin.attention_kv_cache_enable_sliding_window_for_seq")
_commit = get_global_func("vm.builtin.attention_kv_cache_commit_accepted_token_tree_nodes")
_attend = get_global_func("vm.builtin.attention_kv_cache_attention_with_fused_qkv")
_self_attention = get_global_func("vm.builtin.attention_kv_cache_self_attention")
_cross_attention = get_global_func("vm.builtin.attention_kv_cache_cross_attention")
_append_mla = get_global_func("vm.builtin.attention_kv_cache_append_mla_kv")
_merge = get_global_func("vm.builtin.attention_kv_cache_merge_attn_output_inplace")

# MLA layers: width of the latent, of its rotary part, and of the heads that the latent expands to
LATENT, LATENT_ROPE, EXPANDED_QK, EXPANDED_V = 512, 64, 192, 128


def _case(name, **fields):
    case = dict(
        name=name,
        path="cache",        # "cache": MHA layers through the cache object; "mla": MLA layers; "launch": one kernel launch
        storage="float16",
        layers=8, q_heads=32, kv_heads=8, head_dim=128, page=16,
        batch=1,             # sequences of the step
        decoding=1,          # how many of them append one token; the others append new_lo..new_hi
        ctx_lo=0, ctx_hi=0,  # cached tokens of a sequence before the step
        fresh=False,         # the sequences that do not decode are new prompts: nothing cached
        new_lo=1, new_hi=1,
        steps=1,             # consecutive steps of a pass
        shared=0,            # tokens of a prompt that all sequences are forked from
        tree=0,              # draft tokens of a binary tree that every sequence verifies
        windows="none",      # "sequence": attention sinks and a window per sequence; "layer": every other layer has a window
        window=0, sinks=0,
        lengths=1)
    case.update(fields)
    return case


def listed():
    return [
        # One user's conversation, one token: 32 layers whose launches take longer than their 4 MB each.
        _case("decode_one_sequence", layers=32, ctx_lo=1117, ctx_hi=1117),
        # The ordinary load of a server: 64 users at once, contexts from a paragraph to a long document.
        _case("decode_batch", batch=64, decoding=64, ctx_lo=1024, ctx_hi=8192, steps=2),
        # Long documents, many query heads, one layer by its bare launch over a pool that has been in use (page ids permuted).
        _case("decode_long_context", path="launch", layers=1, q_heads=64, batch=8, decoding=8, ctx_lo=32768, ctx_hi=131072,
              lengths=3),
        # 64 conversations behind one system prompt: the prompt is cached once.
        _case("decode_shared_prompt", batch=64, decoding=64, ctx_lo=256, ctx_hi=2048, shared=4096, steps=2, lengths=5),
        # Endless conversations: attention sinks and a sliding window per sequence, RoPE inside the kernels.
        _case("decode_sequence_windows", layers=4, batch=64, decoding=64, ctx_lo=4200, ctx_hi=4700, windows="sequence",
              window=4096, sinks=4, steps=2, lengths=7),
        # Continuous batching on a small model whose layers alternate between a window and full attention:
        # most sequences decode, a few new prompts of odd lengths come in with them.
        _case("mixed_step_layer_windows", head_dim=64, batch=40, decoding=32, fresh=True, ctx_lo=90, ctx_hi=6000, new_lo=17,
              new_hi=777, windows="layer", window=1024, lengths=9),
        # Prompts in chunks, each behind what is cached of it already.
        _case("prefill_chunked", batch=8, decoding=0, ctx_lo=0, ctx_hi=4096, new_lo=128, new_hi=2048, lengths=2),
        # The same in a cache with sequence windows, at the head dim between 64 and 128 that has no tuned kernel there.
        _case("prefill_sequence_windows", layers=2, q_heads=32, kv_heads=32, head_dim=96, batch=6, decoding=0, ctx_lo=2100,
              ctx_hi=2600, new_lo=100, new_hi=1000, windows="sequence", window=2047, sinks=4, lengths=11),
        # Speculative decoding: every sequence verifies a tree of draft tokens and commits a path of it.
        _case("verify_trees", layers=4, batch=64, decoding=0, ctx_lo=1024, ctx_hi=8192, tree=31, lengths=7),
        # A latent cache, one token per sequence.
        _case("mla_decode", path="mla", layers=4, q_heads=128, kv_heads=1, head_dim=LATENT + LATENT_ROPE, page=64, batch=32,
              decoding=32, ctx_lo=2048, ctx_hi=8192, lengths=4),
        # A latent cache, chunks of prompts behind cached prefixes.
        _case("mla_prefill_chunked", path="mla", layers=1, q_heads=128, kv_heads=1, head_dim=LATENT + LATENT_ROPE, page=64,
              batch=4, decoding=0, ctx_lo=1500, ctx_hi=2600, new_lo=600, new_hi=1400, lengths=8),
        # float32 storage, a step of decoding sequences and prompts.
        _case("mixed_step_float32", storage="float32", layers=2, batch=24, decoding=20, fresh=True, ctx_lo=200, ctx_hi=4000,
              new_lo=50, new_hi=700, lengths=13),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    """A case of the ranges of the listed ones: one of their kinds, other heads, batches, lengths and pages."""
    templates = listed()
    limit = 0.8 * max(_seconds(c) for c in templates)
    while True:
        case = dict(rng.choice(templates))
        kind = case.pop("name")
        case["lengths"] = rng.randint(100, 1 << 20)
        case["layers"] = _log_int(rng, max(1, case["layers"] // 2), case["layers"])
        if case["path"] == "mla":
            case["q_heads"] = rng.choice([16, 32, 64, 128])
            case["page"] = rng.choice([16, 32, 64])
        else:
            case["q_heads"], case["kv_heads"] = rng.choice([(32, 8), (32, 8), (64, 8), (32, 4), (28, 4), (8, 8), (16, 2), (32, 1)])
            case["page"] = rng.choice([16, 16, 16, 32, 64])
            if case["path"] == "cache" and case["storage"] == "float16":
                dims = [64, 128, 128, 128, 256]
                if case["windows"] != "layer" and not case["tree"]:
                    dims += [80, 96]
                case["head_dim"] = rng.choice(dims)
            else:
                case["head_dim"] = rng.choice([64, 128])
            if rng.random() < 0.1 and case["path"] == "cache" and not case["tree"]:
                case["page"] = rng.choice([12, 24])
        if kind == "decode_one_sequence":
            case["batch"] = case["decoding"] = _log_int(rng, 1, 16)
            case["ctx_lo"] = case["ctx_hi"] = _log_int(rng, 100, 4000)
            if case["batch"] > 1:
                case["ctx_hi"] = case["ctx_lo"] + _log_int(rng, 1, 4000)
        elif kind == "decode_long_context":
            case["batch"] = case["decoding"] = _log_int(rng, 1, 12)
            case["ctx_lo"] = _log_int(rng, 8192, 65536)
            case["ctx_hi"] = 2 * case["ctx_lo"]
        elif kind in ("decode_batch", "decode_shared_prompt", "decode_sequence_windows", "mla_decode"):
            case["batch"] = case["decoding"] = _log_int(rng, 16, 200)
            if kind == "decode_sequence_windows":
                case["window"] = rng.randint(1000, 4096)
                case["sinks"] = rng.choice([0, 4, 16])
                case["ctx_lo"], case["ctx_hi"] = case["window"] + 30, case["window"] + 700
            else:
                case["ctx_lo"] = _log_int(rng, 64, 2048)
                case["ctx_hi"] = _log_int(rng, case["ctx_lo"], 8192 if kind != "decode_shared_prompt" else 2048)
            if case["shared"]:
                case["shared"] = _log_int(rng, 300, 6000)
        elif kind in ("mixed_step_layer_windows", "mixed_step_float32"):
            case["batch"] = rng.randint(4, 48)
            case["decoding"] = rng.randint(0, case["batch"] - 1)
            case["new_hi"] = min(2000, 7000 // (case["batch"] - case["decoding"]))
            case["new_lo"] = max(5, min(case["new_lo"], case["new_hi"] // 3))
            if case["windows"] == "layer":
                case["window"] = rng.choice([512, 1024, 2048])
        elif kind in ("prefill_chunked", "prefill_sequence_windows", "mla_prefill_chunked"):
            case["batch"] = _log_int(rng, 1, 16)
            case["new_hi"] = _log_int(rng, 60, 7000 // case["batch"])
            case["new_lo"] = _log_int(rng, 20, case["new_hi"])
            if kind == "prefill_sequence_windows":
                case["window"] = rng.randint(1000, 4096)
                case["ctx_lo"], case["ctx_hi"] = case["window"] + 30, case["window"] + 700
            else:
                case["ctx_hi"] = rng.choice([0, _log_int(rng, 100, 6000)]) if kind == "prefill_chunked" else _log_int(rng, 200, 6000)
                case["ctx_lo"] = rng.randint(case["ctx_hi"] // 4, case["ctx_hi"])
        elif kind == "verify_trees":
            case["batch"] = _log_int(rng, 8, 96)
            case["tree"] = rng.randint(7, 63)
            case["ctx_lo"] = _log_int(rng, 200, 4000)
            case["ctx_hi"] = _log_int(rng, case["ctx_lo"], 8192)
        # a state has to fit the card three times over
        cached = case["layers"] * (case["batch"] * (case["ctx_hi"] + 4 * case["page"]) + case["shared"])
        cached *= case["head_dim"] * 2 * (1 if case["path"] == "mla" else 2 * case["kv_heads"]) * (2 if case["storage"] == "float32" else 1)
        if _seconds(case) <= limit and cached < 30e9:
            return case


# ---------------------------------------------------------------------------------------- lengths and work
def _lengths(case):
    """(cached tokens, appended tokens) of every sequence."""
    rng = random.Random(case["lengths"])
    ctx, new = [], []
    for b in range(case["batch"]):
        c, n = rng.randint(case["ctx_lo"], case["ctx_hi"]), rng.randint(case["new_lo"], case["new_hi"])
        decodes = b < case["decoding"]
        ctx.append(0 if case["fresh"] and not decodes else c)
        new.append(case["tree"] if case["tree"] else 1 if decodes else n)
    return ctx, new


def _tree(nodes):
    """Parents of a binary tree in level order, and the path from its root to its last node."""
    parents = [(i - 1) // 2 if i else -1 for i in range(nodes)]
    path, at = [], nodes - 1
    while at >= 0:
        path.append(at)
        at = parents[at]
    return parents, path[::-1]


def _pairs_and_keys(case, windowed):
    """(query, key) pairs of one layer over a pass, keys that have to be read in it, tokens it appends."""
    ctx, new = _lengths(case)
    depth_sum = 0
    if case["tree"]:
        parents, _ = _tree(case["tree"])
        depths = []
        for p in parents:
            depths.append(1 if p < 0 else depths[p] + 1)
        depth_sum = sum(depths)
    pairs = keys = tokens = 0
    for step in range(case["steps"]):
        for c, n in zip(ctx, new):
            cached = c + step * n
            if case["windows"] == "sequence":
                cached = min(cached, case["window"])
            own = depth_sum if case["tree"] else n * (n + 1) // 2
            if windowed:
                w = case["window"]
                seen = sum(min(cached, max(w - r - 1, 0)) for r in range(min(n, w)))
                cached = min(cached, w - 1)
                pairs += seen + own
            else:
                pairs += n * (cached + case["shared"]) + own
            keys += cached + n
            tokens += n
        keys += case["shared"]
    return pairs, keys, tokens


def work(case):
    size = 4 if case["storage"] == "float32" else 2
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    nbytes = flops = 0.0
    if case["path"] == "mla":
        ctx, new = _lengths(case)
        decode = case["decoding"] == case["batch"]
        tokens = sum(new) * case["steps"]
        cached = case["steps"] * sum(c + (1 if decode else 0) for c in ctx)
        self_pairs = 0 if decode else case["steps"] * sum(n * (n + 1) // 2 for n in new)
        cross_pairs = case["steps"] * sum(n * (c + (1 if decode else 0)) for c, n in zip(ctx, new))
        flops = 2.0 * hq * (self_pairs * (EXPANDED_QK + EXPANDED_V) + cross_pairs * (d + LATENT))
        nbytes = 2.0 * (cached * d + 2 * tokens * d)                    # latent rows; the new ones in and out
        if cross_pairs:
            nbytes += tokens * hq * ((d + LATENT) * 2.0 + 4)            # absorbed query, latent output, lse
        if not decode:
            nbytes += tokens * hq * ((2 * EXPANDED_QK + 2 * EXPANDED_V) * 2.0 + 4)
            if cross_pairs:
                nbytes += tokens * hq * EXPANDED_V * 2.0                # the projected output that is merged
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}
    for layer in range(case["layers"]):
        windowed = case["windows"] == "layer" and layer % 2 == 0
        pairs, keys, tokens = _pairs_and_keys(case, windowed)
        flops += 4.0 * hq * d * pairs
        nbytes += size * d * (2.0 * hkv * keys + 2 * hkv * tokens + (2 * hq + 2 * hkv) * tokens)
        if case["path"] == "launch":
            nbytes += 4 * hq * tokens
    return {"bytes": nbytes, "flops": flops}


def _seconds(case):
    """A rough price of a pass, for keeping drawn cases below the largest listed one."""
    w = work(case)
    plain = case["page"] % 16 == 0 and (case["head_dim"] in (64, 128, 256) or case["windows"] == "none")
    rate = 6e13 if case["storage"] == "float32" or not plain else 1e14 if case["windows"] == "sequence" else 8e14
    if case["head_dim"] == 256:
        rate *= 0.6
    return max(w["bytes"] / 6e12, w["flops"] / rate)


def tolerance(case):
    # Measured on small cases of every kind against the same path with its sums and rotations in 64 bits: fp16 outputs
    # are off by 2.7e-4 to 4.6e-4 of their norm (the rounding of the output, the probabilities and rotated rows to fp16),
    # float32 ones by 8.1e-7.  About four times that:
    return {"rel": 3.2e-6} if case["storage"] == "float32" else {"rel": 2e-3}


# ---------------------------------------------------------------------------------------- states
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(*shape, scale=1.0):
        dtype = torch.float32 if case["storage"] == "float32" else torch.float16
        out = torch.empty(shape, dtype=dtype, device="cuda")
        rows = max(1, (1 << 26) // max(1, math.prod(shape[1:])))
        for lo in range(0, shape[0], rows):  # in float32 first, a part at a time
            part = out[lo:lo + rows]
            part.copy_(torch.randn(part.shape, generator=gen, device="cuda").mul_(scale))
        return out

    return {"cache": _prepare_cache, "mla": _prepare_mla, "launch": _prepare_launch}[case["path"]](case, normal)


def _fill_steps(lengths, limit):
    """Chunked-prefill steps that bring the sequences to their lengths, all of them side by side."""
    left = dict(lengths)
    while left:
        share = max(1, limit // len(left))
        ids = list(left)[:limit]
        new = [min(left[s], share) for s in ids]
        yield ids, new
        for s, n in zip(ids, new):
            left[s] -= n
            if not left[s]:
                del left[s]


def _prepare_cache(case, normal):
    ctx, new = _lengths(case)
    batch, layers, page, steps = case["batch"], case["layers"], case["page"], case["steps"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    chunk = max(8192, sum(new))
    if case["windows"] == "sequence":
        capacity = batch * (case["window"] + case["sinks"] + max(max(new), chunk // batch + 1, 700) + 4 * page)
    else:
        capacity = sum(ctx) + case["shared"] + steps * sum(new) + (3 * batch + 4) * page
    kinds = [MHA_SLIDING if case["windows"] == "layer" and layer % 2 == 0 else MHA for layer in range(layers)]
    config = [batch + 1, capacity, chunk, page, int(case["windows"] == "sequence")]
    if case["windows"] == "layer":
        config.append(case["window"])
    sample = normal(1)
    cache = _create(config, [0, layers], hq, hkv, d, d, kinds, False, ROPE_NORMAL, 1.0, 1e4, None, sample)
    cache.set_stream(torch.cuda.current_stream().cuda_stream)
    scale = d ** -0.5

    fill = normal(chunk, hq + 2 * hkv, d)
    sink = torch.empty((chunk, hq, d), dtype=fill.dtype, device="cuda")

    def forward(ids, lengths):
        total = sum(lengths)
        _begin(cache, ids, lengths, None)
        for layer in range(layers):
            _attend(cache, layer, scale, fill[:total], sink[:total])
        _end(cache)
        fill.copy_(torch.roll(fill, 1 + total % 61, 0))  # other rows for the next chunk

    if case["shared"]:
        _add(cache, batch)
        for ids, lengths in _fill_steps({batch: case["shared"]}, chunk):
            forward(ids, lengths)
    for b in range(batch):
        if case["shared"]:
            _fork(cache, batch, b)
        else:
            _add(cache, b)
        if case["windows"] == "sequence":
            _set_window(cache, b, case["window"], case["sinks"])
    for ids, lengths in _fill_steps({b: c for b, c in enumerate(ctx) if c}, chunk):
        forward(ids, lengths)

    total = sum(new)
    qkv = [[normal(total, hq + 2 * hkv, d) for _ in range(layers)] for _ in range(steps)]
    out = torch.zeros((steps, layers, total, hq, d), dtype=fill.dtype, device="cuda")
    tree = leaves = None
    grown = [steps * n for n in new]
    if case["tree"]:
        parents, path = _tree(case["tree"])
        tree, leaves = parents * batch, [case["tree"] - 1] * batch
        grown = [len(path)] * batch
    if case["windows"] == "sequence":
        grown = [0] * batch
    return dict(path="cache", cache=cache, ids=list(range(batch)), new=new, tree=tree, leaves=leaves, grown=grown, qkv=qkv,
                out=out, outs=[[out[s, layer] for layer in range(layers)] for s in range(steps)], scale=scale)


def _prepare_mla(case, normal):
    ctx, new = _lengths(case)
    batch, layers, page, hq, width = case["batch"], case["layers"], case["page"], case["q_heads"], case["head_dim"]
    chunk = max(8192, sum(new))
    capacity = sum(ctx) + sum(new) + (2 * batch + 4) * page
    cache = _create([batch + 1, capacity, chunk, page, 0], [0, layers], hq, 1, width, LATENT, [MLA] * layers, False, 0, 1.0, 1e4,
                    None, normal(1))
    cache.set_stream(torch.cuda.current_stream().cuda_stream)
    fill = normal(chunk, width, scale=0.5)
    for b in range(batch):
        _add(cache, b)
    for ids, lengths in _fill_steps({b: c for b, c in enumerate(ctx) if c}, chunk):
        _begin(cache, ids, lengths, None)
        for layer in range(layers):
            _append_mla(cache, layer, fill[:sum(lengths)])
        _end(cache)
        fill.copy_(torch.roll(fill, 1 + sum(lengths) % 61, 0))
    total = sum(new)
    decode = case["decoding"] == batch
    parts = []
    for _ in range(layers):
        part = dict(row=normal(total, width, scale=0.5), q=normal(total, hq, width, scale=0.5),
                    o=torch.zeros((total, hq, LATENT), dtype=torch.float16, device="cuda"),
                    lse=torch.zeros((total, hq), dtype=torch.float32, device="cuda"))
        if not decode:  # expanded heads of the chunk, and the cross output as its projection leaves it
            part.update(xq=normal(total, hq, EXPANDED_QK, scale=0.5), xk=normal(total, hq, EXPANDED_QK, scale=0.5),
                        xv=normal(total, hq, EXPANDED_V, scale=0.5), projected=normal(total, hq, EXPANDED_V, scale=0.5),
                        xo=torch.zeros((total, hq, EXPANDED_V), dtype=torch.float16, device="cuda"),
                        xlse=torch.zeros((total, hq), dtype=torch.float32, device="cuda"))
        parts.append(part)
    return dict(path="mla", cache=cache, ids=list(range(batch)), new=new, parts=parts, decode=decode, cached=sum(ctx) > 0,
                scale=EXPANDED_QK ** -0.5)


def _prepare_launch(case, normal):
    ctx, new = _lengths(case)
    batch, page, hq, hkv, d = case["batch"], case["page"], case["q_heads"], case["kv_heads"], case["head_dim"]
    pages_of = [(c + 1 + page - 1) // page for c in ctx]
    pool = sum(pages_of) + 64
    ids = list(range(pool))
    random.Random(case["lengths"]).shuffle(ids)
    indptr, slots, at = [0], [], 0
    for c, n in zip(ctx, pages_of):
        slots.append(ids[at + c // page] * page + c % page)
        at += n
        indptr.append(at)

    def i32(values):
        return torch.tensor(values, dtype=torch.int32, device="cuda")

    return dict(path="launch", pages=normal(pool, 2, hkv, page, d), qkv=normal(batch, hq + 2 * hkv, d), indptr=i32(indptr),
                values=i32(ids[:at]), last=i32([c % page + 1 for c in ctx]), positions=i32(ctx), slots=i32(slots),
                out=torch.zeros((batch, hq, d), dtype=torch.float16, device="cuda"),
                lse=torch.zeros((batch, hq), dtype=torch.float32, device="cuda"), scale=d ** -0.5)


# ---------------------------------------------------------------------------------------- one pass
def run(state):
    return {"cache": _run_cache, "mla": _run_mla, "launch": _run_launch}[state["path"]](state)


def _run_cache(state):
    cache, scale = state["cache"], state["scale"]
    for qkv, out in zip(state["qkv"], state["outs"]):
        _begin(cache, state["ids"], state["new"], state["tree"])
        for layer, (x, o) in enumerate(zip(qkv, out)):
            _attend(cache, layer, scale, x, o)
        _end(cache)
    if state["tree"] is not None:
        _commit(cache, state["ids"], state["leaves"])
    for b, n in zip(state["ids"], state["grown"]):
        if n:
            _popn(cache, b, n)
    return state["out"]


def _run_mla(state):
    cache, scale = state["cache"], state["scale"]
    _begin(cache, state["ids"], state["new"], None)
    outputs = []
    for layer, p in enumerate(state["parts"]):
        _append_mla(cache, layer, p["row"])
        if state["decode"]:
            _cross_attention(cache, layer, scale, p["q"], p["o"], p["lse"])
            outputs += [p["o"], p["lse"]]
            continue
        _self_attention(cache, layer, scale, p["xq"], p["xk"], p["xv"], p["xo"], p["xlse"])
        if state["cached"]:
            _cross_attention(cache, layer, scale, p["q"], p["o"], p["lse"])
            _merge(cache, p["xo"], p["xlse"], p["projected"], p["lse"])
            outputs += [p["o"], p["lse"]]
        outputs += [p["xo"], p["xlse"]]
    _end(cache)
    for b, n in zip(state["ids"], state["new"]):
        _popn(cache, b, n)
    return outputs


def _run_launch(state):
    kernels.fused_decode_step(state["qkv"], state["pages"], state["indptr"], state["values"], state["last"], state["positions"],
                              state["slots"], state["out"], state["lse"], 1, 1.0, 1e4, state["scale"])
    return {"out": state["out"], "lse": state["lse"], "pages": state["pages"]}
