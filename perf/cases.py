"""Performance cases of the framework's main path: encoding prompts, paging their
cross-attention K/V, the decode step (attention, decoder layers, whole step) and sampling.

Models are BART / Florence-2 shapes (d_model 768 or 1024, 64-wide heads, vocab 50265 or
51289) with random weights; lengths, beam forks and rows come from the case alone, values
and block placement from the seed.  Decode cases are one HIP-graph replay of the public
entry points over staged step metadata, which is how the engine runs a decode step.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch
import torch.nn.functional as F

from vflorence_amd import decoder_ops, hip_attn
from vflorence_amd.layers import attention, bart
from vflorence_amd.utils.context import set_context
from vflorence_amd.utils.loader import repack_decode_weights

BLOCK = 16
HEAD = 64
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # One image-caption prompt being admitted (an image's tokens plus a short text).
        dict(name="encode_single", kind="encode", dim=768, prompts=1, shortest=590, longest=590,
             dtype="bf16"),
        # A step that admits a batch of documents of mixed lengths, packed back to back.
        dict(name="encode_ragged", kind="encode", dim=1024, prompts=48, shortest=19, longest=1021,
             dtype="bf16"),
        # The encoder K/V of 64 admitted prompts written to their pages, one layer.
        dict(name="page_kv", kind="page", dim=1024, prompts=64, shortest=256, longest=1024,
             dtype="bf16"),
        # A lone interactive request with four beams: the attention of one step.
        dict(name="attend_single", kind="attend", dim=768, layers=6, requests=1, beams=4,
             context=24, shortest=590, longest=590, dtype="bf16"),
        # The throughput batch, 64 requests x 4 beams over 12 layers.
        dict(name="attend_batch", kind="attend", dim=1024, layers=12, requests=64, beams=4,
             context=72, shortest=256, longest=1024, dtype="bf16"),
        # The engine's default data type with beams.
        dict(name="attend_fp32", kind="attend", dim=1024, layers=12, requests=16, beams=4,
             context=72, shortest=256, longest=1024, dtype="fp32"),
        # Greedy decoding under continuous batching: rows at every length, an odd count.
        dict(name="attend_greedy", kind="attend", dim=1024, layers=12, requests=93, beams=1,
             context=1000, shortest=20, longest=700, dtype="fp16"),
        # The decoder stack of a lone four-beam request (a six-layer decoder).
        dict(name="decode_single", kind="decode", dim=1024, layers=6, requests=1, beams=4,
             context=40, shortest=400, longest=400, dtype="bf16", vocab=0),
        # The decoder stack at the largest steps a beam batch makes.
        dict(name="decode_wide", kind="decode", dim=1024, layers=4, requests=128, beams=4,
             context=40, shortest=100, longest=600, dtype="bf16", vocab=0),
        # A whole step of the throughput batch, token ids to logits.
        dict(name="step_batch", kind="decode", dim=1024, layers=12, requests=64, beams=4,
             context=72, shortest=256, longest=1024, dtype="bf16", vocab=50265),
        # Sampling for a lone four-beam request.
        dict(name="sample_single", kind="sample", rows=4, vocab=51289, keep=8, beam=True,
             phase="middle", dtype="bf16"),
        # Sampling for the throughput batch.
        dict(name="sample_batch", kind="sample", rows=256, vocab=50265, keep=8, beam=True,
             phase="middle", dtype="bf16"),
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("encode", "page", "attend", "attend", "decode", "decode", "sample"))
    dim = rng.choice((768, 1024))
    if kind == "sample":
        beam = rng.random() < 0.7
        return dict(kind=kind, rows=_spread(rng, 1, 256), vocab=rng.choice((50265, 51289)),
                    keep=2 * rng.randint(2, 8) if beam else 1, beam=beam,
                    phase=rng.choice(("first", "middle", "middle", "last")),
                    dtype=rng.choice(("bf16", "fp16", "fp32")))
    longest = _spread(rng, 24, 1024)
    shortest = max(1, int(longest * rng.uniform(0.05, 1.0)))
    half = rng.choice(("bf16", "fp16"))
    if kind in ("encode", "page"):
        return dict(kind=kind, dim=dim, prompts=_spread(rng, 1, 48), shortest=shortest,
                    longest=longest, dtype=half)
    beams = rng.choice((1, 2, 3, 4, 5, 8))
    if kind == "attend":
        dtype = rng.choice((half, half, "fp32"))
        rows = 64 if dtype == "fp32" else 256
        return dict(kind=kind, dim=dim, layers=6, requests=_spread(rng, 1, rows // beams),
                    beams=beams, context=_spread(rng, 2, 140 if beams > 1 else 900),
                    shortest=shortest, longest=longest, dtype=dtype)
    return dict(kind=kind, dim=dim, layers=rng.choice((2, 4, 6)),
                requests=_spread(rng, 1, 512 // beams), beams=beams, context=_spread(rng, 2, 140),
                shortest=min(shortest, 600), longest=min(longest, 600), dtype=half, vocab=0)


# ---------------------------------------------------------------------------
# what the case alone decides
# ---------------------------------------------------------------------------
def _lengths(case, count):
    """``count`` prompt lengths evenly over [shortest, longest], in a fixed mixed order."""
    low, high = case["shortest"], case["longest"]
    lens = [low + round((high - low) * (i + 0.5) / count) for i in range(count)]
    random.Random(count).shuffle(lens)
    return lens


def _rows(case):
    """Per row (a request's beams adjacent): context length, and per block position the
    owner (row) of the block it reads.  Beams share a prefix of their first beam's blocks
    up to where they forked from it; the block of the new token is each row's own.  Also the
    rows whose last block was just forked: it still has to be copied from its sibling's."""
    rng = random.Random(1000 * case["requests"] + case["beams"])
    requests, beams, context = case["requests"], case["beams"], case["context"]
    lens, owners, forked = [], [], []
    for r in range(requests):
        length = context if beams > 1 else max(1, round(context * (r + 0.5) / requests))
        blocks = -(-length // BLOCK)
        first = r * beams
        for b in range(beams):
            lens.append(length)
            shared = rng.randint(0, blocks - 1) if b else 0
            owners.append([first] * shared + [first + b] * (blocks - shared))
            if b and (length - 1) % BLOCK and rng.random() < 0.2:
                owners[-1] = [first] * (blocks - 1) + [first + b]
                forked.append((first, first + b))
    if beams == 1:
        order = list(range(requests))
        rng.shuffle(order)
        lens, owners = [lens[i] for i in order], [[i] * len(owners[j]) for i, j in enumerate(order)]
    return lens, owners, forked


def _read_tokens(lens, owners):
    """Tokens of distinct blocks that the rows read."""
    used = {}
    for length, row in zip(lens, owners):
        for i, owner in enumerate(row):
            used[owner, i] = max(used.get((owner, i), 0), min(BLOCK, length - BLOCK * i))
    return sum(used.values())


def _attention_work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    lens, owners, _ = _rows(case)
    enc = _lengths(case, case["requests"])
    rows, dim = len(lens), case["dim"]
    # K and V read once, the queries, new keys and values read, outputs and new K/V written
    cells = 2 * (_read_tokens(lens, owners) + sum(enc)) + 8 * rows
    flops = 4 * (sum(lens) + case["beams"] * sum(enc))
    return dict(bytes=case["layers"] * cells * dim * size, flops=case["layers"] * flops * dim)


def work(case):
    kind = case["kind"]
    if kind == "sample":
        size = 4 if case["dtype"] == "fp32" else 2
        return dict(bytes=case["rows"] * (case["vocab"] * size + 12 * case["keep"]),
                    flops=case["rows"] * case["vocab"] * 4)
    if kind == "encode":
        dim, lens = case["dim"], _lengths(case, case["prompts"])
        return dict(bytes=2 * (2 * sum(lens) * dim + 4 * dim * dim),
                    flops=8 * sum(lens) * dim * dim + 4 * dim * sum(n * n for n in lens))
    if kind == "page":
        return dict(bytes=2 * 4 * sum(_lengths(case, case["prompts"])) * case["dim"], flops=0)
    w = _attention_work(case)
    if kind == "decode":
        rows, dim = case["requests"] * case["beams"], case["dim"]
        weights = case["layers"] * 14 * dim * dim + case["vocab"] * dim
        w["bytes"] += 2 * (weights + rows * (dim + case["vocab"]))
        w["flops"] += 2 * rows * weights
    return w


def tolerance(case):
    """About four times the distance from 64 bits that the kernels show over the ranges."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind == "page":  # K/V rows are moved, not computed
        return "exact"
    if kind == "sample":  # 32-bit scores; equal logits are ordered by token id
        return {"rel": 2e-6, "max": 2e-5}
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 5e-4}
    if kind == "decode":  # a rounding in one layer travels through those that follow
        return {"rel": 0.03 if bf16 else 5e-3, "max": 0.3 if bf16 else 0.05}
    if kind == "encode":  # 16-bit projections around the attention
        return {"rel": 0.02 if bf16 else 2.5e-3, "max": 0.2 if bf16 else 0.025}
    return {"rel": 7e-3 if bf16 else 9e-4, "max": 0.07 if bf16 else 9e-3}


# ---------------------------------------------------------------------------
# what the seed decides
# ---------------------------------------------------------------------------
def _normal(gen, shape, dtype, std):
    """N(0, std^2) of ``shape`` in ``dtype``, drawn in 32 bits."""
    return torch.randn(shape, generator=gen, device="cuda").mul_(std).to(dtype)


def _gens(seed):
    return (torch.Generator(device="cuda").manual_seed(seed),
            torch.Generator().manual_seed(seed))


class _Layer:
    """A decoder layer's pools, as the attention ops and ``stage_cross`` read them."""

    def __init__(self, heads):
        self.self_attn = SimpleNamespace(num_heads=heads, head_dim=HEAD)
        self.encoder_attn = SimpleNamespace(num_heads=heads, head_dim=HEAD)


def _stage(case, layers, gen, host_gen):
    """Pools for ``layers`` and the step's metadata on the device: the Context's fields."""
    dtype, heads = DTYPES[case["dtype"]], case["dim"] // HEAD
    lens, owners, forked = _rows(case)
    rows, beams = len(lens), case["beams"]
    width = max(map(len, owners))
    ids, tables = {}, []
    count = sum(o == r for r, row in enumerate(owners) for o in row)
    place = torch.randperm(count, generator=host_gen).tolist()
    for r, row in enumerate(owners):
        for i, owner in enumerate(row):
            if owner == r:
                ids[r, i] = place[len(ids)]
        tables.append([ids[o, i] for i, o in enumerate(row)] + [0] * (width - len(row)))
    slots = [t[(n - 1) // BLOCK] * BLOCK + (n - 1) % BLOCK for t, n in zip(tables, lens)]
    last = [(n - 1) // BLOCK for n in lens]
    pairs = [(tables[a][last[a]], tables[b][last[b]]) for a, b in forked]
    # encoder pages, a contiguous run per request
    enc = _lengths(case, case["requests"])
    pages, at = [], 0
    for n in enc:
        p = -(-n // BLOCK)
        pages.append(torch.arange(at, at + p, dtype=torch.int32))
        at += p
    for layer in layers:
        for attn, blocks in ((layer.self_attn, count), (layer.encoder_attn, at)):
            shape = (blocks, heads, BLOCK, HEAD)
            attn.k_cache, attn.v_cache = (_normal(gen, shape, dtype, 1.0) for _ in range(2))
    host_tables = torch.tensor(tables, dtype=torch.int32)
    host_lens = torch.tensor(lens, dtype=torch.int32)
    common = dict(num_reqs=rows, num_heads=heads, num_kv_heads=heads, head_dim=HEAD, dtype=dtype,
                  block_size=BLOCK, fuse_kv_write=True)
    copies = None
    if beams > 1:
        starts = torch.arange(0, rows + 1, beams, dtype=torch.int32)
        plan = hip_attn.build_group_plan(host_tables, host_lens, starts, num_blocks=count)
        folded = hip_attn.plan_copies_supported(dtype, HEAD, BLOCK) and hip_attn.fold_plan_copies(
            plan, [a for a, _ in pairs], [b for _, b in pairs], num_blocks=count)
        if pairs and not folded:
            copies = tuple(torch.tensor(p, device="cuda") for p in zip(*pairs))
        meta = hip_attn.get_scheduler_metadata(
            group_start=starts.cuda(), max_group_size=hip_attn.MAX_GROUP_SIZE, own_tables=True,
            group_plan=plan.to("cuda"), **common)
    else:
        order = torch.tensor(hip_attn.longest_first(lens), dtype=torch.int32, device="cuda")
        meta = hip_attn.get_scheduler_metadata(group_order=order, **common)
    buffers = attention.CrossStagingBuffers(rows, max(map(len, pages)), "cuda")
    staged = attention.stage_cross(layers, [p for p in pages for _ in range(beams)],
                                   [n for n in enc for _ in range(beams)], BLOCK, "gfx950",
                                   buffers=buffers, slots=case["requests"])
    context = dict(context_lens=host_lens.cuda(), block_tables=host_tables.cuda(),
                   slot_mapping=torch.tensor(slots, device="cuda"),
                   query_start_loc=torch.arange(rows + 1, dtype=torch.int32, device="cuda"),
                   self_metadata=meta, isa="gfx950", cross_staged=staged)
    caches = [c for layer in layers for c in (layer.self_attn.k_cache, layer.self_attn.v_cache)]
    copier = hip_attn.BlockCopier(caches)
    return SimpleNamespace(context=context, copies=copies, copier=copier, caches=caches,
                           buffers=buffers, lens=lens, tables=tables, slots=slots, pairs=pairs,
                           enc=enc, pages=pages)


def _capture(stage, step):
    """The step's graph, captured as the engine does: once eagerly, then recorded."""
    def call():
        set_context(**stage.context)
        try:
            if stage.copies is not None:
                stage.copier(*stage.copies)
            return step()
        finally:
            set_context()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = call()
    return graph, outputs


def _attend_state(case, seed):
    gen, host_gen = _gens(seed)
    dtype, dim = DTYPES[case["dtype"]], case["dim"]
    heads = dim // HEAD
    layers = [_Layer(heads) for _ in range(case["layers"])]
    stage = _stage(case, layers, gen, host_gen)
    rows = len(stage.lens)
    qkv = [_normal(gen, (rows, 3 * dim), dtype, 1.0) for _ in layers]
    queries = [_normal(gen, (rows, heads, HEAD), dtype, 1.0) for _ in layers]
    return SimpleNamespace(stage=stage, layers=layers, qkv=qkv, queries=queries)


def _attend_step(s):
    out = []
    for i, (layer, qkv, query) in enumerate(zip(s.layers, s.qkv, s.queries)):
        q, k, v = (t.view(query.shape) for t in qkv.chunk(3, dim=-1))
        a = layer.self_attn
        out.append((attention.decoder_self_attention(q, k, v, a.k_cache, a.v_cache, HEAD**-0.5),
                    attention.decoder_cross_attention(query, i, HEAD**-0.5),
                    a.k_cache, a.v_cache))
    return out


def _random_weights(module, gen):
    for name, p in module.named_parameters():
        if "norm" in name and name.endswith("weight"):
            p.copy_(1 + 0.1 * torch.randn(p.shape, generator=gen, device="cuda"))
        else:
            std = 0.02 if p.dim() == 1 or "embed" in name else p.shape[-1]**-0.5
            p.copy_(_normal(gen, p.shape, p.dtype, std))


def _decode_state(case, seed):
    from transformers import BartConfig

    gen, host_gen = _gens(seed)
    dtype, dim = DTYPES[case["dtype"]], case["dim"]
    heads = dim // HEAD
    vocab = case["vocab"] or 1024
    config = BartConfig(vocab_size=vocab, d_model=dim, encoder_layers=0,
                        decoder_layers=case["layers"], encoder_attention_heads=heads,
                        decoder_attention_heads=heads, encoder_ffn_dim=4 * dim,
                        decoder_ffn_dim=4 * dim)
    with torch.device("meta"):
        model = bart.BartForConditionalGeneration(config).to(dtype)
    model = model.to_empty(device="cuda").eval()
    _random_weights(model.model.decoder, gen)
    model.model.decoder.embed_tokens.weight = model.lm_head.weight
    model.lm_head.weight.copy_(_normal(gen, model.lm_head.weight.shape, dtype, 0.05))
    model.final_logits_bias.zero_()
    repack_decode_weights(model)
    layers = list(model.decoder_layers)
    stage = _stage(case, layers, gen, host_gen)
    rows = len(stage.lens)
    ids = torch.randint(3, vocab, (rows,), generator=gen, device="cuda")
    positions = torch.tensor(stage.lens, device="cuda") - 1
    return SimpleNamespace(stage=stage, model=model, ids=ids, positions=positions)


def _decode_step(case, s):
    if case["vocab"]:
        return [s.model(s.ids, s.positions)] + s.stage.caches
    return [s.model.model.decoder(s.ids, s.positions)] + s.stage.caches


def _encode_state(case, seed):
    gen, _ = _gens(seed)
    dtype, dim = DTYPES[case["dtype"]], case["dim"]
    with torch.device("meta"):
        layer = bart.BartEncoderSelfAttention(dim, dim // HEAD).to(dtype)
    layer = layer.to_empty(device="cuda").eval()
    _random_weights(layer, gen)
    with torch.no_grad():  # attention of a trained model is peaked: scores of a few units
        layer.qkv_proj.weight[:2 * dim].mul_(1.5)
    counts = {}
    for n in _lengths(case, case["prompts"]):
        counts[n] = counts.get(n, 0) + 1
    segments, at = [], 0
    for n, c in counts.items():
        segments.append((at, c, n))
        at += c * n
    x = _normal(gen, (at, dim), dtype, 1.0)
    return SimpleNamespace(layer=layer, x=x, segments=segments)


def _page_state(case, seed):
    gen, host_gen = _gens(seed)
    dtype, dim = DTYPES[case["dtype"]], case["dim"]
    heads, lens = dim // HEAD, _lengths(case, case["prompts"])
    blocks = sum(-(-n // BLOCK) for n in lens)
    place = torch.randperm(blocks, generator=host_gen)
    slots, at = [], 0
    for n in lens:
        p = -(-n // BLOCK)
        t = torch.arange(n)
        slots.append(place[at:at + p][t // BLOCK] * BLOCK + t % BLOCK)
        at += p
    tokens = sum(lens)
    kv = _normal(gen, (tokens, 2 * dim), dtype, 1.0)
    key, value = (t.view(tokens, heads, HEAD) for t in kv.chunk(2, dim=-1))
    k_cache, v_cache = (torch.zeros(blocks, heads, BLOCK, HEAD, dtype=dtype, device="cuda")
                        for _ in range(2))
    return SimpleNamespace(key=key, value=value, k_cache=k_cache, v_cache=v_cache,
                           slots=torch.cat(slots).cuda())


def _sample_state(case, seed):
    gen, _ = _gens(seed)
    rows, vocab = case["rows"], case["vocab"]
    logits = _normal(gen, (rows, vocab), DTYPES[case["dtype"]], 2.5)
    low, high = {"first": (1, 2), "middle": (10, 130), "last": (140, 142)}[case["phase"]]
    lengths = torch.randint(low, high, (rows,), generator=gen, device="cuda")
    rules = decoder_ops.TopkRules(eos=[2], suppress=[], begin_suppress=[], forced_bos=[0],
                                  forced_eos=[2], min_length=56, max_length=142, begin_index=2,
                                  device="cuda")
    return SimpleNamespace(logits=logits, lengths=lengths, rules=rules)


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "encode":
        s = _encode_state(case, seed)
    elif kind == "page":
        s = _page_state(case, seed)
    elif kind == "sample":
        s = _sample_state(case, seed)
    else:
        with torch.inference_mode():
            if kind == "attend":
                s = _attend_state(case, seed)
                s.graph, s.outputs = _capture(s.stage, lambda: _attend_step(s))
            else:
                s = _decode_state(case, seed)
                s.graph, s.outputs = _capture(s.stage, lambda: _decode_step(case, s))
    s.case = case
    return s


@torch.inference_mode()
def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "encode":
        return state.layer(state.x, state.segments)
    if kind == "page":
        attention.reshape_and_cache(state.key, state.value, state.k_cache, state.v_cache,
                                    state.slots)
        return [state.k_cache, state.v_cache]
    if kind == "sample":
        return decoder_ops.logprob_topk(state.logits, case["keep"], log_softmax=case["beam"],
                                        lengths=state.lengths, rules=state.rules)
    state.graph.replay()
    return state.outputs


# ---------------------------------------------------------------------------
# the same in plain torch and 64 bits
# ---------------------------------------------------------------------------
def _logical(pool, value):
    """A pool as [blocks, heads, tokens, dims]: 16-bit V pools interleave four tokens."""
    if not value or pool.dtype == torch.float32:
        return pool
    n, h, b, d = pool.shape
    return pool.view(n, h, b // 4, d, 4).transpose(3, 4).reshape(n, h, b, d)


def _softmax_attention(q, k, v):
    """q [rows, heads, D] over k, v [heads, tokens, D]."""
    p = torch.softmax(torch.einsum("rhd,htd->hrt", q, k) * HEAD**-0.5, -1)
    return torch.einsum("hrt,htd->rhd", p, v)


def _exact_self(stage, layer, q, k, v):
    kc = _logical(layer.self_attn.k_cache, False).clone()
    vc = _logical(layer.self_attn.v_cache, True).clone()
    if stage.pairs:
        src, dst = (torch.tensor(p, device="cuda") for p in zip(*stage.pairs))
        kc[dst], vc[dst] = kc[src], vc[src]
    out = []
    for r, (n, table, slot) in enumerate(zip(stage.lens, stage.tables, stage.slots)):
        blocks = torch.tensor(table[:-(-n // BLOCK)], device="cuda")
        row = [c[blocks].double().transpose(0, 1).flatten(1, 2)[:, :n].clone() for c in (kc, vc)]
        row[0][:, n - 1], row[1][:, n - 1] = k[r], v[r]
        out.append(_softmax_attention(q[r:r + 1], *row))
    return torch.cat(out)


def _exact_cross(stage, layer, q):
    kc, vc = _logical(layer.encoder_attn.k_cache, False), _logical(layer.encoder_attn.v_cache, True)
    beams = len(stage.lens) // len(stage.enc)
    out = []
    for r, (n, pages) in enumerate(zip(stage.enc, stage.pages)):
        blocks = pages.long().cuda()
        row = (c[blocks].double().transpose(0, 1).flatten(1, 2)[:, :n] for c in (kc, vc))
        out.append(_softmax_attention(q[r * beams:(r + 1) * beams], *row))
    return torch.cat(out)


def _linear(x, m):
    return F.linear(x, m.weight.double(), None if m.bias is None else m.bias.double())


def _norm(x, m):
    return F.layer_norm(x, x.shape[-1:], m.weight.double(), m.bias.double(), m.eps)


def _exact_decode(case, s):
    decoder, stage = s.model.model.decoder, s.stage
    heads = case["dim"] // HEAD
    rows = len(stage.lens)
    h = _norm(decoder.embed_tokens.weight[s.ids].double() +
              decoder.embed_positions.weight[s.positions + 2].double(),
              decoder.layernorm_embedding)
    for layer in decoder.layers:
        a, c = layer.self_attn, layer.encoder_attn
        q, k, v = (t.view(rows, heads, HEAD) for t in _linear(h, a.qkv_proj).chunk(3, -1))
        h = _norm(h + _linear(_exact_self(stage, layer, q, k, v).flatten(1), a.out_proj),
                  layer.self_attn_layer_norm)
        q = _linear(h, c.q_proj).view(rows, heads, HEAD)
        h = _norm(h + _linear(_exact_cross(stage, layer, q).flatten(1), c.out_proj),
                  layer.encoder_attn_layer_norm)
        h = _norm(h + _linear(F.gelu(_linear(h, layer.fc1)), layer.fc2), layer.final_layer_norm)
    if case["vocab"]:
        h = F.linear(h, s.model.lm_head.weight.double(), s.model.final_logits_bias[0].double())
    return [h] + [None] * len(stage.caches)


def _exact_encode(s):
    heads = s.layer.num_heads
    qkv = _linear(s.x.double(), s.layer.qkv_proj)
    out = torch.empty_like(s.x, dtype=torch.float64)
    for start, count, n in s.segments:
        for at in range(start, start + count * n, n):
            q, k, v = (t.view(n, heads, HEAD) for t in qkv[at:at + n].chunk(3, -1))
            out[at:at + n] = _softmax_attention(q, k.transpose(0, 1), v.transpose(0, 1)).flatten(1)
    return _linear(out, s.layer.out_proj)


def _exact_sample(case, s):
    scores = s.logits.double()
    if case["beam"]:
        scores = torch.log_softmax(scores, -1)
    forced_first, forced_last = s.lengths == 1, s.lengths == 141
    scores[:, 2].masked_fill_(s.lengths < 56, -math.inf)
    scores[forced_first | forced_last] = -math.inf
    scores[:, 0].masked_fill_(forced_first, 0.0)
    scores[:, 2].masked_fill_(forced_last, 0.0)
    best, ids = torch.sort(scores, dim=-1, descending=True, stable=True)
    return [best[:, :case["keep"]], ids[:, :case["keep"]]]


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return _exact_encode(_encode_state(case, seed))
    if kind == "page":
        return None
    if kind == "sample":
        return _exact_sample(case, _sample_state(case, seed))
    with torch.inference_mode():
        if kind == "decode":
            return _exact_decode(case, _decode_state(case, seed))
        s = _attend_state(case, seed)
        out = []
        for layer, qkv, query in zip(s.layers, s.qkv, s.queries):
            q, k, v = (t.double().view(query.shape) for t in qkv.chunk(3, dim=-1))
            out.append((_exact_self(s.stage, layer, q, k, v),
                        _exact_cross(s.stage, layer, query.double()), None, None))
        return out
