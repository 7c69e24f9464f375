"""The work that users of this package give it, as cases that can be timed.

A serving engine decodes batches from one sequence to 256 with contexts from a
few tokens to 32k, prefills prompts (fresh, or in chunks behind a cached
prefix), turns projection currents into packed spikes and samples tokens.  Each
case is one call of that kind through the public entry points:

  attn      paged_spike_attn_decode, one layer, eager
  layers    the decode attention of all layers of a step in one hipGraph
  step      paged_attention_fused: decode tokens and prefill chunks, one layer
  lif_pack  lif_pack_write_sites: q/k/v currents to packed words and cache slots
  lif       lif_multistep: dense spikes of the MLP gate (and the membrane)
  sample    sample_tokens over a batch of logits
  decode    a decoder layer's step for a batch in one hipGraph, with or without the head
  prefill   a decoder layer over prompts or chunks, and the last tokens' logits

The decoder has one layer here: a deep stack of spiking layers turns any change
of rounding into other spikes, and two correct runs of 24 layers differ by a
quarter in their logits (2-norm), of one layer by less than 1 %.

Shapes are those of bench.py and the tests (14 query and 2 kv heads, T = 4,
16-token blocks, hidden 896, intermediate 4864, vocabulary 151,936) and generic
ones around them.
"""
from __future__ import annotations

import math

import torch

from spikeinfer_amd.attention import AttentionMetadata, paged_attention_fused
from spikeinfer_amd.kernels import lif_multistep, lif_pack_write_sites, paged_spike_attn_decode
from spikeinfer_amd.model import SpikingDecoder, SpikingQwenConfig
from spikeinfer_amd.sampler import sample_tokens, sample_workspace_bytes
from spikeinfer_amd.spike_cache import PagedSpikeCache

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BS = 16  # tokens per cache block
HIDDEN, INTER, VOCAB, THETA, EPS = 896, 4864, 151936, 1000000.0, 1e-6


# -- the cases -----------------------------------------------------------------
def _attn(n, lo, hi, dtype="f32", T=4, hq=14, hkv=2, D=64, density=0.2):
    return dict(kind="attn", n=n, lo=lo, hi=hi, dtype=dtype, T=T, hq=hq, hkv=hkv, D=D, density=density)


def _step(n_dec, hi, chunks, chunk, ctx, dtype="bf16", D=64, hq=14, hkv=2):
    return dict(kind="step", n_dec=n_dec, hi=hi, chunks=chunks, chunk=chunk, ctx=ctx, dtype=dtype, T=4,
                hq=hq, hkv=hkv, D=D)


def _sample(rows, dtype, top_k, top_p, min_p, rep, scale, temperature=0.8):
    return dict(kind="sample", rows=rows, vocab=VOCAB, dtype=dtype, top_k=top_k, top_p=top_p, min_p=min_p,
                rep=rep, scale=scale, temperature=temperature)


def listed():
    return [
        # one user, a short chat, one layer: latency only
        dict(_attn(1, 128, 128), name="attn_single_128"),
        # a busy chat server's step, all 24 layers as the runner replays them
        dict(kind="layers", n=64, lo=128, hi=192, layers=24, dtype="bf16", T=4, hq=14, hkv=2, D=64,
             density=0.2, name="attn_chat_24_layers"),
        # long documents at the largest batch: bound by reading the cache
        dict(_attn(256, 4096, 32768), name="attn_long_256"),
        # a model with 128-channel heads, mid-length contexts, 16-bit output
        dict(_attn(48, 1000, 8000, "bf16", D=128, hq=16, hkv=4), name="attn_head_dim_128"),
        # continuous batching: decodes beside two chunks of a chunked prefill
        dict(_step(32, 2048, 2, 509, 1024), name="step_decodes_and_chunks"),
        # a long fresh prompt of one user, one layer's attention
        dict(_step(0, 0, 1, 4096, 0), name="step_long_prompt"),
        # q/k/v spikes of 4,096 prompt tokens into the paged cache
        dict(kind="lif_pack", n=4096, dtype="bf16", T=4, hq=14, hkv=2, D=64, name="lif_pack_4096"),
        # the MLP gate's spikes, ragged token count, membrane kept
        dict(kind="lif", n=2047, C=INTER, dtype="bf16", T=4, membrane=True, name="lif_gate_2047"),
        # a full batch's next tokens: top-k 50, top-p 0.9, repetition penalty
        dict(_sample(64, "bf16", 50, 0.9, 0.0, 1.1, 1.0), name="sample_64"),
        # the captured decode step of a full batch, to its logits, and a layer for a few users
        dict(kind="decode", n=64, lo=128, hi=192, layers=1, head=True, name="decode_step_64"),
        dict(kind="decode", n=5, lo=300, hi=900, layers=1, head=False, name="decode_layer_5"),
        # prompts of eight users in one forward
        dict(kind="prefill", prompts=8, plen=251, ctx=0, layers=1, name="prefill_8_prompts"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn"] * 4 + ["layers"] + ["step"] * 3 + ["lif_pack", "lif", "sample", "decode"] +
                      ["prefill"] * 2)
    if kind in ("attn", "layers"):
        hq, hkv, D = rng.choice([(14, 2, 64)] * 4 + [(8, 1, 64), (16, 4, 128), (16, 2, 128)])
        hi = _log(rng, 64, 32768)
        # at most the tokens (and the words) of the largest listed batch
        n = min(_log(rng, 1, 256), max(1, 4_000_000 // (hi * hkv * D // 128)))
        c = dict(_attn(n, max(1, hi // rng.choice([1, 2, 8])), hi, rng.choice(["f32", "bf16", "f16"]),
                       T=rng.choice([4, 4, 4, 2, 8]) if hi < 16384 else 4, hq=hq, hkv=hkv, D=D,
                       density=rng.choice([0.05, 0.2, 0.5])), kind=kind)
        if kind == "layers":
            c["layers"] = rng.randint(4, 24)
            c["hi"] = min(c["hi"], 2048)
            c["lo"] = min(c["lo"], c["hi"])
            c["n"] = min(c["n"], 64)
        return c
    if kind == "step":
        chunks = rng.choice([1, 1, 2, 4])
        chunk = _log(rng, 17, 4096 // chunks)
        ctx = rng.choice([0, _log(rng, 16, 4096)])
        D, hq, hkv = rng.choice([(64, 14, 2)] * 3 + [(64, 8, 8), (128, 8, 2)])
        return _step(rng.choice([0, _log(rng, 1, 64)]), _log(rng, 64, 4096), chunks, chunk, ctx,
                     rng.choice(["bf16", "bf16", "f16"]), D, hq, hkv)
    if kind == "lif_pack":
        hq, hkv, D = rng.choice([(14, 2, 64)] * 3 + [(16, 4, 128), (8, 8, 32)])
        return dict(kind=kind, n=_log(rng, 1, 8192), dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                    T=rng.choice([4, 4, 2, 8]), hq=hq, hkv=hkv, D=D)
    if kind == "lif":
        return dict(kind=kind, n=_log(rng, 1, 4096), C=rng.choice([INTER, INTER, 8960, 1728, 777]),
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), T=rng.choice([4, 4, 2, 8]),
                    membrane=rng.random() < 0.3)
    if kind == "sample":
        k, tp, mp = rng.choice([(50, 0.9, 0.0), (20, 1.0, 0.0), (-1, 0.9, 0.0), (-1, 1.0, 0.05), (1, 1.0, 0.0)])
        return _sample(_log(rng, 1, 128), rng.choice(["bf16", "bf16", "f32"]), k, tp, mp,
                       rng.choice([1.0, 1.1]), rng.choice([1.0, 6.0]), round(rng.uniform(0.5, 1.2), 3))
    if kind == "decode":
        hi = _log(rng, 32, 2048)
        return dict(kind=kind, n=_log(rng, 1, 64), lo=max(1, hi // 2), hi=hi, layers=1,
                    head=rng.random() < 0.5)
    prompts, ctx = rng.choice([1, 1, 2, 4, 7]), rng.choice([0, 0, _log(rng, 16, 2048)])
    return dict(kind=kind, prompts=prompts, plen=_log(rng, 20, (1000 if ctx else 2000) // prompts), ctx=ctx,
                layers=1)


# -- inputs --------------------------------------------------------------------
def _gens(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device=DEV).manual_seed(seed + 1)


def _words(shape, density, g):
    """Packed spike words whose bits are set with probability ~density (in 1/256)."""
    d = max(1, round(density * 256))
    w = torch.zeros(shape, dtype=torch.int32, device=DEV)
    for b in range(8):
        r = torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=DEV, generator=g)
        w = (w | r) if (d >> b) & 1 else (w & r)
    return w


def _tables(lens, max_blocks, g, pool=0):
    """Shuffled physical blocks for sequences of `lens` tokens out of a pool of at
    least `pool` -> ([n, max_blocks] host table padded with the last block, number
    of blocks)."""
    need = [-(-int(x) // BS) for x in lens]
    total = max(pool, sum(need)) + 1
    perm = torch.randperm(total - 1, generator=g).int()
    tables = torch.full((len(need), max_blocks), total - 1, dtype=torch.int32)
    at = 0
    for i, nb in enumerate(need):
        tables[i, :nb] = perm[at:at + nb]
        at += nb
    return tables, total


def _lens(n, lo, hi, g):
    lens = torch.randint(lo, hi + 1, (n,), generator=g, dtype=torch.int32)
    if n > 1:
        lens[0] = hi  # so that the table's width is the longest sequence's
    return lens


def _attn_inputs(c, seed, layers=1):
    gc, g = _gens(seed)
    lens = _lens(c["n"], c["lo"], c["hi"], gc)
    tables, blocks = _tables(lens, -(-c["hi"] // BS), gc)
    W = c["D"] // 32
    kv = (c["T"], c["hkv"], blocks * BS, W)
    return dict(lens=lens.to(DEV), tables=tables.to(DEV),
                q=[_words((c["T"], c["n"], c["hq"], W), c["density"], g) for _ in range(layers)],
                k=[_words(kv, c["density"], g) for _ in range(layers)],
                v=[_words(kv, c["density"], g) for _ in range(layers)])


def _chunk_lens(c):
    """Chunk lengths and cached prefixes of a step: ragged after the first."""
    return [(max(1, c["chunk"] - 37 * i), max(0, c["ctx"] - 101 * i) if c["ctx"] else 0)
            for i in range(c["chunks"])]


def _batch(n_dec, lo, hi, chunks, gc):
    """Metadata of decodes with `lo`..`hi` tokens and chunks (length, cached
    prefix): positions, slots, the block tables of both and the cache's blocks."""
    dec = _lens(n_dec, lo, hi, gc) if n_dec else torch.empty(0, dtype=torch.int32)
    every = dec.tolist() + [q + p for q, p in chunks]
    width = max(-(-x // BS) for x in every)
    pool = n_dec * -(-hi // BS) + sum(-(-(q + p) // BS) for q, p in chunks)
    tables, blocks = _tables(every, width, gc, pool)
    pos, seq = [], []
    for i, x in enumerate(dec.tolist()):
        pos.append(torch.tensor([x - 1]))
        seq.append(torch.tensor([i]))
    for i, (q, p) in enumerate(chunks):
        pos.append(torch.arange(p, p + q))
        seq.append(torch.full((q,), n_dec + i))
    pos, seq = torch.cat(pos), torch.cat(seq)
    slots = tables[seq, pos // BS].long() * BS + pos % BS
    starts, at = [], n_dec
    for q, _ in chunks:
        starts.append(at)
        at += q
    meta = AttentionMetadata(
        slot_mapping=slots.to(DEV), block_size=BS, num_decode_tokens=n_dec,
        block_tables=tables[:n_dec].to(DEV) if n_dec else None, seq_lens=dec.to(DEV) if n_dec else None,
        prefill_query_starts=starts, prefill_query_lens=[q for q, _ in chunks],
        prefill_context_lens=[p for _, p in chunks],
        prefill_block_tables=[t.to(DEV) for t in tables[n_dec:]])
    return meta, pos.to(DEV), blocks


def _lif_params(g, n):
    """Decay and threshold per channel, as trained values spread around 0.9 and 1."""
    return (0.9 + 0.05 * torch.randn(n, device=DEV, generator=g),
            1.0 + 0.1 * torch.rand(n, device=DEV, generator=g))


def _step_inputs(c, seed):
    gc, g = _gens(seed)
    meta, _, blocks = _batch(c["n_dec"], max(1, c["hi"] // 4), c["hi"], _chunk_lens(c), gc)
    n, dt, T, D = meta.slot_mapping.numel(), DTYPES[c["dtype"]], c["T"], c["D"]
    cur = lambda h: torch.randn((T, n, h, D), device=DEV, generator=g).to(dt)
    kv = (T, c["hkv"], blocks * BS, D // 32)
    return dict(q=cur(c["hq"]), k=cur(c["hkv"]), v=cur(c["hkv"]), meta=meta,
                lif=[_lif_params(g, D) for _ in range(3)], kc=_words(kv, 0.2, g), vc=_words(kv, 0.2, g))


def _weights(layers, g):
    """A state dict of the reference's parameter names: projections N(0, 0.02) as
    bench.py, embeddings N(0, 1) (torch's default for a table), so that a layer
    adds to a residual stream larger than its update, as in a trained model."""
    hq, hkv, D = 14, 2, 64

    def w(*shape, std=0.02):
        return torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(0.0, std, generator=g)

    def near(v, n):
        return (v + 0.05 * torch.randn(n, device=DEV, generator=g)).bfloat16()

    sd = {"model.embed_tokens.weight": w(VOCAB, HIDDEN, std=1.0), "model.norm.weight": near(1.0, HIDDEN)}
    for i in range(layers):
        p = f"model.layers.{i}."
        a, m = p + "self_attn.", p + "mlp."
        sd[p + "input_layernorm.weight"] = near(1.0, HIDDEN)
        sd[p + "post_attention_layernorm.weight"] = near(1.0, HIDDEN)
        for s, h in (("q", hq), ("k", hkv), ("v", hkv)):
            sd[a + f"{s}_proj.weight"], sd[a + f"{s}_proj.bias"] = w(h * D, HIDDEN), w(h * D)
            sd[a + f"lif_{s}.lif.beta"], sd[a + f"lif_{s}.lif.threshold"] = near(0.9, D), near(1.0, D)
        sd[a + "o_proj.weight"] = w(HIDDEN, hq * D)
        sd[m + "gate_proj.weight"], sd[m + "up_proj.weight"] = w(INTER, HIDDEN), w(INTER, HIDDEN)
        sd[m + "down_proj.weight"] = w(HIDDEN, INTER)
        sd[m + "lif_gate.lif.beta"], sd[m + "lif_gate.lif.threshold"] = near(0.9, INTER), near(1.0, INTER)
    return sd


def _model_inputs(c, seed):
    gc, g = _gens(seed)
    if c["kind"] == "decode":
        meta, pos, blocks = _batch(c["n"], c["lo"], c["hi"], [], gc)
    else:
        meta, pos, blocks = _batch(0, 0, 0, [(c["plen"], c["ctx"])] * c["prompts"], gc)
    kv = (4, 2, blocks * BS, 2)
    caches = [(_words(kv, 0.2, g), _words(kv, 0.2, g)) for _ in range(c["layers"])]
    ids = torch.randint(0, VOCAB, (pos.numel(),), device=DEV, generator=g)
    return dict(sd=_weights(c["layers"], g), meta=meta, pos=pos, blocks=blocks, caches=caches, ids=ids,
                last=torch.tensor([s + q - 1 for s, q in zip(meta.prefill_query_starts,
                                                             meta.prefill_query_lens)], device=DEV))


def _captured(step):
    """A user's program captures its step once and replays it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


@torch.no_grad()
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("attn", "layers"):
        s = _attn_inputs(c, seed, c.get("layers", 1))
        if kind == "layers":
            out = torch.empty((c["layers"], c["T"], c["n"], c["hq"], c["D"]), dtype=DTYPES[c["dtype"]], device=DEV)

            def step():
                for i in range(c["layers"]):
                    paged_spike_attn_decode(s["q"][i], s["k"][i], s["v"][i], s["tables"], s["lens"], c["D"], BS,
                                            c["hq"], c["hkv"], out=out[i])
                return out

            s["graph"], s["out"] = _captured(step)
    elif kind == "step":
        s = _step_inputs(c, seed)
    elif kind == "lif_pack":
        s = _lif_pack_inputs(c, seed)
    elif kind == "lif":
        _, g = _gens(seed)
        s = dict(x=torch.randn((c["T"], c["n"], c["C"]), device=DEV, generator=g).to(DTYPES[c["dtype"]]),
                 lif=_lif_params(g, c["C"]))
    elif kind == "sample":
        s = _sample_inputs(c, seed)
        s["ws"] = torch.empty(sample_workspace_bytes(c["rows"]), dtype=torch.uint8, device=DEV)
    else:
        s = _model_inputs(c, seed)
        model = SpikingDecoder(SpikingQwenConfig(num_hidden_layers=c["layers"]), device=DEV)
        model.load_reference_state_dict(s.pop("sd"))
        cache = PagedSpikeCache(c["layers"], 4, 2, 64, s["blocks"], BS, device=DEV)
        for (k, v), (k0, v0) in zip(cache.layers, s.pop("caches")):
            k.copy_(k0)
            v.copy_(v0)
        s.update(model=model, cache=cache)
        if kind == "decode":
            logits = torch.empty((c["n"], VOCAB), dtype=torch.bfloat16, device=DEV)

            def step():
                hidden = model.forward_paged(s["ids"], s["pos"], cache.layers, s["meta"])
                return (hidden, model.compute_logits(hidden, out=logits)) if c["head"] else (hidden,)

            s["graph"], s["out"] = _captured(step)
    s["case"] = c
    return s


def _lif_pack_inputs(c, seed):
    gc, g = _gens(seed)
    n, T, D, dt = c["n"], c["T"], c["D"], DTYPES[c["dtype"]]
    slots = BS * (-(-n // BS) * 2 + 1)
    # one projection output, its q, k and v heads viewed in place
    qkv = torch.randn((T, n, c["hq"] + 2 * c["hkv"], D), device=DEV, generator=g).to(dt)
    kv = (T, c["hkv"], slots, -(-D // 32))
    return dict(qkv=qkv, lif=[_lif_params(g, D) for _ in range(3)],
                slots=torch.randperm(slots, generator=gc)[:n].to(DEV),
                q=torch.zeros((T, n, c["hq"], kv[3]), dtype=torch.int32, device=DEV),
                kc=torch.zeros(kv, dtype=torch.int32, device=DEV), vc=torch.zeros(kv, dtype=torch.int32, device=DEV))


def _sample_inputs(c, seed):
    _, g = _gens(seed)
    R, V = c["rows"], c["vocab"]
    full = lambda v, dt=torch.float32: torch.full((R,), v, dtype=dt, device=DEV)
    return dict(logits=(torch.randn((R, V), device=DEV, generator=g) * c["scale"]).to(DTYPES[c["dtype"]]),
                temperature=full(c["temperature"]), k=full(c["top_k"], torch.int32), p=full(c["top_p"]),
                mp=full(c["min_p"]), rep=full(c["rep"]),
                hist=torch.randint(0, V, (R, 256), device=DEV, generator=g),
                hlen=full(150, torch.int32), u=torch.rand(R, device=DEV, generator=g))


# -- one pass --------------------------------------------------------------------
@torch.no_grad()
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "attn":
        return paged_spike_attn_decode(s["q"][0], s["k"][0], s["v"][0], s["tables"], s["lens"], c["D"], BS,
                                       c["hq"], c["hkv"], dtype=DTYPES[c["dtype"]])
    if kind in ("layers", "decode"):
        s["graph"].replay()
        if kind == "decode":
            return s["out"], s["cache"].layers[0]
        return s["out"]
    if kind == "step":
        out = paged_attention_fused(s["q"], s["k"], s["v"], *s["lif"], s["kc"], s["vc"], s["meta"], c["hq"],
                                    c["hkv"], c["D"])
        return out, s["kc"], s["vc"]
    if kind == "lif_pack":
        x, hq, hkv = s["qkv"], c["hq"], c["hkv"]
        lif_pack_write_sites([(x[:, :, :hq], *s["lif"][0], s["q"], False),
                              (x[:, :, hq:hq + hkv], *s["lif"][1], s["kc"], True),
                              (x[:, :, hq + hkv:], *s["lif"][2], s["vc"], True)], s["slots"])
        return s["q"], s["kc"], s["vc"]
    if kind == "lif":
        return lif_multistep(s["x"], *s["lif"], return_membrane=c["membrane"])
    if kind == "sample":
        k = c["top_k"]
        return sample_tokens(s["logits"], s["temperature"], s["k"], s["p"], s["mp"], s["rep"],
                             history=s["hist"], history_len=s["hlen"], uniforms=s["u"], workspace=s["ws"],
                             stages=1 if 0 < k <= 256 else 2)
    hidden = s["model"].forward_paged(s["ids"], s["pos"], s["cache"].layers, s["meta"])
    return hidden, s["model"].compute_logits(hidden, s["last"]), s["cache"].layers[0]


# -- what a pass cannot do without -------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    es = DTYPES[c["dtype"]].itemsize if "dtype" in c else 2
    if kind in ("attn", "layers"):
        L = c.get("layers", 1)
        lens = _lens(c["n"], c["lo"], c["hi"], torch.Generator().manual_seed(0))
        tok = int(lens.sum())
        words = c["D"] // 8
        return {"bytes": L * (tok * c["T"] * c["hkv"] * 2 * words + c["n"] * c["T"] * c["hq"] * (words + c["D"] * es)
                              + (tok // BS + 2 * c["n"]) * 4),
                "flops": L * 4 * tok * c["T"] * c["hq"] * c["D"]}
    if kind == "step":
        dec = c["n_dec"] * (c["hi"] * 5 // 8)
        chunks = _chunk_lens(c)
        n = c["n_dec"] + sum(q for q, _ in chunks)
        pairs = dec + sum(q * p + q * (q + 1) // 2 for q, p in chunks)
        seen = dec + sum(q + p for q, p in chunks)
        T, D = c["T"], c["D"]
        return {"bytes": T * D * (n * (2 * c["hq"] + 2 * c["hkv"]) * es + seen * c["hkv"] * 2 // 8),
                "flops": 4 * pairs * T * c["hq"] * D}
    if kind == "lif_pack":
        x = c["T"] * c["n"] * (c["hq"] + 2 * c["hkv"]) * c["D"]
        return {"bytes": x * es + x // 8 + 8 * c["n"], "flops": 6 * x}
    if kind == "lif":
        x = c["T"] * c["n"] * c["C"]
        return {"bytes": 2 * x * es + (4 * c["n"] * c["C"] if c["membrane"] else 0), "flops": 6 * x}
    if kind == "sample":
        return {"bytes": c["rows"] * (c["vocab"] * es + 8 * 150), "flops": 4 * c["rows"] * c["vocab"]}
    per_layer = HIDDEN * (18 * 64 + 14 * 64 + 3 * INTER)
    if kind == "decode":
        tok = c["n"] * (c["lo"] + c["hi"]) // 2
        n, pairs = c["n"], tok
        heads = c["n"] if c["head"] else 0
    else:
        n, heads = c["prompts"] * c["plen"], c["prompts"]
        tok = c["prompts"] * (c["plen"] + c["ctx"])
        pairs = c["prompts"] * (c["plen"] * c["ctx"] + c["plen"] * (c["plen"] + 1) // 2)
    return {"bytes": 2 * (c["layers"] * per_layer + bool(heads) * VOCAB * HIDDEN + heads * VOCAB + n * HIDDEN) +
            c["layers"] * tok * 4 * 2 * 2 * 8,
            "flops": 2 * (c["layers"] * per_layer * 4 * n + VOCAB * HIDDEN * heads) +
            c["layers"] * 4 * pairs * 4 * 14 * 64}


def tolerance(case):
    """Bits, words and tokens are whole.  Floating outputs: the output type's
    rounding (fp32: sums of 32-bit terms in another order); a decoder layer adds
    what other sums' bf16 roundings, and the few spikes they turn, change."""
    if case["kind"] in ("lif_pack", "lif", "sample"):
        return "exact"
    if case["kind"] == "decode":
        return {"rel": 5e-3, "max": 0.1, "differ": 1e-4}
    if case["kind"] == "prefill":
        return {"rel": 2e-2, "max": 0.3, "differ": 4e-4}
    return {"f32": {"rel": 1e-6, "max": 1e-5}, "f16": {"rel": 1e-3, "max": 4e-3},
            "bf16": {"rel": 8e-3, "max": 3e-2}}[case["dtype"]]


# -- the same in 64 bits, by plain torch -------------------------------------------
def _bits(words, D):
    """int32 [..., W] -> float64 [..., D] of 0 / 1: bit i of word w is channel 32 w + i."""
    b = (words[..., None] >> torch.arange(32, device=words.device, dtype=torch.int32)) & 1
    return b.flatten(-2)[..., :D].double()


def _pack(spikes):
    """0 / 1 [..., D] -> int32 [..., W]."""
    W = -(-spikes.shape[-1] // 32)
    b = torch.nn.functional.pad((spikes != 0).long(), (0, 32 * W - spikes.shape[-1]))
    w = (b.view(*b.shape[:-1], W, 32) << torch.arange(32, device=b.device)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).int()


def _lif(x, beta, th):
    """Spikes (bool) and final membrane.  A spike is decided by the fp32
    recurrence, multiply and add rounded separately: that is the operation."""
    beta, th = beta.float().clamp(0, 1), th.float()
    u = torch.zeros(x.shape[1:], device=x.device)
    out = []
    for t in range(x.shape[0]):
        r = (u - th > 0).float()
        u = beta * u + x[t].float() - r * th
        out.append(u - th > 0)
    return torch.stack(out), u


def _seq_kv(cache, table, n, D):
    """[T, Hkv, n, D] spikes of a sequence's first n tokens."""
    pos = torch.arange(n, device=cache.device)
    return _bits(cache.index_select(2, table.long()[pos // BS] * BS + pos % BS), D)


def _attend(q, k, v, first):
    """q [T, Hq, n, D] at positions first.. on k, v [T, Hkv, S, D], causal."""
    rep = q.shape[1] // k.shape[1]
    n, S, out = q.shape[2], k.shape[2], torch.empty_like(q)
    at = torch.arange(S, device=q.device)
    for t in range(q.shape[0]):
        for h in range(k.shape[1]):
            for a in range(0, n, 1024):
                b = min(n, a + 1024)
                s = q[t, h * rep:(h + 1) * rep, a:b] @ k[t, h].t() / math.sqrt(q.shape[-1])
                s = s.masked_fill(at > first + torch.arange(a, b, device=q.device)[:, None], -math.inf)
                out[t, h * rep:(h + 1) * rep, a:b] = torch.softmax(s, -1) @ v[t, h]
    return out


def _paged(q, kc, vc, meta, D):
    """Attention of a batch from its spikes q [T, n, Hq, D]: [T, n, Hq, D]."""
    out = torch.empty_like(q)
    for i in range(meta.num_decode_tokens):
        S, tab = int(meta.seq_lens[i]), meta.block_tables[i]
        o = _attend(q[:, i:i + 1].transpose(1, 2), _seq_kv(kc, tab, S, D), _seq_kv(vc, tab, S, D), S - 1)
        out[:, i:i + 1] = o.transpose(1, 2)
    for a, n, p, tab in zip(meta.prefill_query_starts, meta.prefill_query_lens, meta.prefill_context_lens,
                            meta.prefill_block_tables):
        o = _attend(q[:, a:a + n].transpose(1, 2), _seq_kv(kc, tab, p + n, D), _seq_kv(vc, tab, p + n, D), p)
        out[:, a:a + n] = o.transpose(1, 2)
    return out


def _norm(h, w):
    x = (h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS)).bfloat16().double()
    return (w.double() * x).bfloat16().double()


def _model_exact(c, s):
    """The decoder with its sums in 64 bits; values are rounded to bf16 where
    the model's type rounds them, since those roundings decide spikes."""
    b16 = lambda t: t.bfloat16().double()
    sd, T, n, D = s["sd"], 4, s["ids"].numel(), 64
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D)).to(DEV)
    fr = s["pos"].float()[:, None] * inv
    emb = torch.cat((fr, fr), -1)
    cos, sin = (f(emb).bfloat16().double()[None, :, None] for f in (torch.cos, torch.sin))
    h = sd["model.embed_tokens.weight"][s["ids"]].double().expand(T, n, HIDDEN)
    for i, (kc, vc) in enumerate(s["caches"]):
        p = f"model.layers.{i}."
        w = lambda name: sd[p + name].double()
        x = _norm(h, sd[p + "input_layernorm.weight"])
        spk = {}
        for site, heads in (("q", 14), ("k", 2), ("v", 2)):
            y = b16(x @ w(f"self_attn.{site}_proj.weight").t() + w(f"self_attn.{site}_proj.bias"))
            y = y.view(T, n, heads, D)
            if site != "v":
                rot = torch.cat((-y[..., D // 2:], y[..., :D // 2]), -1)
                y = b16(b16(y * cos) + b16(rot * sin))
            spk[site] = _lif(y, sd[p + f"self_attn.lif_{site}.lif.beta"],
                             sd[p + f"self_attn.lif_{site}.lif.threshold"])[0]
        for cache, site in ((kc, "k"), (vc, "v")):
            cache.index_copy_(2, s["meta"].slot_mapping, _pack(spk[site]).transpose(1, 2).contiguous())
        o = b16(_paged(spk["q"].double(), kc, vc, s["meta"], D)).view(T, n, 14 * D)
        h = b16(h + b16(o @ w("self_attn.o_proj.weight").t()))
        x = _norm(h, sd[p + "post_attention_layernorm.weight"])
        gate = _lif(b16(x @ w("mlp.gate_proj.weight").t()), sd[p + "mlp.lif_gate.lif.beta"],
                    sd[p + "mlp.lif_gate.lif.threshold"])[0]
        y = gate.double() * b16(x @ w("mlp.up_proj.weight").t())
        h = b16(h + b16(y @ w("mlp.down_proj.weight").t()))
    hidden = _norm(h, sd["model.norm.weight"]).mean(0)
    if c["kind"] == "decode" and not c["head"]:
        return (hidden,)
    rows = hidden if c["kind"] == "decode" else hidden[s["last"]]
    return hidden, b16(rows) @ sd["model.embed_tokens.weight"].double().t()


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("attn", "layers"):
        s = _attn_inputs(c, seed, c.get("layers", 1))
        out = torch.empty((c.get("layers", 1), c["T"], c["n"], c["hq"], c["D"]), dtype=torch.float64, device=DEV)
        for i in range(out.shape[0]):
            q = _bits(s["q"][i], c["D"])
            for j, S in enumerate(s["lens"].tolist()):
                k, v = (_seq_kv(s[x][i], s["tables"][j], S, c["D"]) for x in "kv")
                out[i, :, j:j + 1] = _attend(q[:, j:j + 1].transpose(1, 2), k, v, S - 1).transpose(1, 2)
        return out if kind == "layers" else out[0]
    if kind == "step":
        s = _step_inputs(c, seed)
        spk = [_lif(s[x], *s["lif"][i])[0] for i, x in enumerate("qkv")]
        for cache, x in ((s["kc"], spk[1]), (s["vc"], spk[2])):
            cache.index_copy_(2, s["meta"].slot_mapping, _pack(x).transpose(1, 2).contiguous())
        o = _paged(spk[0].double(), s["kc"], s["vc"], s["meta"], c["D"])
        return o.view(c["T"], 1, o.shape[1], -1), s["kc"], s["vc"]
    if kind == "lif":
        _, g = _gens(seed)
        x = torch.randn((c["T"], c["n"], c["C"]), device=DEV, generator=g).to(DTYPES[c["dtype"]])
        spikes, u = _lif(x, *_lif_params(g, c["C"]))
        return (spikes.double(), u.double()) if c["membrane"] else spikes.double()
    if kind in ("decode", "prefill"):
        s = _model_inputs(c, seed)
        out = _model_exact(c, s)
        return (out, (None, None)) if kind == "decode" else (*out, (None, None))
    return None  # whole numbers
