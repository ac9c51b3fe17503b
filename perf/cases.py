"""The work this package is timed on: attention steps, layers and packing.

Every case is one step of a serving engine through the package's public entry
points: a decode or verify gear replayed from its HIP graph, an eager step
(packing, step plan, the attention of some layers with the KV write), a whole
attention sub-block of a model layer, or the packing of a step alone.  A case
is a dict of plain values; its context lengths follow from the case alone
(``shape_seed``), its tensors from ``prepare``'s seed.

Head shapes are those the package is configured for elsewhere: 16/8/128
(Qwen3-0.6B), 28/4/128 (Qwen2-7B), 32/8/128 (MiMo-7B), 64/8/128
(Qwen2.5-72B), 14/2/64 (Qwen2.5-0.5B) and 16 latent heads of 512 + 64
(DeepSeek-V2-Lite).
"""
import math
import random

import torch

from auto_infer_amd import ops, packing
from auto_infer_amd.attention.gqa import GqaHipBackend
from auto_infer_amd.attention.metadata import step_plan
from auto_infer_amd.attention.mla import MlaHipBackend
from auto_infer_amd.execution import BatchPlan, RequestView, ScheduledRequest
from auto_infer_amd.graph import DecodeGraph, LatentDecodeGraph

BF16 = torch.bfloat16
LATENT, ROPE, NOPE, VDIM = 512, 64, 128, 128      # absorbed MLA
EPS = 1e-6

# Fields every case has.  kind: graph | latent_graph | step | latent_step |
# gqa_layer | mla_layer | pack.  rows: decode (verify) requests of `width`
# query tokens with contexts in [lo, hi] (`spread`); prompts: requests of
# [plo, phi] query tokens behind a prefix of [prefix_lo, prefix_hi] tokens.
DEFAULTS = dict(hq=16, hkv=8, d=128, bs=128, layers=1, rows=0, width=1, lo=128, hi=2048,
                spread="uniform", prompts=0, plo=512, phi=512, prefix_lo=0, prefix_hi=0,
                shared=0.0, layout="nd", hidden=0, shape_seed=1)


def _case(**kw):
    bad = set(kw) - set(DEFAULTS) - {"name", "kind"}
    assert not bad, bad
    return {**DEFAULTS, **kw}


def listed():
    return [
        # One decode step of a small model at its usual batch: 8 layers of a
        # captured gear, metadata restaged first (launch and latency bound).
        _case(name="decode_graph_b16", kind="graph", hq=16, hkv=8, layers=8, rows=16,
              lo=128, hi=2048, shape_seed=11),
        # A single user's long conversation, eager, small blocks: the smallest
        # batch, where one request must fill the chip.
        _case(name="decode_1x32k", kind="step", hq=28, hkv=4, bs=16, layers=8, rows=1,
              lo=31847, hi=31847, shape_seed=12),
        # A large model's decode batch with a long tail of contexts, packed
        # and attended eagerly: the bandwidth-bound extreme.
        _case(name="decode_b256_tail", kind="step", hq=64, hkv=8, rows=256, lo=64, hi=32768,
              spread="lognormal", shape_seed=13),
        # A full token budget of a continuous-batching scheduler: prefill
        # chunks beside decode rows, some sharing a cached prefix.
        _case(name="mixed_budget", kind="step", hq=28, hkv=4, rows=512, lo=256, hi=4096,
              prompts=3, plo=512, phi=512, prefix_hi=1024, shared=0.25, shape_seed=14),
        # Short new prompts of mixed lengths on the head_dim-64 model, blocks
        # of 16.
        _case(name="prompts_d64", kind="step", hq=14, hkv=2, d=64, bs=16, layers=4, prompts=7,
              plo=37, phi=1900, shape_seed=15),
        # One chunk of a long document: 512 tokens at the end of 32K keys.
        _case(name="chunk_at_32k", kind="step", hq=28, hkv=4, layers=2, prompts=1,
              prefix_lo=32256, prefix_hi=32256, shape_seed=16),
        # Speculative verify of one draft per request, in the graph gear of
        # the reference's NZ cache layout.
        _case(name="verify_graph_b16_nz", kind="graph", hq=32, hkv=8, layers=4, rows=16, width=2,
              lo=1024, hi=4096, layout="nz", shape_seed=17),
        # Latent (MLA) decode gear at a serving batch.
        _case(name="mla_decode_graph_b64", kind="latent_graph", layers=4, rows=64, lo=512, hi=8192,
              spread="log", shape_seed=18),
        # Latent prefill: prompts of mixed lengths, some behind a prefix.
        _case(name="mla_prompts", kind="latent_step", layers=2, prompts=5, plo=200, phi=2048,
              prefix_hi=3000, shape_seed=19),
        # A whole attention sub-block (projections, QK-norm, RoPE, KV write,
        # attention, output projection) over a prefill step.
        _case(name="gqa_layer_prefill", kind="gqa_layer", hq=16, hkv=8, layers=2, hidden=1024,
              prompts=4, plo=300, phi=900, shape_seed=20),
        # The same for an MLA layer: latent projections, W_UK and W_UV products.
        _case(name="mla_layer_prefill", kind="mla_layer", layers=2, hidden=2048, prompts=4,
              plo=300, phi=900, shape_seed=21),
        # Packing of a step alone: 240 decode rows and two prompt chunks into
        # device metadata.
        _case(name="pack_mixed", kind="pack", rows=240, lo=64, hi=8192, spread="log", prompts=2,
              plo=700, phi=1100, shape_seed=22),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["graph", "graph", "step", "step", "step", "step", "latent_graph",
                       "latent_step", "latent_step", "gqa_layer", "mla_layer", "pack"])
    hq, hkv, d = rng.choice([(16, 8, 128), (28, 4, 128), (32, 8, 128), (64, 8, 128), (14, 2, 64)])
    kw = dict(kind=kind, hq=hq, hkv=hkv, d=d, bs=rng.choice([16, 16, 32, 64, 128, 128]),
              shape_seed=rng.randrange(1 << 20))
    if kind in ("graph", "step"):
        kw["layout"] = rng.choice(["nd", "nd", "nz"])
    lo = _log_int(rng, 64, 4096)
    hi = min(32768, _log_int(rng, lo, 16 * lo))
    row_bytes = 1152 if kind in ("latent_graph", "latent_step", "mla_layer") else 4 * hkv * d

    def decode_rows(most, budget):      # rows whose keys stay within `budget` bytes
        return max(1, min(_log_int(rng, 1, most), int(budget / (hi * row_bytes))))

    def prompts(most_tokens):           # ragged prompts within a token budget
        phi = _log_int(rng, 33, most_tokens)
        return dict(prompts=max(1, min(_log_int(rng, 1, 12), most_tokens // phi)),
                    plo=max(9, phi // rng.choice([1, 2, 8])), phi=phi,
                    prefix_hi=rng.choice([0, 0, 700, _log_int(rng, 512, 12000)]))
    if kind in ("graph", "latent_graph"):
        kw.update(layers=2, rows=min(64, decode_rows(64, 5e8)), lo=lo, hi=hi, spread="log",
                  width=rng.choice([1, 1, 1, 2, 3]))
    elif kind == "step":
        form = rng.choice(["decode", "decode", "prompts", "mixed"])
        if form != "prompts":
            kw.update(rows=decode_rows(256, 1.5e9), lo=lo, hi=hi, spread="log")
        if form != "decode":
            kw.update(prompts(3000))
        kw["layers"] = 1 if form == "mixed" else 2
    elif kind == "latent_step":
        kw.update(prompts(3000), layers=1)
        if rng.random() < 0.3:
            kw.update(rows=rng.randint(1, 16), lo=lo, hi=hi, spread="log")
    elif kind in ("gqa_layer", "mla_layer"):
        kw.update(hidden=rng.choice([512, 1024, 2048]))
        if rng.random() < 0.4:
            kw.update(rows=min(128, decode_rows(128, 5e8)), lo=lo, hi=hi, spread="log")
        else:
            kw.update(prompts(3000))
    else:
        kw.update(rows=_log_int(rng, 1, 256), lo=lo, hi=hi, spread="log")
        if rng.random() < 0.4:
            kw.update(prompts(2000))
    return _case(**kw)


# ------------------------------------------------------------------ shapes

def _lengths(case):
    """(query tokens, context length) of each request, prompts first."""
    rng = random.Random(case["shape_seed"])
    out = []
    for _ in range(case["prompts"]):
        lq = _log_int(rng, case["plo"], case["phi"])
        out.append((lq, lq + rng.randint(case["prefix_lo"], case["prefix_hi"])))
    for _ in range(case["rows"]):
        lo, hi = case["lo"], case["hi"]
        if case["spread"] == "uniform":
            lk = rng.randint(lo, hi)
        elif case["spread"] == "log":
            lk = _log_int(rng, lo, hi)
        else:
            lk = int(min(hi, max(lo, rng.lognormvariate(math.log(2048), 1.0))))
        out.append((case["width"], max(lk, case["width"])))
    return out


def _is_latent(case):
    return case["kind"] in ("latent_graph", "latent_step", "mla_layer")


def _tables(case):
    """Physical block ids of every request: a seeded permutation of the pool;
    a `shared` part of the requests has its first four blocks in common.
    Returns (tables, pool size without the gear's scratch blocks)."""
    rng = random.Random(case["shape_seed"] + 7)
    bs = case["bs"]
    need = [(lk + bs - 1) // bs for _, lk in _lengths(case)]
    pool = sum(need) + sum(need) // 8 + 1
    ids = list(range(pool))
    rng.shuffle(ids)
    tables, common = [], None
    for (lq, lk), n in zip(_lengths(case), need):
        row, ids = ids[:n], ids[n:]
        if case["shared"] and lk - lq >= 4 * bs and rng.random() < case["shared"]:
            if common is None:
                common = row[:4]
            row = common + row[4:]
        tables.append(row)
    return tables, pool


def _visible(lq, lk):        # (query, key) pairs under the causal mask
    return lq * (lk - lq) + lq * (lq + 1) // 2


def work(case):
    lens = _lengths(case)
    T = sum(lq for lq, _ in lens)
    if case["kind"] == "pack":      # ids in, tokens/positions/slots and tables out
        blocks = sum(len(t) for t in _tables(case)[0])
        return {"bytes": 28 * T + 8 * blocks + 12 * len(lens), "flops": 0}
    tables, _ = _tables(case)
    keys = len({b for t in tables for b in t}) * case["bs"] - sum(
        -lk % case["bs"] for _, lk in lens)
    pairs = sum(_visible(lq, lk) for lq, lk in lens)
    if _is_latent(case):
        H = 16
        row = 2 * (LATENT + ROPE)
        flops = 2 * (2 * LATENT + ROPE) * H * pairs
        nbytes = keys * row + T * row + 2 * T * H * (2 * LATENT + ROPE)
    else:
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        flops = 4 * d * hq * pairs
        nbytes = 4 * hkv * d * (keys + T) + 4 * T * hq * d
    if case["kind"] == "gqa_layer":
        hid, width = case["hidden"], (hq + 2 * hkv) * d
        flops += 2 * T * hid * (width + hq * d)
        nbytes = 4 * hkv * d * keys + 2 * hid * (width + hq * d) + 4 * T * hid
    elif case["kind"] == "mla_layer":
        hid = case["hidden"]
        weights = hid * H * (NOPE + ROPE) + hid * (LATENT + ROPE) + H * VDIM * hid
        up = H * LATENT * (NOPE + VDIM)
        flops += 2 * T * (weights + up)
        nbytes = keys * row + 2 * (weights + up) + 4 * T * hid
    return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}


# bf16 inputs and outputs with fp32 sums.  An attention output rounds its
# probabilities and itself to bf16; a layer also rounds every projection.
# About four times the error measured against 64-bit arithmetic.
def tolerance(case):
    if case["kind"] == "pack":
        return "exact"
    if case["kind"] in ("gqa_layer", "mla_layer"):
        return {"rel": 2e-2, "max": 0.16}
    return {"rel": 1e-2, "max": 0.08}


# ------------------------------------------------------------------ inputs

def _randn(gen, *shape, scale=1.0):
    t = torch.randn(*shape, generator=gen, device="cuda", dtype=BF16)
    return t.mul_(scale) if scale != 1.0 else t


def _inputs(case, seed):
    """This step's tensors: caches (one allocation over the layers), query
    and new K/V rows or hidden states, weights, rotary tables."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lens = _lengths(case)
    T, L, bs = sum(lq for lq, _ in lens), case["layers"], case["bs"]
    tables, pool = _tables(case)
    pool += case["rows"]                       # a gear's scratch blocks
    x = {"lens": lens, "tables": tables, "pool": pool, "tokens": T}
    if case["kind"] == "pack":
        return x
    if _is_latent(case):
        H = 16
        x["cache"] = _randn(gen, L, pool, bs, 1, LATENT + ROPE)
        if case["kind"] != "mla_layer":
            x["q"] = _randn(gen, L, T, H, LATENT + ROPE)
            x["new"] = _randn(gen, L, T, 1, LATENT + ROPE)
    else:
        x["cache"] = _randn(gen, L, 2, pool, bs, case["hkv"], case["d"])
        if case["kind"] != "gqa_layer":
            x["q"] = _randn(gen, L, T, case["hq"], case["d"])
            x["k"] = _randn(gen, L, T, case["hkv"], case["d"])
            x["v"] = _randn(gen, L, T, case["hkv"], case["d"])
    if case["kind"] in ("gqa_layer", "mla_layer"):
        hid = case["hidden"]
        x["x"] = _randn(gen, T, hid)
        width = case["d"] if case["kind"] == "gqa_layer" else ROPE
        pos = torch.tensor([p for lq, lk in lens for p in range(lk - lq, lk)], device="cuda",
                           dtype=torch.float64)
        inv = 1e4 ** (-torch.arange(0, width, 2, device="cuda", dtype=torch.float64) / width)
        ang = (pos[:, None] * inv).repeat(1, 2)[:, None]
        x["cos"], x["sin"] = ang.cos().to(BF16), ang.sin().to(BF16)
        w = x["w"] = {}
        for i in range(L):
            p = f"model.layers.{i}.self_attn."
            if case["kind"] == "gqa_layer":
                hq, hkv, d = case["hq"], case["hkv"], case["d"]
                w[p + "qkv_proj.weight"] = _randn(gen, (hq + 2 * hkv) * d, hid, scale=hid ** -0.5)
                w[p + "q_norm.weight"] = 1 + _randn(gen, d, scale=0.1)
                w[p + "k_norm.weight"] = 1 + _randn(gen, d, scale=0.1)
                w[p + "o_proj.weight"] = _randn(gen, hid, hq * d, scale=(hq * d) ** -0.5)
            else:
                w[p + "q_proj.weight"] = _randn(gen, H * (NOPE + ROPE), hid, scale=hid ** -0.5)
                w[p + "kv_a_proj_with_mqa.weight"] = _randn(gen, LATENT + ROPE, hid,
                                                            scale=hid ** -0.5)
                w[p + "kv_a_layernorm.weight"] = 1 + _randn(gen, LATENT, scale=0.1)
                w[p + "kv_b_proj.weight"] = _randn(gen, H * (NOPE + VDIM), LATENT,
                                                   scale=LATENT ** -0.5)
                w[p + "o_proj.weight"] = _randn(gen, hid, H * VDIM, scale=(H * VDIM) ** -0.5)
    return x


def _scale(case):
    return (NOPE + ROPE) ** -0.5 if _is_latent(case) else case["d"] ** -0.5


def _batch_plan(case, x, seed):
    """The scheduler's immutable snapshot of this step."""
    rng = random.Random(seed)
    views, tables, items = {}, {}, []
    draft_depth = case["width"] - 1 if case["kind"] in ("graph", "latent_graph") else 0
    for i, ((lq, lk), blocks) in enumerate(zip(x["lens"], x["tables"])):
        rid, prompt = f"r{i}", i < case["prompts"]
        start = rng.randrange(1 << 16)
        tokens = tuple((start + 31 * t) % 151936 for t in range(lk - draft_depth))
        drafts = tuple(rng.randrange(151936) for _ in range(draft_depth))
        views[rid] = RequestView(rid, tokens, lk - lq, lk if prompt else 1, lk if prompt else 1,
                                 drafts)
        tables[rid] = tuple(blocks)
        items.append(ScheduledRequest(rid, lq, prompt, tuple(blocks)))
    return BatchPlan.make(items, views, tables)


# One compute stream for all captured gears, as an engine has.
_STREAM = []


def _gear_stream():
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def _stager(case, x):
    g, w = case["rows"], case["width"]
    most = max(len(t) for t in x["tables"])

    def zeros(n, dtype):
        return torch.zeros(n, dtype=dtype, device="cuda")
    common = dict(tid=zeros(g * w, torch.long), positions=zeros(g * w, torch.long),
                  slots=zeros(g * w, torch.int32),
                  block_table=torch.zeros(g, most, dtype=torch.int32, device="cuda"),
                  block_size=case["bs"], scratch0=x["pool"] - g)
    if w == 1:
        return packing.DecodeInputStager(**common)
    return packing.SpecDecodeInputStager(
        drafts=torch.zeros(g, w - 1, dtype=torch.long, device="cuda"), draft_depth=w - 1, **common)


def prepare(case, seed):
    x = _inputs(case, seed)
    s = {"case": case, "x": x, "plan": _batch_plan(case, x, seed)}
    kind = case["kind"]
    if kind in ("graph", "latent_graph"):
        stream = _gear_stream()
        stager = _stager(case, x)
        if kind == "graph":
            g = DecodeGraph(stager, [(c[0], c[1]) for c in x["cache"]], num_q_heads=case["hq"],
                            num_kv_heads=case["hkv"], head_dim=case["d"], stream=stream,
                            kv_layout=case["layout"])
            g.q, g.k_new, g.v_new = x["q"], x["k"], x["v"]
        else:
            g = LatentDecodeGraph(stager, list(x["cache"]), num_heads=16, scale=_scale(case),
                                  stream=stream)
            g.q, g.latent_new = x["q"], x["new"]
        torch.cuda.synchronize()
        g.stage(s["plan"])
        g.capture()
        s["gear"] = g
        return s
    s["packer"] = packing.DeviceBatchPacker(case["bs"], "cuda")
    if kind == "gqa_layer":
        s["backend"] = GqaHipBackend(case["hq"], case["hkv"], case["d"], _scale(case),
                                     case["layers"], "cuda", BF16, w=x["w"], rms_eps=EPS)
        s["caches"] = list(x["cache"])
    elif kind == "mla_layer":
        s["backend"] = MlaHipBackend(x["w"], num_heads=16, qk_nope=NOPE, qk_rope=ROPE,
                                     v_head_dim=VDIM, kv_lora_rank=LATENT, q_lora_rank=None,
                                     rms_eps=EPS, softmax_scale=_scale(case),
                                     num_layers=case["layers"], device="cuda", dtype=BF16)
        s["caches"] = [(c, c) for c in x["cache"]]
    return s


def run(s):
    case, x = s["case"], s["x"]
    kind, L = case["kind"], case["layers"]
    if "gear" in s:
        g = s["gear"]
        staged = g.stage(s["plan"])
        g.replay()
        return {"out": g.out, "cache": x["cache"], "slots": staged.slots}
    ctx, _, _ = s["packer"].build(s["plan"], s.get("backend"), s.get("caches"))
    if kind == "pack":
        return {"token_ids": ctx.token_ids, "positions": ctx.positions,
                "slots": ctx.slot_mapping, "block_table": ctx.block_table,
                "cu_seqlens_q": ctx.aia_cu_seqlens_q, "seqlens_kv": ctx.aia_seqlens_kv}
    if kind in ("gqa_layer", "mla_layer"):
        ctx.cos, ctx.sin = x["cos"], x["sin"]
        outs = [s["backend"].attention(i, x["x"], ctx) for i in range(L)]
    elif kind == "latent_step":
        plan = step_plan(ctx, 16, 1, LATENT, case["bs"])
        outs = []
        for i in range(L):
            ops.write_kv(x["new"][i], None, x["cache"][i], None, ctx.slot_mapping)
            outs.append(ops.paged_attention_mla(x["q"][i], x["cache"][i], plan, _scale(case)))
    else:
        plan = step_plan(ctx, case["hq"], case["hkv"], case["d"], case["bs"])
        outs = [ops.paged_attention_gqa(x["q"][i], x["cache"][i, 0], x["cache"][i, 1], plan,
                                        _scale(case), key_new=x["k"][i], value_new=x["v"][i],
                                        kv_layout=case["layout"])
                for i in range(L)]
    return {"out": outs, "cache": x["cache"], "slots": ctx.slot_mapping}


# ------------------------------------------------------------------ 64 bits

def _write_rows(case, cache, rows, x):
    """rows (T, heads, dim) at this step's slots of one cache, in its layout."""
    bs = case["bs"]
    slots = torch.tensor([t[p // bs] * bs + p % bs for (lq, lk), t in zip(x["lens"], x["tables"])
                          for p in range(lk - lq, lk)], device="cuda")
    if case["layout"] == "nz":
        nz = cache.view(cache.shape[0], -1, bs, 16)
        nz[slots // bs, :, slots % bs] = rows.reshape(rows.shape[0], -1, 16)
    else:
        cache.view(-1, *cache.shape[2:])[slots] = rows


def _keys(case, cache, table, lk):
    """The first lk keys of a request, (lk, heads, dim) in 64 bits."""
    blocks = cache[torch.tensor(table, device="cuda")].double()
    n, bs, heads, dim = blocks.shape
    if case["layout"] == "nz":
        blocks = blocks.view(n, -1, bs, 16).transpose(1, 2)
    return blocks.reshape(n * bs, heads, dim)[:lk]


def _attend(case, q, kc, vc, vdim, x):
    """Softmax attention of this step's rows over one layer's caches."""
    out = torch.empty(*q.shape[:2], vdim, dtype=torch.float64, device="cuda")
    t0 = 0
    for (lq, lk), table in zip(x["lens"], x["tables"]):
        k = _keys(case, kc, table, lk)
        v = k if vc is kc else _keys(case, vc, table, lk)
        group = q.shape[1] // k.shape[1]
        hidden = (torch.arange(lk, device="cuda")[None] >
                  torch.arange(lk - lq, lk, device="cuda")[:, None]) if lq > 1 else None
        for h in range(k.shape[1]):
            kt, vh = k[:, h].t().contiguous(), v[:, h, :vdim].contiguous()
            for j in range(h * group, (h + 1) * group):
                sc = (q[t0:t0 + lq, j].double() @ kt) * _scale(case)
                if hidden is not None:
                    sc.masked_fill_(hidden, -math.inf)
                out[t0:t0 + lq, j] = torch.softmax(sc, dim=-1) @ vh
        t0 += lq
    return out


def _norm(v, w):
    return v * torch.rsqrt((v * v).mean(-1, keepdim=True) + EPS) * w


def _rope(v, x):
    a, b = v.chunk(2, dim=-1)
    return v * x["cos"].double() + torch.cat((-b, a), -1) * x["sin"].double()


def _pairs(v):               # interleaved pairs to halves
    return torch.cat((v[..., 0::2], v[..., 1::2]), -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "pack":
        return None
    if sum(lk for _, lk in _lengths(case)) > 2_000_000:
        return None
    x = _inputs(case, seed)
    T, L = x["tokens"], case["layers"]
    # A layer's written rows are computed; elsewhere they are the inputs.
    layer = kind in ("gqa_layer", "mla_layer")
    cache = x["cache"].double() if layer else x["cache"]
    outs = []
    for i in range(L):
        w = {k.split("self_attn.")[1][:-7]: v.double() for k, v in x["w"].items()
             if k.startswith(f"model.layers.{i}.")} if layer else None
        h = x["x"].double() if layer else None
        if kind == "gqa_layer":
            hq, hkv, d = case["hq"], case["hkv"], case["d"]
            qkv = (h @ w["qkv_proj"].t()).view(T, hq + 2 * hkv, d)
            q = _rope(_norm(qkv[:, :hq], w["q_norm"]), x)
            k = _rope(_norm(qkv[:, hq:hq + hkv], w["k_norm"]), x)
            v = qkv[:, hq + hkv:]
        elif kind == "mla_layer":
            q = (h @ w["q_proj"].t()).view(T, 16, NOPE + ROPE)
            wb = w["kv_b_proj"].view(16, NOPE + VDIM, LATENT)
            ql = torch.stack([q[:, j, :NOPE] @ wb[j, :NOPE] for j in range(16)], 1)
            q = torch.cat((ql, _rope(_pairs(q[..., NOPE:]), x)), -1)
            ckv = h @ w["kv_a_proj_with_mqa"].t()
            k = torch.cat((_norm(ckv[:, :LATENT], w["kv_a_layernorm"]).unsqueeze(1),
                           _rope(_pairs(ckv[:, None, LATENT:]), x)), -1)
        elif _is_latent(case):
            q, k = x["q"][i], x["new"][i]
        else:
            q, k, v = x["q"][i], x["k"][i], x["v"][i]
        if _is_latent(case):
            _write_rows(case, cache[i], k, x)
            o = _attend(case, q, cache[i], cache[i], LATENT, x)
            if kind == "mla_layer":
                o = torch.stack([o[:, j] @ wb[j, NOPE:].t() for j in range(16)], 1)
        else:
            _write_rows(case, cache[i, 0], k, x)
            _write_rows(case, cache[i, 1], v, x)
            o = _attend(case, q, cache[i, 0], cache[i, 1], case["d"], x)
        outs.append(o.reshape(T, -1) @ w["o_proj"].t() if layer else o)
    if kind in ("graph", "latent_graph"):
        outs = torch.stack(outs)
    return {"out": outs, "cache": cache.double(), "slots": None}
