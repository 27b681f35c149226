"""The work that a user of this framework has it do, as cases to time and compare.

Every case is one pass through the public entry points (``OpsEngine``,
``WeaverEngine``, ``WeaverKvCache``) over synthetic inputs made on the GPU from a
seed.  Widths are those of the model presets (``fabric.model_dims``: llama8b,
granite2b, qwen05b, deepseek_r1_1_5b); pools, windows and dictionaries those of
``workloads.py`` and of the benchmark.

Kinds of case (the field ``kind``):
  attention  causal GQA attention of the newest ``queries`` tokens over
             contiguous K and V caches (``OpsEngine.multihead_attention``)
  mlp        a layer's MLP: norm, gate, up, SiLU gate, down, residual add
  qkv        a layer's attention input: norm, q/k/v products, RoPE, cache append
  forward    a prompt through whole layers to the last token's logits
  weaver     batched hot+cold decode over two pools (``decode_device``)
  tiered     one step of the tiered KV cache over its layers (``append``, ``attend``)
  distill    hot blocks to SparseCodes with their entropy proxy (``encode_device``)
"""
from __future__ import annotations

import math

import torch

from aether_nexus_amd import workloads
from aether_nexus_amd.inference import WeaverKvCache
from aether_nexus_amd.ops import OpsEngine
from aether_nexus_amd.weaver import WeaverEngine, make_encode_desc

DEVICE = "cuda:0"
EPS = 1e-5
THETA = 500000.0

#: (q_heads, kv_heads, head_dim, hidden, inter, vocab) of the presets in fabric.hip.
WIDTHS = {
    "llama8b": (32, 8, 128, 4096, 14336, 128256),
    "granite2b": (32, 8, 64, 2048, 8192, 49155),
    "qwen05b": (14, 2, 64, 896, 4864, 151936),
    "deepseek_r1_1_5b": (12, 2, 128, 1536, 8960, 151936),
}


def _model(name: str) -> dict:
    q_heads, kv_heads, head_dim, hidden, inter, vocab = WIDTHS[name]
    return {"q_heads": q_heads, "kv_heads": kv_heads, "head_dim": head_dim, "hidden": hidden, "inter": inter,
            "vocab": vocab}


def _only(d: dict, *names: str) -> dict:
    return {n: d[n] for n in names}


def _attention(model: str, queries: int, kv_len: int) -> dict:
    return {"kind": "attention", **_only(_model(model), "q_heads", "kv_heads", "head_dim"), "queries": queries,
            "kv_len": kv_len}


def _mlp(model: str, tokens: int) -> dict:
    return {"kind": "mlp", **_only(_model(model), "hidden", "inter"), "tokens": tokens}


def _qkv(model: str, tokens: int, start: int) -> dict:
    return {"kind": "qkv", **_only(_model(model), "q_heads", "kv_heads", "head_dim", "hidden"), "tokens": tokens,
            "start": start}


def _forward(model: str, layers: int, tokens: int) -> dict:
    return {"kind": "forward", **_model(model), "layers": layers, "tokens": tokens}


def _weaver(batch: int, hot: int, cold: int, *, layers: int = 1, queries: int = 1, atoms: int = 4096,
            dict_heads: int = 1, zipf: float = 0.0, head_blocked: bool = True) -> dict:
    return {"kind": "weaver", "layers": layers, "batch": batch, "queries": queries, "q_heads": 32, "kv_heads": 8,
            "head_dim": 128, "hot": hot, "cold": cold, "atoms": atoms, "dict_heads": dict_heads, "zipf": zipf,
            "head_blocked": head_blocked}


def _tiered(model: str, layers: int, queries: int, hot: int, cold: int) -> dict:
    return {"kind": "tiered", **_only(_model(model), "q_heads", "kv_heads", "head_dim"), "layers": layers,
            "queries": queries, "hot": hot, "cold": cold, "atoms": 512}


def _distill(model: str, blocks: int, atoms: int, entropy: bool, head_blocked: bool) -> dict:
    m = _model(model)
    return {"kind": "distill", **_only(m, "kv_heads", "head_dim"), "blocks": blocks, "atoms": atoms,
            "dict_heads": m["kv_heads"], "entropy": entropy, "head_blocked": head_blocked}


def listed() -> list:
    def named(name: str, case: dict) -> dict:
        return {"name": name, **case}
    return [
        # One new token over a full cache: the attention of a decode step, one layer.
        named("attention_decode", _attention("llama8b", 1, 4096)),
        # A piece of a prompt behind an earlier part of it: ragged sizes, 7 q heads to a kv head, 64 dims.
        named("attention_chunk", _attention("qwen05b", 509, 1531)),
        # A whole prompt at once.
        named("attention_prefill", _attention("llama8b", 2048, 2048)),
        # A layer's MLP for one new token (decode): reading the weights is all of it.
        named("mlp_decode", _mlp("llama8b", 1)),
        # The same for the 16 tokens that one forward batch holds at most (drafts, prompt pieces).
        named("mlp_batch", _mlp("llama8b", 16)),
        # The same for a prompt.
        named("mlp_prefill", _mlp("llama8b", 2048)),
        # A short prompt of odd length into a layer's attention: too many tokens for the decode products, few for tiles.
        named("qkv_chunk", _qkv("granite2b", 117, 1000)),
        # A prompt through four whole layers to logits: the ops in the order of the inference loop.
        named("forward_prefill", _forward("llama8b", 4, 512)),
        # The batched decode of the benchmark's head line: 64 sequences, 2048 exact and 32768 coded tokens each.
        named("weaver_batch", _weaver(64, 2048, 32768)),
        # A verify step of 8 drafts for 8 sequences over long coded contexts (4 of the benchmark's 32 layers).
        named("weaver_verify", _weaver(8, 2048, 65536, layers=4, queries=8)),
        # One decode step of one long conversation in the tiered cache, over the layers of a quarter of a model.
        named("tiered_step", _tiered("llama8b", 8, 1, 2048, 32768)),
        # One pass of the distiller over the whole hot region of a fabric, with the proxies that choose blocks.
        named("distill", _distill("llama8b", 8192, 512, True, True)),
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """A whole number in lo..hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["attention", "attention", "mlp", "mlp", "qkv", "forward", "weaver", "weaver", "tiered",
                       "distill"])
    model = rng.choice(sorted(WIDTHS))
    if kind == "attention":
        queries = _spread(rng, 1, 2048)
        return _attention(model, queries, queries + _spread(rng, 1, 4096) - 1)
    if kind == "mlp":
        return _mlp(model, _spread(rng, 1, 2048))
    if kind == "qkv":
        return _qkv(model, _spread(rng, 1, 2048), rng.randrange(0, 4096))
    if kind == "forward":
        return _forward(model, rng.randrange(1, 5), _spread(rng, 1, 512))
    if kind == "weaver":
        if rng.random() < 0.3:  # verify steps, causal drafts
            return _weaver(rng.randrange(1, 9), 16 * rng.randrange(1, 129), 16 * _spread(rng, 64, 4096),
                           layers=rng.randrange(1, 5), queries=rng.randrange(2, 9))
        per_head = rng.random() < 0.4  # the fabric's own dictionaries, else the shared one of the sweep
        return _weaver(_spread(rng, 1, 64), 16 * rng.randrange(1, 129), 16 * _spread(rng, 64, 2048),
                       atoms=512 if per_head else 4096, dict_heads=8 if per_head else 1,
                       zipf=1.1 if rng.random() < 0.3 else 0.0, head_blocked=rng.random() < 0.7)
    if kind == "tiered":
        return _tiered(rng.choice(["llama8b", "granite2b"]), rng.randrange(1, 9), rng.randrange(1, 9),
                       16 * rng.randrange(8, 129), 16 * _spread(rng, 16, 2048))
    return _distill(model, _spread(rng, 16, 8192), 512, rng.random() < 0.5, rng.random() < 0.7)


# ---------------------------------------------------------------- inputs

_engines: dict = {}


def _engine() -> WeaverEngine:
    """The engine of the process, as a program keeps one per GPU."""
    if "weaver" not in _engines:
        torch.zeros(1, device=DEVICE)
        _engines["weaver"] = WeaverEngine()
        _engines["ops"] = OpsEngine(_engines["weaver"])
    return _engines["weaver"]


class _Rand:
    """Normal f16 tensors on the GPU from one seed."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def __call__(self, *shape, scale: float = 1.0, mean: float = 0.0) -> torch.Tensor:
        t = torch.randn(shape, generator=self.gen, device=DEVICE, dtype=torch.float32)
        return t.mul_(scale).add_(mean).to(torch.float16)


def _empty(*shape, dtype=torch.float16) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=DEVICE)


def _blocks_up(tokens: int) -> int:
    return -(-tokens // 16) * 16


def _attention_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    cap = _blocks_up(c["kv_len"])
    return {"q": r(c["queries"], c["q_heads"], c["head_dim"]), "k": r(cap, c["kv_heads"], c["head_dim"]),
            "v": r(cap, c["kv_heads"], c["head_dim"])}


def _mlp_weights(r: _Rand, hidden: int, inter: int) -> dict:
    return {"ln2": r(hidden, scale=0.1, mean=1.0), "wg": r(inter, hidden, scale=hidden ** -0.5),
            "wu": r(inter, hidden, scale=hidden ** -0.5), "wd": r(hidden, inter, scale=inter ** -0.5)}


def _qkv_weights(r: _Rand, hidden: int, nq: int, nkv: int) -> dict:
    s = hidden ** -0.5
    return {"ln1": r(hidden, scale=0.1, mean=1.0), "wq": r(nq, hidden, scale=s), "wk": r(nkv, hidden, scale=s),
            "wv": r(nkv, hidden, scale=s)}


def _mlp_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    return {"x": r(c["tokens"], c["hidden"]), **_mlp_weights(r, c["hidden"], c["inter"])}


def _qkv_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    return {"x": r(c["tokens"], c["hidden"]),
            **_qkv_weights(r, c["hidden"], c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"])}


def _forward_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    h, nq, nkv = c["hidden"], c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    layers = [{**_qkv_weights(r, h, nq, nkv), "wo": r(h, nq, scale=nq ** -0.5), **_mlp_weights(r, h, c["inter"])}
              for _ in range(c["layers"])]
    ids = torch.randint(0, c["vocab"], (c["tokens"],), generator=r.gen, device=DEVICE, dtype=torch.int32)
    return {"layers": layers, "ids": ids, "embed": r(c["vocab"], h), "ln": r(h, scale=0.1, mean=1.0),
            "head": r(c["vocab"], h, scale=h ** -0.5)}


def _weaver_inputs(c: dict, seed: int) -> workloads.Workload:
    geom = workloads.Geometry(layers=c["layers"], batch=c["batch"], queries=c["queries"], q_heads=c["q_heads"],
                              kv_heads=c["kv_heads"], head_dim=c["head_dim"], dict_size=c["atoms"],
                              dict_heads=c["dict_heads"], hot_count=c["hot"] // 16, cold_count=c["cold"] // 16,
                              scale=c["head_dim"] ** -0.5, causal=c["queries"] > 1, zipf=c["zipf"] or None)
    return workloads.generate(geom, seed=seed, device=DEVICE)


def _tiered_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    shape = (c["kv_heads"], c["head_dim"])
    n = c["hot"] + c["cold"]
    d = torch.randn((c["layers"], c["kv_heads"], c["atoms"], c["head_dim"]), generator=r.gen, device=DEVICE)
    return {"dicts": (d / d.norm(dim=-1, keepdim=True)).to(torch.float16),
            "ks": [r(n, *shape) for _ in range(c["layers"])], "vs": [r(n, *shape) for _ in range(c["layers"])],
            "k": [r(c["queries"], *shape) for _ in range(c["layers"])],
            "v": [r(c["queries"], *shape) for _ in range(c["layers"])],
            "q": [r(c["queries"], c["q_heads"], c["head_dim"]) for _ in range(c["layers"])]}


def _distill_inputs(c: dict, seed: int) -> dict:
    r = _Rand(seed)
    d = torch.randn((c["dict_heads"], c["atoms"], c["head_dim"]), generator=r.gen, device=DEVICE)
    return {"hot": r(c["blocks"], 16, c["kv_heads"], c["head_dim"]),
            "dict": (d / d.norm(dim=-1, keepdim=True)).to(torch.float16),
            "src": torch.arange(c["blocks"], dtype=torch.int32, device=DEVICE)}


def prepare(case: dict, seed: int) -> dict:
    c, engine = case, _engine()
    st = {"case": c, "engine": engine, "ops": _engines["ops"]}
    kind = c["kind"]
    if kind == "attention":
        st.update(_attention_inputs(c, seed))
        st["out"] = torch.empty_like(st["q"])
    elif kind == "mlp":
        st.update(_mlp_inputs(c, seed))
        t, h, n = c["tokens"], c["hidden"], c["inter"]
        st.update(hid=_empty(t, h), norm=_empty(t, h), gate=_empty(t, n), up=_empty(t, n))
    elif kind == "qkv":
        st.update(_qkv_inputs(c, seed))
        t, kvd = c["tokens"], c["kv_heads"] * c["head_dim"]
        st.update(norm=_empty(t, c["hidden"]), q=_empty(t, c["q_heads"] * c["head_dim"]), k=_empty(t, kvd),
                  v=_empty(t, kvd), k_cache=torch.zeros((c["start"] + t, kvd), dtype=torch.float16, device=DEVICE),
                  v_cache=torch.zeros((c["start"] + t, kvd), dtype=torch.float16, device=DEVICE))
    elif kind == "forward":
        st.update(_forward_inputs(c, seed))
        t, h, n = c["tokens"], c["hidden"], c["inter"]
        qd, kvd = c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        caches = [torch.zeros((_blocks_up(t), kvd), dtype=torch.float16, device=DEVICE) for _ in range(2 * c["layers"])]
        st.update(hid=_empty(t, h), norm=_empty(t, h), q=_empty(t, qd), att=_empty(t, qd), k=_empty(t, kvd),
                  v=_empty(t, kvd), gate=_empty(t, n), up=_empty(t, n), last=_empty(1, h),
                  k_cache=caches[:c["layers"]], v_cache=caches[c["layers"]:],
                  logits=_empty(1, c["vocab"], dtype=torch.float32))
    elif kind == "weaver":
        wl = _weaver_inputs(c, seed)
        out = _empty(*wl.out_shape())
        cold = None
        if c["head_blocked"]:  # the order in which a fabric keeps its codes on the device
            cold = workloads.head_blocked(wl.cold)
            wl.cold = None
        st.update(out=out, desc=workloads.device_desc(wl, out, cold_head_blocked=cold))
    elif kind == "tiered":
        i = _tiered_inputs(c, seed)
        cache = WeaverKvCache(c["layers"], c["kv_heads"], c["head_dim"], i["dicts"], hot_window=c["hot"],
                              max_seq_len=c["hot"] + c["cold"] + 64, device=DEVICE)
        cache.extend(engine, i["ks"], i["vs"])
        st.update(cache=cache, q=i["q"], k=i["k"], v=i["v"], out=[torch.empty_like(q) for q in i["q"]])
    elif kind == "distill":
        i = _distill_inputs(c, seed)
        cold = torch.zeros((c["blocks"] * 16 * c["kv_heads"], 8), dtype=torch.int16, device=DEVICE)
        ent = _empty(c["blocks"], dtype=torch.float32) if c["entropy"] else None
        st.update(cold=cold, ent=ent, desc=make_encode_desc(
            kv_heads=c["kv_heads"], head_dim=c["head_dim"], dict_size=c["atoms"], dict_heads=c["dict_heads"],
            hot_blocks=c["blocks"], cold_blocks=c["blocks"], hot=i["hot"], dictionary=i["dict"],
            src_blocks=i["src"], cold=cold, entropy=ent, cold_head_blocked=c["head_blocked"]))
    return st


# ---------------------------------------------------------------- one pass


def _run_mlp(ops: OpsEngine, w: dict, st: dict, hid: torch.Tensor, t: int, h: int, n: int) -> None:
    """The MLP half of a layer on the residual stream ``hid``: the fused gate up to the 64 rows that it takes."""
    ops.rms_norm(hid, w["ln2"], st["norm"], h, t, EPS)
    if t <= 64:
        ops.matmul_silu_gate(st["norm"], w["wg"], w["wu"], st["gate"], t, n, h)
    else:
        ops.matmul(st["norm"], w["wg"], st["gate"], t, n, h)
        ops.matmul(st["norm"], w["wu"], st["up"], t, n, h)
        ops.silu_gate(st["gate"], st["up"], st["gate"], t * n)
    ops.matmul_add_residual(st["gate"], w["wd"], hid, t, h, n)


def _run_qkv(ops: OpsEngine, c: dict, w: dict, st: dict, x: torch.Tensor, k_cache: torch.Tensor,
             v_cache: torch.Tensor, start: int) -> None:
    t, h = c["tokens"], c["hidden"]
    qd, kvd = c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    ops.rms_norm(x, w["ln1"], st["norm"], h, t, EPS)
    ops.matmul_qkv(st["norm"], w["wq"], w["wk"], w["wv"], st["q"], st["k"], st["v"], t, qd, kvd, h)
    ops.rope(st["q"], st["k"], t, c["q_heads"], c["kv_heads"], c["head_dim"], start, THETA)
    ops.copy_buffer(st["k"], k_cache, t * kvd, 0, start * kvd)
    ops.copy_buffer(st["v"], v_cache, t * kvd, 0, start * kvd)


def run(state: dict):
    st, c, engine, ops = state, state["case"], state["engine"], state["ops"]
    kind = c["kind"]
    if kind == "attention":
        ops.multihead_attention(st["q"], st["k"], st["v"], st["out"], c["kv_len"], c["head_dim"], c["q_heads"],
                                c["kv_heads"], c["queries"])
        return st["out"]
    if kind == "mlp":
        t, h, n = c["tokens"], c["hidden"], c["inter"]
        ops.copy_buffer(st["x"], st["hid"], t * h, 0, 0)  # the residual stream arrives
        _run_mlp(ops, st, st, st["hid"], t, h, n)
        return st["hid"]
    if kind == "qkv":
        _run_qkv(ops, c, st, st, st["x"], st["k_cache"], st["v_cache"], c["start"])
        return {"q": st["q"], "k": st["k_cache"][c["start"]:], "v": st["v_cache"][c["start"]:]}
    if kind == "forward":
        t, h, n, qd = c["tokens"], c["hidden"], c["inter"], c["q_heads"] * c["head_dim"]
        ops.embed_lookup(st["ids"], st["embed"], st["hid"], h, t)
        for w, k_cache, v_cache in zip(st["layers"], st["k_cache"], st["v_cache"]):
            _run_qkv(ops, c, w, st, st["hid"], k_cache, v_cache, 0)
            ops.multihead_attention(st["q"], k_cache, v_cache, st["att"], t, c["head_dim"], c["q_heads"],
                                    c["kv_heads"], t)
            ops.matmul_add_residual(st["att"], w["wo"], st["hid"], t, h, qd)
            _run_mlp(ops, w, st, st["hid"], t, h, n)
        ops.rms_norm(st["hid"][t - 1:], st["ln"], st["last"], h, 1, EPS)
        ops.matmul_scaled(st["last"], st["head"], st["logits"], 1, c["vocab"], h, 1.0)
        return {"logits": st["logits"], "hidden": st["hid"]}
    if kind == "weaver":
        engine.decode_device(st["desc"])
        return st["out"]
    if kind == "tiered":
        cache = st["cache"]
        for layer in range(c["layers"]):
            cache.append(layer, st["k"][layer], st["v"][layer])
            cache.attend(engine, layer, st["q"][layer], st["out"][layer])
        return st["out"]
    engine.encode_device(st["desc"])
    return {"codes": st["cold"], "entropy": st["ent"]} if c["entropy"] else {"codes": st["cold"]}


# ---------------------------------------------------------------- what a pass cannot do without


def _attention_flops(queries: int, kv_len: int, q_heads: int, head_dim: int) -> int:
    pairs = queries * (kv_len - queries) + queries * (queries + 1) // 2
    return 4 * pairs * q_heads * head_dim


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind == "attention":
        kv = 2 * c["kv_len"] * c["kv_heads"] * c["head_dim"] * 2
        qo = 2 * c["queries"] * c["q_heads"] * c["head_dim"] * 2
        return {"bytes": kv + qo, "flops": _attention_flops(c["queries"], c["kv_len"], c["q_heads"], c["head_dim"])}
    if kind == "mlp":
        w = 3 * c["hidden"] * c["inter"]
        return {"bytes": 2 * (w + c["hidden"] + 2 * c["tokens"] * c["hidden"]), "flops": 2 * c["tokens"] * w}
    if kind == "qkv":
        n = (c["q_heads"] + 2 * c["kv_heads"]) * c["head_dim"]
        return {"bytes": 2 * (n * c["hidden"] + c["hidden"] + c["tokens"] * (c["hidden"] + n)),
                "flops": 2 * c["tokens"] * n * c["hidden"]}
    if kind == "forward":
        h, qd, kvd = c["hidden"], c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        w = c["layers"] * h * (2 * qd + 2 * kvd + 3 * c["inter"])
        att = c["layers"] * _attention_flops(c["tokens"], c["tokens"], c["q_heads"], c["head_dim"])
        io = c["tokens"] * h * 2 + c["layers"] * 2 * c["tokens"] * kvd  # rows looked up, hidden out, caches
        return {"bytes": 2 * (w + c["vocab"] * h + io) + 4 * c["vocab"],
                "flops": 2 * c["tokens"] * w + att + 2 * c["vocab"] * h}
    if kind == "distill":
        rows = c["blocks"] * 16 * c["kv_heads"]
        return {"bytes": rows * (2 * c["head_dim"] + 16) + 2 * c["dict_heads"] * c["atoms"] * c["head_dim"],
                "flops": 2 * rows * c["atoms"] * c["head_dim"]}
    # weaver and tiered: hot rows (K and V in the cache's own tiers), codes, dictionary, queries and outputs.
    seqs = c["layers"] * c.get("batch", 1)
    hot = seqs * c["hot"] * c["kv_heads"] * c["head_dim"] * 2 * (2 if kind == "tiered" else 1)
    cold = seqs * c["cold"] * c["kv_heads"] * 16
    dic = c["layers"] * c.get("dict_heads", c["kv_heads"]) * c["atoms"] * c["head_dim"] * 2
    rows = seqs * c["queries"] * c["q_heads"]
    refs = seqs * (c["hot"] + c["cold"]) // 16 * 4
    flops = 4 * rows * c["hot"] * c["head_dim"] + rows * c["cold"] * 16 + 4 * rows * c["atoms"] * c["head_dim"]
    return {"bytes": hot + cold + dic + refs + 4 * rows * c["head_dim"], "flops": flops}


def tolerance(case: dict):
    """About four times what the paths were measured to be off from 64 bits."""
    kind = case["kind"]
    if kind == "distill":
        return "exact"  # codes and proxies are defined to the bit
    return {"attention": {"rel": 1e-3}, "mlp": {"rel": 1.5e-3}, "qkv": {"rel": 1.5e-3}, "forward": {"rel": 4e-3},
            "weaver": {"rel": 1e-3}, "tiered": {"rel": 1e-3}}[kind]


# ---------------------------------------------------------------- the same in 64 bits


def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x: torch.Tensor, start: int) -> torch.Tensor:
    t, _, d = x.shape
    freq = THETA ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEVICE) / d)
    angle = (start + torch.arange(t, dtype=torch.float64, device=DEVICE))[:, None, None] * freq
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], -1)


def _attention64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, kv_len: int) -> torch.Tensor:
    """q [n][q_heads][d], k and v [kv_len][kv_heads][d]; query i sees kv_len - n + 1 + i positions."""
    n, q_heads, d = q.shape
    group = q_heads // k.shape[1]
    hidden = torch.arange(kv_len, device=DEVICE)[None, :] > (kv_len - n + torch.arange(n, device=DEVICE))[:, None]
    out = torch.empty_like(q)
    for h in range(q_heads):
        s = (q[:, h] @ k[:, h // group].T) / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, h // group]
    return out


def _mlp64(x: torch.Tensor, w: dict) -> torch.Tensor:
    y = _norm64(x, w["ln2"])
    gate = y @ w["wg"].double().T
    return x + (gate * torch.sigmoid(gate) * (y @ w["wu"].double().T)) @ w["wd"].double().T


def _qkv64(c: dict, x: torch.Tensor, w: dict, start: int):
    y, t, d = _norm64(x, w["ln1"]), c["tokens"], c["head_dim"]
    q = _rope64((y @ w["wq"].double().T).view(t, c["q_heads"], d), start)
    k = _rope64((y @ w["wk"].double().T).view(t, c["kv_heads"], d), start)
    return q, k, (y @ w["wv"].double().T).view(t, c["kv_heads"], d)


def _code_rows(words: torch.Tensor, dictionary: torch.Tensor) -> torch.Tensor:
    """Rows sum_k c_k D[idx_k] of codes [n][8] in 64 bits."""
    coef = words[:, 4:].contiguous().view(torch.float16).double()
    idx = words[:, :4].long() & 0xFFFF
    return sum(coef[:, j, None] * dictionary[idx[:, j]] for j in range(4))


def _two_tiers64(q, hot_k, hot_v, cold, scale: float, causal: bool) -> torch.Tensor:
    """q [n][group][d] of one kv head over its hot rows and cold rows (keys and values alike)."""
    n = q.shape[0]
    k, v = torch.cat([cold, hot_k]), torch.cat([cold, hot_v])
    s = (q @ k.T) * scale
    if causal:
        seen = k.shape[0] - n + torch.arange(n, device=DEVICE)
        s = s.masked_fill((torch.arange(k.shape[0], device=DEVICE)[None, :] > seen[:, None])[:, None, :], -math.inf)
    return torch.softmax(s, -1) @ v


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    if kind == "attention":
        i = _attention_inputs(c, seed)
        return _attention64(i["q"].double(), i["k"].double()[:c["kv_len"]], i["v"].double()[:c["kv_len"]], c["kv_len"])
    if kind == "mlp":
        i = _mlp_inputs(c, seed)
        return _mlp64(i["x"].double(), i)
    if kind == "qkv":
        i = _qkv_inputs(c, seed)
        q, k, v = _qkv64(c, i["x"].double(), i, c["start"])
        return {"q": q.flatten(1), "k": k.flatten(1), "v": v.flatten(1)}
    if kind == "forward":
        i = _forward_inputs(c, seed)
        x = i["embed"][i["ids"].long()].double()
        for w in i["layers"]:
            q, k, v = _qkv64(c, x, w, 0)
            x = x + _attention64(q, k, v, c["tokens"]).flatten(1) @ w["wo"].double().T
            x = _mlp64(x, w)
        return {"logits": _norm64(x[-1:], i["ln"]) @ i["head"].double().T, "hidden": x}
    if kind == "weaver":
        wl = _weaver_inputs(c, seed)
        g, d, nh = wl.geom, c["head_dim"], c["hot"] // 16
        out = torch.empty(wl.out_shape(), dtype=torch.float64, device=DEVICE)
        for l in range(c["layers"]):
            dic = wl.dictionary[l].double()
            for b in range(c["batch"]):
                refs = wl.refs[0, l, b].long()
                hot = wl.hot_k[l, refs[:nh]].double().flatten(0, 1)
                codes = wl.cold[l, refs[nh:]].flatten(0, 1)
                for h in range(c["kv_heads"]):
                    heads = slice(h * g.gqa, (h + 1) * g.gqa)
                    cold = _code_rows(codes[:, h], dic[h if c["dict_heads"] > 1 else 0])
                    out[l, b, :, heads] = _two_tiers64(wl.q[l, b, :, heads].double(), hot[:, h], hot[:, h], cold,
                                                       g.scale, g.causal)
        return out
    if kind == "distill":
        if not c["entropy"]:
            return {"codes": None}
        hot = _distill_inputs(c, seed)["hot"].double().flatten(1)
        return {"codes": None, "entropy": hot.var(dim=1, correction=0)}
    i = _tiered_inputs(c, seed)
    outs, cold_n = [], c["cold"]
    for l in range(c["layers"]):
        out = torch.empty(i["q"][l].shape, dtype=torch.float64, device=DEVICE)
        k = torch.cat([i["ks"][l], i["k"][l]]).double()
        v = torch.cat([i["vs"][l], i["v"][l]]).double()
        group = c["q_heads"] // c["kv_heads"]
        for h in range(c["kv_heads"]):
            dic = i["dicts"][l, h].double()
            coef, idx = torch.topk(k[:cold_n, h] @ dic.T, 4)  # a code: the four largest products, in f16
            cold = sum(coef[:, j, None].to(torch.float16).double() * dic[idx[:, j]] for j in range(4))
            heads = slice(h * group, (h + 1) * group)
            out[:, heads] = _two_tiers64(i["q"][l][:, heads].double(), k[cold_n:, h], v[cold_n:, h], cold,
                                         c["head_dim"] ** -0.5, True)
        outs.append(out)
    return outs
