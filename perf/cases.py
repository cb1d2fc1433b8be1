"""The work whose speed is measured: what a program that serves a model through this
package has it do, over the range of sizes, types and directions such programs meet.

Three kinds of case:

* ``step``: one engine step's paged attention (append + attention) of ``layers``
  layers of one geometry, through ``PagedKVCache.append_attention``, with the step's
  metadata built beforehand as the engine builds it once per step. ``prompts``
  sequences bring ``new`` prompt tokens each after ``prefix`` tokens already cached
  (a prefix-cache hit; 0: a fresh prompt); ``decodes`` sequences bring one token
  after ``cached`` tokens. ``graph``: the layers' launches are captured in a HIP graph
  beforehand and replayed, as the engine and the benchmark run decode steps; otherwise
  they are issued one by one, as the engine runs steps with prompts.
* ``copy``: a compaction round, ``PagedKVCache.copy_blocks`` over all layers.
* ``model``: a whole forward pass of the 0.5B-dimension model: ``prompts`` through
  ``Qwen2Paged.forward``, or ``decodes`` rows as a captured pass over the layers and the
  LM head's logits.

Lengths are drawn from the case alone (``lengths`` seeds them), so that a case is the
same work for every seed of its inputs.
"""
from __future__ import annotations

import math
import random

import torch

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
# query heads, kv heads, head dim
GEOMETRY = {"qwen": (14, 2, 64), "llama": (32, 8, 128)}
MODEL = dict(n_layers=24, n_heads=14, n_kv_heads=2, d_model=896, head_dim=64, d_ff=4864, vocab_size=151936,
             rms_eps=1e-6, rope_theta=1e6, max_position=32768)


def _step(name, geometry, dtype, layers, *, prompts=0, new="1:1", prefix="0:0", decodes=0, cached="1:1",
          rope=True, graph=False, block=16, lengths=1):
    return {"name": name, "kind": "step", "geometry": geometry, "dtype": dtype, "layers": layers, "prompts": prompts,
            "new": new, "prefix": prefix, "decodes": decodes, "cached": cached, "rope": rope, "graph": graph,
            "block": block, "lengths": lengths}


def listed():
    return [
        # the smallest step: the fp32 parity configuration, eight short sequences
        _step("decode fp32 8 short", "qwen", "float32", 24, decodes=8, cached="16:256", rope=False, graph=True),
        # the engine's serving decode: 32 running requests some way into their answers
        _step("decode bf16 32 serving", "qwen", "bfloat16", 24, decodes=32, cached="58:770", graph=True, lengths=2),
        # the benchmark's headline decode step
        _step("decode fp16 64 headline", "qwen", "float16", 8, decodes=64, cached="512:4096", rope=False, graph=True,
              lengths=3),
        # a large batch of long contexts at the 8B geometry: the largest case
        _step("decode bf16 256 long", "llama", "bfloat16", 1, decodes=256, cached="lognormal:8192:0.5:1024:32768",
              rope=False, graph=True, lengths=4),
        # fresh prompts of all lengths up to the engine's longest (max_model_len 4096)
        _step("prompts bf16 to 4096", "qwen", "bfloat16", 2, prompts=4, new="700:4095", lengths=5),
        # fresh prompts at the 8B geometry, some long
        _step("prompts bf16 8B", "llama", "bfloat16", 1, prompts=3, new="600:8192", lengths=6),
        # prompts that hit the prefix cache: a cached system prompt or conversation, a new turn after it
        _step("prefix hits fp16", "qwen", "float16", 4, prompts=12, new="16:400", prefix="600:3600", lengths=7),
        # one mixed step: eight new prompts beside 56 running requests
        _step("mixed bf16 8 + 56", "qwen", "bfloat16", 8, prompts=8, new="512:512", decodes=56, cached="256:2048",
              graph=True, lengths=8),
        # the reference's precision: short and medium prompts in fp32
        _step("prompts fp32", "qwen", "float32", 2, prompts=6, new="60:700", lengths=9),
        # compaction after evictions: 1024 blocks moved in each of 24 layers
        {"name": "compaction 1024", "kind": "copy", "geometry": "qwen", "dtype": "bfloat16", "layers": 24,
         "blocks": 8192, "pairs": 1024, "block": 16},
        # a whole decode pass of 32 requests
        {"name": "model decode 32", "kind": "model", "prompts": 0, "new": "1:1", "decodes": 32, "cached": "58:770",
         "lengths": 11},
        # a whole pass over the prompts of one step (the engine's budget of 2048 tokens)
        {"name": "model prompts 2048", "kind": "model", "prompts": 5, "new": "300:509", "decodes": 0, "cached": "1:1",
         "lengths": 12},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """A case of the ranges above: decode batches, prompts, prefix hits, mixed steps,
    copies and model passes of other sizes, each no more work than the largest above."""
    lengths = rng.randrange(1, 1 << 20)
    kind = rng.choice(["decode", "decode", "prompts", "prompts", "hits", "mixed", "fp32", "copy", "model"])
    if kind == "decode":
        g = rng.choice(["qwen", "llama"])
        dt = rng.choice(["float16", "bfloat16", "bfloat16"])
        n = _log_int(rng, 1, 256)
        hi = _log_int(rng, 64, 8192 if n <= 128 else 4096)
        lo = max(1, hi // rng.randint(2, 16))
        per = n * hi * (512 if g == "qwen" else 4096)
        c = _step("", g, dt, max(1, min(24, (1 << 30) // per)), decodes=n, cached=f"{lo}:{hi}",
                  rope=rng.random() < 0.5, graph=True, block=rng.choice([16, 16, 32]), lengths=lengths)
    elif kind == "prompts":
        g = rng.choice(["qwen", "llama"])
        hi = _log_int(rng, 24, 4096)
        n = rng.randint(1, max(1, min(8, 10000 // hi)))
        c = _step("", g, rng.choice(["float16", "bfloat16"]), 2, prompts=n, new=f"{max(16, hi // 3)}:{hi}",
                  block=rng.choice([16, 16, 32]), lengths=lengths)
    elif kind == "hits":
        hi = _log_int(rng, 20, 600)
        c = _step("", rng.choice(["qwen", "llama"]), rng.choice(["float16", "bfloat16"]), 2, prompts=rng.randint(1, 16),
                  new=f"{max(1, hi // 8)}:{hi}", prefix=f"64:{_log_int(rng, 100, 3600)}", lengths=lengths)
    elif kind == "mixed":
        hi = _log_int(rng, 32, 2000)
        c = _step("", "qwen", rng.choice(["float16", "bfloat16"]), 4, prompts=rng.randint(1, 8),
                  new=f"{max(16, hi // 2)}:{hi}", decodes=rng.randint(1, 64), cached="58:2048",
                  graph=rng.random() < 0.5, lengths=lengths)
    elif kind == "fp32":
        hi = _log_int(rng, 20, 700)
        c = _step("", "qwen", "float32", 2, prompts=rng.randint(0, 6), new=f"{max(2, hi // 6)}:{hi}",
                  decodes=rng.randint(1, 16), cached="16:900", lengths=lengths)
    elif kind == "copy":
        c = {"kind": "copy", "geometry": "qwen", "dtype": rng.choice(["bfloat16", "float32"]),
             "layers": rng.randint(2, 24), "blocks": 4096, "pairs": _log_int(rng, 3, 1500), "block": 16}
    else:
        c = {"kind": "model", "prompts": rng.randint(1, 6), "new": "20:330", "decodes": rng.randint(0, 16),
             "cached": "20:700", "lengths": lengths}
    c.pop("name", None)
    return c


# ---- what a case's sizes come to ------------------------------------------------
def _draws(rng, spec, n):
    if spec.startswith("lognormal:"):
        median, sigma, lo, hi = (float(x) for x in spec.split(":")[1:])
        return [int(min(hi, max(lo, round(median * math.exp(sigma * rng.gauss(0, 1)))))) for _ in range(n)]
    lo, hi = (int(x) for x in spec.split(":"))
    return [rng.randint(lo, hi) for _ in range(n)]


def _sequences(case):
    """(cached, new) of every sequence of the step, prompts first (the engine's order)."""
    rng = random.Random(case["lengths"])
    new = _draws(rng, case["new"], case["prompts"])
    prefix = _draws(rng, case.get("prefix", "0:0"), case["prompts"])
    # prefix hits are whole blocks
    seqs = [(p // 16 * 16, n) for p, n in zip(prefix, new)]
    return seqs + [(c, 1) for c in _draws(rng, case["cached"], case["decodes"])]


def _geometry(case):
    return GEOMETRY[case["geometry"]] if "geometry" in case else (MODEL["n_heads"], MODEL["n_kv_heads"],
                                                                  MODEL["head_dim"])


def work(case):
    hq, hkv, d = _geometry(case)
    if case["kind"] == "copy":
        block = 2 * hkv * case["block"] * d * DTYPES[case["dtype"]].itemsize
        return {"bytes": 2 * case["pairs"] * block * case["layers"], "flops": 0}
    seqs = _sequences(case)
    rows = sum(n for _, n in seqs)
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in seqs)
    if case["kind"] == "model":
        b, layers = 2, MODEL["n_layers"]
        dm, ff = MODEL["d_model"], MODEL["d_ff"]
        per_layer = dm * (hq + 2 * hkv) * d + hq * d * dm + 3 * dm * ff
        head = MODEL["vocab_size"] * dm
        weights = b * (layers * per_layer + head)
        extra = 2 * rows * layers * per_layer + 2 * len(seqs) * head
        out = 4 * len(seqs) * MODEL["vocab_size"]
        kv = sum((c + 2 * n) * 2 * hkv * d * b for c, n in seqs)
        kv -= sum(n * 2 * hkv * d * b for _, n in seqs)   # the new rows are made and stored, not read
        return {"bytes": weights + layers * kv + out, "flops": extra + layers * 4 * hq * d * pairs}
    b = DTYPES[case["dtype"]].itemsize
    # per sequence: the cached rows read, the new rows read and stored; q and the outputs
    kv = sum((c + 2 * n) * 2 * hkv * d * b for c, n in seqs)
    return {"bytes": case["layers"] * (kv + 2 * rows * hq * d * b), "flops": case["layers"] * 4 * hq * d * pairs}


def tolerance(case):
    # About four times the distance of each path from its 64-bit results. One layer (measured
    # 1.5e-7 in fp32, 3.6e-4 in fp16, 2.6e-3 in bf16): the rounding of the outputs, of the
    # probabilities and, with RoPE, of the rotated keys. The whole model (measured 0.034): those
    # of 24 layers, each carried through all that follow.
    if case["kind"] == "copy":
        return "exact"
    if case["kind"] == "model":
        return {"rel": 0.13, "max": 0.7}
    return {"float32": {"rel": 1e-6, "max": 2e-5}, "float16": {"rel": 1.5e-3, "max": 1e-2},
            "bfloat16": {"rel": 1.1e-2, "max": 8e-2}}[case["dtype"]]


# ---- inputs (the same for prepare and exact) ---------------------------------------
def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _rope_tables(d):
    half = 1.0 / (MODEL["rope_theta"] ** (torch.arange(0, d, 2, device=_dev()).float() / d))
    angle = torch.arange(MODEL["max_position"], device=_dev()).float()[:, None] * half[None, :]
    return angle.cos(), angle.sin()


def _tables(seqs, block, seed):
    """Block tables over a shuffled pool, and the pool's size (1 in 16 of it unused)."""
    need = [-(-(c + n) // block) for c, n in seqs]
    total = sum(need)
    total += total // 16 + 1
    ids = list(range(total))
    random.Random(seed).shuffle(ids)
    tables, at = [], 0
    for k in need:
        tables.append(ids[at:at + k])
        at += k
    return tables, total


def _rows(seqs):
    slices, positions, at = [], [], 0
    for c, n in seqs:
        slices.append((at, at + n))
        positions.extend(range(c, c + n))
        at += n
    return slices, positions


def _step_inputs(case, seed, storage):
    """q, k, v [layers, rows, heads, d], and the pools' contents into ``storage``."""
    g = _generator(seed)
    hq, hkv, d = _geometry(case)
    rows = sum(n for _, n in _sequences(case))
    dt, dev = DTYPES[case["dtype"]], _dev()
    q, k, v = (torch.randn(case["layers"], rows, h, d, generator=g, device=dev).to(dt) for h in (hq, hkv, hkv))
    if case.get("prefix", "0:0") != "0:0" or case["decodes"]:
        for layer in storage:
            layer.normal_(generator=g)
    return q, k, v


def _step_shape(case, seed):
    hq, hkv, d = _geometry(case)
    tables, blocks = _tables(_sequences(case), case["block"], seed)
    return tables, (case["layers"], blocks, 2, hkv, case["block"], d)


_STREAM = {}


def _capture(run):
    """The launches of ``run()`` as a HIP graph, captured on one stream kept for it."""
    s = _STREAM.setdefault(torch.cuda.current_device(), None) or torch.cuda.Stream()
    _STREAM[torch.cuda.current_device()] = s
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run()
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        run()
    return graph


def _step_meta(cache, positions, host_positions, slices, tables, ctx, hq):
    cache.step_metadata(positions, slices, tables, ctx, rows_per_item=cache.rows_per_item(hq),
                        host_positions=host_positions, num_heads=hq)


def prepare(case, seed):
    from tinybatch_amd import PagedKVCache
    from tinybatch_amd.ops import Rope

    dev = _dev()
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    if case["kind"] == "copy":
        hq, hkv, d = _geometry(case)
        cache = PagedKVCache(case["layers"], case["blocks"], case["block"], hkv, d, dev, DTYPES[case["dtype"]])
        _copy_fill(case, seed, cache.storage)
        src, dst = _copy_ids(case, seed)
        return {"case": case, "cache": cache, "src": src, "dst": dst}
    hq, hkv, d = _geometry(case)
    seqs = _sequences(case)
    tables, shape = _step_shape(case, seed)
    cache = PagedKVCache(case["layers"], shape[1], case["block"], hkv, d, dev, DTYPES[case["dtype"]])
    q, k, v = _step_inputs(case, seed, cache.storage)
    slices, host_positions = _rows(seqs)
    ctx = [c + n for c, n in seqs]
    positions = torch.tensor(host_positions, dtype=torch.int64, device=dev)
    _step_meta(cache, positions, host_positions, slices, tables, ctx, hq)
    out = torch.empty(case["layers"], len(host_positions), hq * d, device=dev, dtype=q.dtype)
    rope = Rope(*_rope_tables(d)) if case["rope"] else None

    def layers():
        for i in range(case["layers"]):
            cache.append_attention(i, q[i], k[i], v[i], positions, slices, tables, ctx, num_heads=hq, out=out[i],
                                   rope=rope)

    state = {"case": case, "cache": cache, "layers": layers, "out": out, "graph": None}
    if case["graph"]:
        state["graph"] = _capture(layers)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "copy":
        state["cache"].copy_blocks(state["src"], state["dst"])
        return state["cache"].storage
    if case["kind"] == "model":
        return _run_model(state)
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        state["layers"]()
    return {"out": state["out"], "pool": state["cache"].storage}


# ---- compaction ----------------------------------------------------------------------
def _copy_fill(case, seed, storage):
    g = _generator(seed)
    for layer in storage:
        layer.normal_(generator=g)


def _copy_ids(case, seed):
    ids = random.Random(seed).sample(range(case["blocks"]), 2 * case["pairs"])
    return ids[:case["pairs"]], ids[case["pairs"]:]


# ---- the whole model -------------------------------------------------------------------
def _model_inputs(case, seed):
    seqs = _sequences(case)
    tables, blocks = _tables(seqs, 16, seed)
    g = _generator(seed + 1)
    tokens = torch.randint(0, MODEL["vocab_size"], (sum(n for _, n in seqs),), generator=g, device=_dev())
    return seqs, tables, blocks, tokens, g


def _model_pool(case, storage, g):
    """K/V of the cached positions, with the keys' and values' scale in this model."""
    if case["decodes"]:
        for layer in storage:
            layer.normal_(0.0, 0.6, generator=g)


def _prepare_model(case, seed):
    from tinybatch_amd import PagedKVCache
    from tinybatch_amd.model import ModelConfig, Qwen2Paged

    dev = _dev()
    cfg = ModelConfig(tie_embeddings=True, **MODEL)
    model = Qwen2Paged(cfg, dev, torch.bfloat16, seed=seed)
    seqs, tables, blocks, tokens, g = _model_inputs(case, seed)
    cache = PagedKVCache(cfg.n_layers, blocks, 16, cfg.n_kv_heads, cfg.head_dim, dev, torch.bfloat16)
    _model_pool(case, cache.storage, g)
    slices, host_positions = _rows(seqs)
    ctx = [c + n for c, n in seqs]
    positions = torch.tensor(host_positions, dtype=torch.int64, device=dev)
    _step_meta(cache, positions, host_positions, slices, tables, ctx, cfg.n_heads)
    state = {"case": case, "model": model, "cache": cache, "graph": None,
             "args": (tokens, positions, slices, tables, ctx, cache)}
    if not case["prompts"]:
        def attention(i, q, k, v):
            return cache.append_attention(i, q, k, v, positions, slices, tables, ctx, rope=model.rope)

        def layers():
            state["hidden"] = model.run_layers(tokens, positions, attention, fused_rope=True)

        with torch.inference_mode():
            state["graph"] = _capture(layers)
    return state


def _run_model(state):
    model = state["model"]
    if state["graph"] is None:
        logits = model.forward(*state["args"])
    else:
        state["graph"].replay()
        with torch.inference_mode():
            logits = torch.nn.functional.linear(state["hidden"], model.lm_head).float()
    return {"logits": logits, "pool": state["cache"].storage}


# ---- 64-bit results ----------------------------------------------------------------------
def _rotate(x, cos, sin):
    """Rotate-half RoPE of x [rows, heads, d] with cos / sin [rows, d / 2]."""
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend(q, k, v, pool, seqs, tables, block):
    """Appends k, v [rows, hkv, d] to the 64-bit or native ``pool`` [blocks, 2, hkv, block, d]
    and returns the attention rows [rows, hq * d]; everything computed in 64 bits."""
    hq, d = q.shape[1], q.shape[2]
    hkv = k.shape[1]
    rep = hq // hkv
    out = torch.empty(q.shape[0], hq, d, dtype=torch.float64, device=q.device)
    at = 0
    for (c, n), table in zip(seqs, tables):
        t = torch.tensor(table, device=q.device)
        pos = torch.arange(c, c + n, device=q.device)
        keys = pool[t].permute(1, 2, 0, 3, 4).reshape(2, hkv, -1, d)[:, :, :c + n].double()
        keys[0, :, c:] = k[at:at + n].transpose(0, 1)
        keys[1, :, c:] = v[at:at + n].transpose(0, 1)
        pool[t[pos // block], 0, :, pos % block] = k[at:at + n].to(pool.dtype)
        pool[t[pos // block], 1, :, pos % block] = v[at:at + n].to(pool.dtype)
        hidden = torch.arange(c + n, device=q.device)[None, :] > pos[:, None]
        for h in range(hkv):
            qh = q[at:at + n, h * rep:(h + 1) * rep].reshape(n * rep, d)
            s = (qh @ keys[0, h].T / math.sqrt(d)).reshape(n, rep, c + n)
            s.masked_fill_(hidden[:, None, :], -math.inf)
            p = torch.softmax(s, dim=-1)
            out[at:at + n, h * rep:(h + 1) * rep] = (p.reshape(n * rep, c + n) @ keys[1, h]).reshape(n, rep, d)
        at += n
    return out.reshape(q.shape[0], hq * d)


@torch.no_grad()
def exact(case, seed):
    dev = _dev()
    if case["kind"] == "model":
        return _exact_model(case, seed)
    if case["kind"] == "copy":
        hq, hkv, d = _geometry(case)
        storage = torch.empty(case["layers"], case["blocks"], 2, hkv, case["block"], d, device=dev,
                              dtype=DTYPES[case["dtype"]])
        _copy_fill(case, seed, storage)
        src, dst = _copy_ids(case, seed)
        storage[:, dst] = storage[:, src]
        return storage
    seqs = _sequences(case)
    tables, shape = _step_shape(case, seed)
    storage = torch.zeros(shape, device=dev, dtype=DTYPES[case["dtype"]])
    q, k, v = _step_inputs(case, seed, storage)
    q, k, v = q.double(), k.double(), v.double()
    if case["rope"]:
        pos = torch.tensor(_rows(seqs)[1], device=dev)
        cos, sin = (x[pos].double() for x in _rope_tables(shape[-1]))
        q = torch.stack([_rotate(x, cos, sin) for x in q])
        k = torch.stack([_rotate(x, cos, sin) for x in k])
    small = storage.numel() * storage.element_size() < 1 << 30
    pools = storage.double() if small else storage
    out = torch.stack([_attend(q[i], k[i], v[i], pools[i], seqs, tables, case["block"])
                       for i in range(case["layers"])])
    return {"out": out, "pool": pools if small else None}


def _exact_model(case, seed):
    dev, m = _dev(), MODEL
    hq, hkv, d, dm, ff = m["n_heads"], m["n_kv_heads"], m["head_dim"], m["d_model"], m["d_ff"]
    gw = _generator(seed)

    def rnd(*shape):
        return (torch.randn(*shape, generator=gw, device=dev, dtype=torch.float32) * 0.02).to(torch.bfloat16)

    def norm(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + m["rms_eps"])

    embed = rnd(m["vocab_size"], dm)
    seqs, tables, blocks, tokens, g = _model_inputs(case, seed)
    storage = torch.zeros(m["n_layers"], blocks, 2, hkv, 16, d, device=dev, dtype=torch.bfloat16)
    _model_pool(case, storage, g)
    pools = storage.double()
    slices, positions = _rows(seqs)
    cos, sin = (x[torch.tensor(positions, device=dev)].double() for x in _rope_tables(d))
    h = embed[tokens].double()
    rows = h.shape[0]
    for i in range(m["n_layers"]):
        w_qkv, b_qkv = rnd((hq + 2 * hkv) * d, dm), rnd((hq + 2 * hkv) * d)
        w_o, w_gu, w_down = rnd(dm, hq * d), rnd(2 * ff, dm), rnd(dm, ff)
        qkv = norm(h) @ w_qkv.double().T + b_qkv.double()
        q = _rotate(qkv[:, :hq * d].reshape(rows, hq, d), cos, sin)
        k = _rotate(qkv[:, hq * d:(hq + hkv) * d].reshape(rows, hkv, d), cos, sin)
        v = qkv[:, (hq + hkv) * d:].reshape(rows, hkv, d)
        h = h + _attend(q, k, v, pools[i], seqs, tables, 16) @ w_o.double().T
        gate, up = (norm(h) @ w_gu.double().T).split(ff, dim=-1)
        h = h + (torch.nn.functional.silu(gate) * up) @ w_down.double().T
    last = torch.tensor([e - 1 for _, e in slices], device=dev)
    return {"logits": norm(h)[last] @ embed.double().T, "pool": pools}
