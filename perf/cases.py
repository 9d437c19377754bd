"""The workloads this framework's speed is measured on.

Every case is a piece of serving work taken through the public entry points
with what a serving program keeps in hand: the page pool, the CSR page table,
planned wrappers, captured graphs and weights.  Head shapes, vocabularies and
context ranges are those of the model presets (Mistral-7B, Qwen2.5-0.5B / 7B /
72B), of the benchmark's batches and of the tests.

Kinds of case:

  decode   one decode step's attention: ``plan`` outside, then a captured graph
           of one RoPE + append + attention launch per layer
  prefill  the attention of a prefill, eager as the engine runs it: ``plan``,
           then RoPE + append and ``run`` per layer; with ``cached`` tokens the
           prompts continue contexts that are already in the pool
  sample   one batched draw: half of the rows greedy, half temperature + top-p
  dense    the element-wise work between the GEMMs of one layer: residual add
           + RMSNorm and SiLU(gate) * up
  model    a whole decode step of a small model: page-table step with the plan,
           then the captured forward; returns the logits
"""

from __future__ import annotations

import math
import random

import torch

from __graft_entry__ import load_package

load_package()

from minimal_inference_amd.decode import BatchDecodeWithPagedKVCacheWrapper  # noqa: E402
from minimal_inference_amd.dense import add_rms_norm, silu_mul  # noqa: E402
from minimal_inference_amd.kv_cache import DevicePageTable, PagedKVCache  # noqa: E402
from minimal_inference_amd.model import AttentionBackend, Model, ModelConfig  # noqa: E402
from minimal_inference_amd.page import rope_append_paged_kv_cache  # noqa: E402
from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper  # noqa: E402
from minimal_inference_amd.sampling import Sampler  # noqa: E402

PAGE = 16
WORKSPACE = 128 << 20  # what the reference's scheduler allocates for each wrapper
ROPE_THETA = 1_000_000.0
EPS = 1e-6

# Query heads, KV heads, head size: the presets' four, and the wide heads that
# the attention tests cover.
HEADS = [(14, 2, 64), (32, 8, 128), (28, 4, 128), (64, 8, 128), (16, 4, 256)]
# hidden, intermediate of the presets
WIDTHS = [(896, 4864), (4096, 14336), (3584, 18944), (8192, 29568)]
VOCABS = [32768, 151936, 152064]


# ------------------------------------------------------------------ the cases
def _decode(heads, batch, lo, hi, layers, log=False):
    hq, hkv, d = heads
    return {"kind": "decode", "hq": hq, "hkv": hkv, "d": d, "batch": batch, "lo": lo, "hi": hi, "log": log,
            "layers": layers}


def _prefill(heads, batch, lo, hi, layers, cached_lo=0, cached_hi=0, log=False):
    hq, hkv, d = heads
    return {"kind": "prefill", "hq": hq, "hkv": hkv, "d": d, "batch": batch, "lo": lo, "hi": hi, "log": log,
            "cached_lo": cached_lo, "cached_hi": cached_hi, "layers": layers}


def listed():
    return [
        # one stream of a chat on Mistral-7B: all 32 layers of its decode step
        {"name": "decode_one_stream", **_decode((32, 8, 128), 1, 1001, 1001, 32)},
        # the benchmark's headline batch: Mistral-7B, 32 requests, prompts U[128, 1024] and the tokens since
        {"name": "decode_batch_32", **_decode((32, 8, 128), 32, 140, 1050, 4)},
        # Qwen2.5-72B heads, 48 requests, contexts log-uniform [512, 4096]
        {"name": "decode_batch_48_wide", **_decode((64, 8, 128), 48, 512, 4096, 2, log=True)},
        # two long documents up to Qwen2.5-7B's 32,768 positions
        {"name": "decode_long_context", **_decode((28, 4, 128), 2, 16001, 32001, 4)},
        # the shortest prefill: one chat prompt on Qwen2.5-0.5B, all its layers
        {"name": "prefill_short_prompt", **_prefill((14, 2, 64), 1, 203, 203, 24)},
        # one request with a page or two of text, Qwen2.5-7B heads
        {"name": "prefill_one_prompt", **_prefill((28, 4, 128), 1, 1537, 1537, 4)},
        # the benchmark's 32 prompts admitted together, Mistral-7B heads
        {"name": "prefill_batch_32", **_prefill((32, 8, 128), 32, 128, 1024, 1)},
        # eight prompts U[256, 2048] at Qwen2.5-72B's heads
        {"name": "prefill_batch_8_wide", **_prefill((64, 8, 128), 8, 256, 2048, 1)},
        # the next turns of four conversations whose earlier turns are in the pool
        {"name": "prefill_cached_turns", **_prefill((32, 8, 128), 4, 61, 413, 2, 2000, 6000)},
        # the draw of a 48-request step at the Qwen vocabulary
        {"name": "sample_batch_48", "kind": "sample", "batch": 48, "vocab": 152064},
        # the element-wise work of one layer over the rows of the benchmark's 32 prompts
        {"name": "dense_prompt_rows", "kind": "dense", "rows": 18240, "hidden": 4096, "inter": 14336},
        # one decode step of Qwen2.5-0.5B for eight requests
        {"name": "model_decode_step", "kind": "model", "batch": 8, "lo": 40, "hi": 310},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """One more case: any head shape, batch and length of the served range."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "sample", "dense"])
    if kind == "sample":
        return {"kind": "sample", "batch": _log_int(rng, 1, 64), "vocab": rng.choice(VOCABS) - rng.choice([0, 0, 7])}
    if kind == "dense":
        hidden, inter = rng.choice(WIDTHS)
        return {"kind": "dense", "rows": _log_int(rng, 1, min(18240, 18240 * 14336 // inter)), "hidden": hidden,
                "inter": inter}
    heads = rng.choice(HEADS)
    if kind == "decode":
        while True:
            batch = _log_int(rng, 1, 64)
            a, b = sorted((_log_int(rng, 16, 32000), _log_int(rng, 16, 32000)))
            case = _decode(heads, batch, a, b, 1, log=rng.random() < 0.5)
            one = work(case)["bytes"]
            if one <= 3.5e8:
                case["layers"] = max(1, min(24, int(1.2e8 / one)))
                return case
    while True:
        batch = _log_int(rng, 1, 32)
        a, b = sorted((_log_int(rng, 5, 4096), _log_int(rng, 5, 4096)))
        cached = rng.random() < 0.4
        c, e = sorted((_log_int(rng, 16, 12000), _log_int(rng, 16, 12000))) if cached else (0, 0)
        case = _prefill(heads, batch, a, b, 1, c, e, log=rng.random() < 0.5)
        w = work(case)
        if w["flops"] <= 2e11 and w["bytes"] <= 6e8:
            case["layers"] = max(1, min(24, int(3e10 / w["flops"]), int(2e8 / w["bytes"])))
            return case


# ------------------------------------------------------------------ lengths and page tables
def _lengths(n, lo, hi, log, salt):
    """n lengths spread over [lo, hi], evenly or evenly in the logarithm, in a fixed mixed order."""
    at = [(i + 0.5) / n for i in range(n)]
    got = [round(lo * (hi / lo) ** x) if log else round(lo + (hi - lo) * x) for x in at]
    random.Random(1000 * n + salt).shuffle(got)
    return got


def _contexts(case):
    """(tokens already in the pool, new tokens) of each request."""
    n = case["batch"]
    new = _lengths(n, case["lo"], case["hi"], case.get("log", False), 1)
    if case["kind"] != "prefill":
        return [(x - 1, 1) for x in new]
    old = _lengths(n, case["cached_lo"], case["cached_hi"], False, 2) if case["cached_hi"] else [0] * n
    return list(zip(old, new))


def _page_table(ctx, seed, device):
    """CSR arrays of requests whose pages lie scattered over the pool, and the pool's page count."""
    npages = [-(-(a + b) // PAGE) for a, b in ctx]
    total = sum(npages) + 1
    gen = torch.Generator().manual_seed(seed)
    ids = torch.randperm(total - 1, generator=gen).to(torch.int32)  # the last page is the scratch page
    indptr, last = [0], []
    for (a, b), n in zip(ctx, npages):
        indptr.append(indptr[-1] + n)
        last.append(a + b - (n - 1) * PAGE)
    i32 = dict(dtype=torch.int32, device=device)
    return torch.tensor(indptr, **i32), ids.to(device), torch.tensor(last, **i32), total


def _rope_tables(rows, d, device):
    freq = 1.0 / ROPE_THETA ** (torch.arange(0, d, 2, dtype=torch.float64) / d)
    ang = torch.outer(torch.arange(rows, dtype=torch.float64), freq)
    ang = torch.cat([ang, ang], dim=1)
    return ang.cos().to(torch.bfloat16).to(device), ang.sin().to(torch.bfloat16).to(device)


def _attention_inputs(case, seed):
    """Pool contents, fused projection rows, page table and RoPE tables of an attention case."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    ctx = _contexts(case)
    hq, hkv, d, layers = case["hq"], case["hkv"], case["d"], case["layers"]
    indptr, indices, last, pages = _page_table(ctx, seed, dev)
    rows = sum(n for _, n in ctx)
    x = {
        "ctx": ctx, "indptr": indptr, "indices": indices, "last": last,
        "pool": torch.randn(layers, pages, 2, PAGE, hkv, d, device=dev, dtype=torch.bfloat16, generator=gen),
        "qkv": torch.randn(layers, rows, (hq + 2 * hkv) * d, device=dev, dtype=torch.bfloat16, generator=gen),
    }
    x["cos"], x["sin"] = _rope_tables(max(a + b for a, b in ctx), d, dev)
    i32 = dict(dtype=torch.int32, device=dev)
    x["positions"] = torch.cat([torch.arange(a, a + n, **i32) for a, n in ctx])
    x["batch_indices"] = torch.cat([torch.full((n,), b, **i32) for b, (_, n) in enumerate(ctx)])
    qo = [0]
    for _, n in ctx:
        qo.append(qo[-1] + n)
    x["qo_indptr"] = torch.tensor(qo, **i32)
    return x


def _pool_of(case, x):
    layers, pages = x["pool"].shape[:2]
    kv = PagedKVCache(layers, case["hkv"], case["d"], 1, PAGE, PAGE, x["pool"].device, max_num_pages=pages)
    kv.data.copy_(x["pool"])
    return kv


def _captured(body):
    """``body`` as a replayable graph, warmed up on a side stream first."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            body()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = body()
    return graph, got


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "sample": _prepare_sample,
            "dense": _prepare_dense, "model": _prepare_model}[case["kind"]](case, seed)


def _prepare_decode(case, seed):
    x = _attention_inputs(case, seed)
    kv = _pool_of(case, x)
    x.pop("pool")
    dev = x["qkv"].device
    wrapper = BatchDecodeWithPagedKVCacheWrapper(torch.empty(WORKSPACE, dtype=torch.uint8, device=dev), "NHD")
    out = torch.empty(case["layers"], case["batch"], case["hq"], case["d"], dtype=torch.bfloat16, device=dev)
    plan = (x["indptr"], x["indices"], x["last"], case["hq"], case["hkv"], case["d"], PAGE)
    wrapper.plan(*plan)

    def layers():
        for i in range(case["layers"]):
            wrapper.run_rope_append(x["qkv"][i], x["cos"], x["sin"], kv.kv_data[i], out=out[i])

    graph, _ = _captured(layers)
    return {"kind": "decode", "inputs": x, "kv": kv, "wrapper": wrapper, "plan": plan, "graph": graph, "out": out}


def _prepare_prefill(case, seed):
    x = _attention_inputs(case, seed)
    kv = _pool_of(case, x)
    x.pop("pool")
    dev, rows = x["qkv"].device, x["qkv"].shape[1]
    wrapper = BatchPrefillWithPagedKVCacheWrapper(torch.empty(WORKSPACE, dtype=torch.uint8, device=dev), "NHD")
    shape = (case["layers"], rows, case["hq"], case["d"])
    return {"kind": "prefill", "case": case, "inputs": x, "kv": kv, "wrapper": wrapper,
            "q": torch.empty(shape[1:], dtype=torch.bfloat16, device=dev),
            "out": torch.empty(shape, dtype=torch.bfloat16, device=dev)}


def _sample_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    logits = torch.randn(case["batch"], case["vocab"], device="cuda", generator=gen)
    return (logits * 3.0).to(torch.bfloat16)


def _prepare_sample(case, seed):
    n = case["batch"]
    sampler = Sampler(torch.device("cuda"), n, seed=seed, vocab=case["vocab"])
    sampler.set_params([0.0 if i % 2 else 0.7 for i in range(n)], [0.9] * n)
    return {"kind": "sample", "logits": _sample_inputs(case, seed), "sampler": sampler}


def _dense_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, device="cuda", dtype=torch.bfloat16, generator=gen)

    return {"x": randn(case["rows"], case["hidden"]), "delta": randn(case["rows"], case["hidden"]),
            "weight": (1.0 + 0.1 * randn(case["hidden"]).float()).to(torch.bfloat16),
            "gate_up": 2.0 * randn(case["rows"], 2 * case["inter"])}


def _prepare_dense(case, seed):
    x = _dense_inputs(case, seed)
    dev = x["x"].device
    return {"kind": "dense", "inputs": x,
            "h": torch.empty_like(x["x"]),
            "act": torch.empty(case["rows"], case["inter"], dtype=torch.bfloat16, device=dev)}


def _model_inputs(case, seed):
    """Weights of the small preset, the contexts already in the pool, and the step's ids."""
    cfg = ModelConfig()
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def randn(*shape, std=0.02):
        return torch.randn(*shape, device=dev, dtype=torch.bfloat16, generator=gen) * std

    nq, nkv, d, h = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.hidden_size
    layers = [{"in_norm": 1 + randn(h, std=0.1), "post_norm": 1 + randn(h, std=0.1),
               "w_qkv": randn((nq + 2 * nkv) * d, h), "b_qkv": randn((nq + 2 * nkv) * d),
               "w_o": randn(h, nq * d), "w_gate_up": randn(2 * cfg.intermediate_size, h),
               "w_down": randn(h, cfg.intermediate_size)} for _ in range(cfg.num_hidden_layers)]
    ctx = [n for n, _ in _contexts(case)]
    npages = [n // PAGE + 1 for n in ctx]
    pages = sum(npages) + 1
    return cfg, {
        "layers": layers, "embed": randn(cfg.vocab_size, h), "norm": 1 + randn(h, std=0.1), "ctx": ctx,
        "npages": npages, "pages": pages,
        "pool": torch.randn(cfg.num_hidden_layers, pages, 2, PAGE, nkv, d, device=dev, dtype=torch.bfloat16,
                            generator=gen),
        "ids": torch.randint(0, cfg.vocab_size, (case["batch"],), device=dev, generator=gen),
        "rope": _rope_tables(max(ctx) + 1, d, dev),
    }


def _prepare_model(case, seed):
    cfg, x = _model_inputs(case, seed)
    dev, n = x["ids"].device, case["batch"]
    model = Model(cfg, dev, max_positions=max(x["ctx"]) + 1)
    for layer, given in zip(model.layers, x["layers"]):
        for name, w in given.items():
            setattr(layer, name, w)
    model.embed = model.lm_head = x["embed"]
    model.norm = x["norm"]
    model.cos, model.sin = x["rope"]
    kv = PagedKVCache(cfg.num_hidden_layers, cfg.num_key_value_heads, cfg.head_dim, n, max(x["ctx"]) + PAGE, PAGE, dev,
                      max_num_pages=x["pages"])
    kv.data.copy_(x["pool"])
    table = DevicePageTable(x["pages"], n, max(x["npages"]) + 1, PAGE, dev)
    i32 = dict(dtype=torch.int32, device=dev)
    csr = [torch.zeros(n + 1, **i32), torch.zeros(x["pages"] + n, **i32), torch.ones(n, **i32), torch.zeros(n, **i32),
           torch.zeros(n, **i32)]
    wrapper = BatchDecodeWithPagedKVCacheWrapper(torch.empty(WORKSPACE, dtype=torch.uint8, device=dev), "NHD")
    rows = [(i, pos) for i, pos in enumerate(x["ctx"])]
    plan = (wrapper, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim)
    table.step([(i, p) for i, p in enumerate(x["npages"])], rows, n, *csr, decode_plan=plan)
    backend = AttentionBackend(kv, wrapper, "decode", csr[0], csr[1], csr[2], None, csr[3], csr[4])
    graph, logits = _captured(lambda: model.forward(x["ids"], csr[4], backend))
    return {"kind": "model", "model": model, "kv": kv, "table": table, "csr": csr, "rows": rows, "plan": plan,
            "graph": graph, "logits": logits, "ids": x["ids"], "backend": backend}


# ------------------------------------------------------------------ run
def run(state):
    kind = state["kind"]
    if kind == "decode":
        state["wrapper"].plan(*state["plan"])
        state["graph"].replay()
        return {"out": state["out"], "pool": state["kv"].data}
    if kind == "prefill":
        c, x, kv, out = state["case"], state["inputs"], state["kv"], state["out"]
        csr = (x["indices"], x["indptr"], x["last"])
        wrapper = state["wrapper"]
        wrapper.plan(x["qo_indptr"], x["indptr"], x["indices"], x["last"], c["hq"], c["hkv"], c["d"], PAGE,
                     causal=True, max_total_q=x["qkv"].shape[1])
        for i in range(c["layers"]):
            q = rope_append_paged_kv_cache(x["qkv"][i], c["hq"], c["hkv"], x["positions"], x["cos"], x["sin"],
                                           x["batch_indices"], x["positions"], kv.kv_data[i], *csr, q_out=state["q"])
            wrapper.run(q, kv.kv_data[i], out=out[i])
        return {"out": out, "pool": kv.data}
    if kind == "sample":
        state["sampler"].rng_offset.zero_()  # a reproducible draw: the same ids for the same logits
        return state["sampler"].sample(state["logits"])
    if kind == "dense":
        x = state["inputs"]
        h = add_rms_norm(x["x"], x["delta"], x["weight"], EPS, write_x=False, h_out=state["h"])
        return {"norm": h, "act": silu_mul(x["gate_up"], out=state["act"])}
    state["table"].step([], state["rows"], len(state["rows"]), *state["csr"], decode_plan=state["plan"])
    state["graph"].replay()
    return {"logits": state["logits"], "pool": state["kv"].data}


# ------------------------------------------------------------------ work
def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": case["batch"] * (2 * case["vocab"] + 16), "flops": 0}
    if kind == "dense":
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 6 * rows * (hidden + inter) + 2 * hidden, "flops": 0}
    if kind == "model":
        cfg = ModelConfig()
        hq, hkv, d, layers = (cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.num_hidden_layers)
        per_layer = cfg.hidden_size * ((2 * hq + 2 * hkv) * d + 3 * cfg.intermediate_size)
        params = layers * per_layer + cfg.vocab_size * cfg.hidden_size
        kv = sum(a + b for a, b in _contexts(case))
        return {"bytes": 2 * params + layers * kv * 4 * hkv * d + 2 * case["batch"] * cfg.vocab_size,
                "flops": 2 * case["batch"] * params + layers * 4 * hq * d * kv}
    ctx = _contexts(case)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    new = sum(n for _, n in ctx)
    read = 2 * new * (hq + 2 * hkv) * d + 4 * hkv * d * sum(a for a, _ in ctx) + 4 * new * d
    write = 2 * new * hq * d + 4 * new * hkv * d
    pairs = sum(a * n + n * (n + 1) // 2 for a, n in ctx)
    return {"bytes": case["layers"] * (read + write), "flops": case["layers"] * 4 * hq * d * pairs}


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    """Relative errors that the data types give, about four times what the start showed against ``exact``."""
    return {
        # bf16 RoPE and probabilities, a bf16 output
        "decode": {"rel": 1.5e-2},
        "prefill": {"rel": 1.3e-2},
        # ids: the same logits and counters give the same draw
        "sample": "exact",
        # one or two bf16 roundings of a 32-bit result
        "dense": {"rel": 1e-2},
        # bf16 activations through 24 layers
        "model": {"rel": 0.12},
    }[case["kind"]]


# ------------------------------------------------------------------ exact
def _rotate(x, cos, sin):
    """Rotate-half RoPE; x [T, H, D], cos / sin [T, D]."""
    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos.unsqueeze(1) + turned * sin.unsqueeze(1)


def _attend(q, k, v, old):
    """Softmax attention of rows q [N, Hq, D] at positions old .. old + N - 1 over k, v [old + N, Hkv, D]."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    group = hq // hkv
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[0], device=q.device)[None, :] <= old + torch.arange(n, device=q.device)[:, None]
    for h in range(hkv):
        qh = q[:, h * group:(h + 1) * group].transpose(0, 1)  # [group, N, D]
        s = torch.matmul(qh, k[:, h].t()) / math.sqrt(d)
        p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
        out[:, h * group:(h + 1) * group] = torch.matmul(p, v[:, h].contiguous()).transpose(0, 1)
    return out


def _exact_attention(case, seed):
    x = _attention_inputs(case, seed)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    pos = x["positions"].long()
    cos, sin = x["cos"].double()[pos], x["sin"].double()[pos]
    out = torch.empty(case["layers"], x["qkv"].shape[1], hq, d, dtype=torch.float64, device=pos.device)
    pool = x.pop("pool").double()
    first = x["indptr"].long()[x["batch_indices"].long()]
    page, slot = x["indices"].long()[first + pos // PAGE], pos % PAGE
    indptr, indices = x["indptr"].tolist(), x["indices"].long()
    for i in range(case["layers"]):
        rows = x["qkv"][i].double().view(-1, hq + 2 * hkv, d)
        q, k = _rotate(rows[:, :hq], cos, sin), _rotate(rows[:, hq:hq + hkv], cos, sin)
        pool[i][page, 0, slot] = k
        pool[i][page, 1, slot] = rows[:, hq + hkv:]
        at = 0
        for b, (old, new) in enumerate(x["ctx"]):
            kv = pool[i][indices[indptr[b]:indptr[b + 1]]]  # [pages, 2, 16, Hkv, D]
            kk = kv[:, 0].reshape(-1, hkv, d)[:old + new]
            vv = kv[:, 1].reshape(-1, hkv, d)[:old + new]
            out[i, at:at + new] = _attend(q[at:at + new], kk, vv, old)
            at += new
    return {"out": out, "pool": pool}


def _exact_model(case, seed):
    cfg, x = _model_inputs(case, seed)
    hq, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    pos = torch.tensor(x["ctx"], device=x["ids"].device)
    cos, sin = x["rope"][0].double()[pos], x["rope"][1].double()[pos]
    pool = x["pool"].double()
    first = [sum(x["npages"][:b]) for b in range(case["batch"])]  # pages are handed out in order

    def norm(y, w):
        return y * torch.rsqrt(y.square().mean(-1, keepdim=True) + cfg.rms_norm_eps) * w.double()

    h = x["embed"].double()[x["ids"]]
    for i, w in enumerate(x["layers"]):
        rows = norm(h, w["in_norm"]) @ w["w_qkv"].double().t() + w["b_qkv"].double()
        rows = rows.view(-1, hq + 2 * hkv, d)
        q, k = _rotate(rows[:, :hq], cos, sin), _rotate(rows[:, hq:hq + hkv], cos, sin)
        o = torch.empty_like(q)
        for b, old in enumerate(x["ctx"]):
            pages = slice(first[b], first[b] + x["npages"][b])
            pool[i][first[b] + old // PAGE, 0, old % PAGE] = k[b]
            pool[i][first[b] + old // PAGE, 1, old % PAGE] = rows[b, hq + hkv:]
            kk = pool[i][pages, 0].reshape(-1, hkv, d)[:old + 1]
            vv = pool[i][pages, 1].reshape(-1, hkv, d)[:old + 1]
            o[b:b + 1] = _attend(q[b:b + 1], kk, vv, old)
        h = h + o.reshape(case["batch"], -1) @ w["w_o"].double().t()
        gate, up = (norm(h, w["post_norm"]) @ w["w_gate_up"].double().t()).chunk(2, dim=-1)
        h = h + (gate * torch.sigmoid(gate) * up) @ w["w_down"].double().t()
    return {"logits": norm(h, x["norm"]) @ x["embed"].double().t(), "pool": pool}


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # ids of a pseudo-random draw: no computed number
    if kind == "dense":
        x = _dense_inputs(case, seed)
        y = x["x"].double() + x["delta"].double()
        h = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * x["weight"].double()
        gate, up = x["gate_up"].double().chunk(2, dim=-1)
        return {"norm": h, "act": gate * torch.sigmoid(gate) * up}
    return _exact_model(case, seed) if kind == "model" else _exact_attention(case, seed)
