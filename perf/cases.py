"""Workloads that the performance of this package is judged by.

Each case is one pass through the package's public entry points as a prefill
program calls them.  The forms of a call (``api``):

* ``attention``  ``ops.optimized_attention``: the validated, allocating call of a
  model's attention layer (mode ``query`` or ``unfused``);
* ``launch``     ``ops.launch_attention`` on buffers that the program keeps (mode
  ``query``), which is what the headline benchmark times;
* ``fused`` / ``separate``  the older API with the model's own attention scale;
* ``factored``   ``ops.launch_factored_attention`` on kept buffers (no RoPE);
* ``norm_rope``  ``ops.norm_rope``: Q/K RMSNorm + RoPE alone.

``layers`` > 0 means that the program has captured the calls of that many
layers into one HIP graph, as a server does with short prefills, and replays
it; 0 means one eager call.  Geometries are those of ``ops.MODELS``; inputs are
N(0,1) activations, gamma = 1 + 0.1 N(0,1) and theta = 1e6, as in the package's
benchmark.  The path is forward only and bf16 only.
"""
import math

import torch

from kernelfuser_amd import ops

EPS = 1e-6
THETA = 1e6


def _case(name, api, model, b, s, *, causal=True, style="hf", mode="query", rope=True, layers=0):
    c = {"api": api, "model": model, "b": b, "s": s, "causal": causal, "style": style, "mode": mode, "rope": rope,
         "layers": layers}
    return dict(c, name=name) if name else c


def listed():
    return [
        # One short prompt through eight layers of the smallest model, replayed from a graph: launch-bound.
        _case("layers 0.6B s128", "launch", "Qwen3-0.6B", 1, 128, layers=8),
        # The same for a D = 256 model without RoPE (factored) at a length where few workgroups exist.
        _case("layers gemma-4B s1024 factored", "factored", "Gemma-3-4B", 1, 1024, rope=False, layers=8),
        # One eager call of a model's attention layer on a short prompt of odd length: host latency.
        _case("call 8B s333", "attention", "Qwen3-8B", 1, 333),
        # A batch of short sequences, bidirectional: the shape the reference quotes for its fused prologue.
        _case("batch 8B b8 s512 full", "attention", "Qwen3-8B", 8, 512, causal=False),
        # A large batch of short prompts of odd length (continuous batching of prefills).
        _case("batch 8B b32 s509", "attention", "Qwen3-8B", 32, 509),
        # The same for a D = 256 model, with its own attention scale.
        _case("batch gemma-12B b8 s512", "fused", "Gemma-3-12B", 8, 512),
        # Ordinary prefill lengths: 2k, a ragged batch, the headline 4k.
        _case("prefill 8B s2048", "launch", "Qwen3-8B", 1, 2048, style="fp32"),
        _case("prefill 8B b4 s1000", "launch", "Qwen3-8B", 4, 1000, style="fp32"),
        _case("prefill 8B s4096", "launch", "Qwen3-8B", 1, 4096, style="fp32"),
        # The factored path at the size it is benchmarked at.
        _case("prefill gemma-12B b2 s2048 factored", "factored", "Gemma-3-12B", 2, 2048, rope=False),
        # The largest call: a long prompt.
        _case("prefill 8B s8192", "launch", "Qwen3-8B", 1, 8192, style="fp32"),
        # Q/K norm + RoPE alone, memory-bound.
        _case("norm_rope 8B b4 s2048", "norm_rope", "Qwen3-8B", 4, 2048, style="fp32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the same ranges: any model of the table, 1 to 32 sequences of 64 to 8192 positions, every form of
    a call, at most 0.6 of the largest listed case's FLOPs and tensors of at most 2^26 elements."""
    while True:
        api = rng.choice(["attention"] * 4 + ["launch"] * 4 + ["fused"] * 2 + ["separate"] + ["factored"] * 3
                         + ["norm_rope"])
        model = rng.choice(sorted(ops.MODELS))
        hq, hkv, d = ops.MODELS[model]
        b, s = _log_int(rng, 1, 32), _log_int(rng, 64, 8192)
        if rng.random() < 0.4 and s >= 128:
            s -= s % 128
        causal = rng.random() < 0.7
        rope = False if api == "factored" else True if api in ("fused", "separate", "norm_rope") else rng.random() < 0.8
        style = "hf" if api in ("fused", "separate") else "fp32" if api == "factored" else rng.choice(
            ["hf", "hf", "fp32", "fp32", "legacy"])
        mode = "unfused" if api == "attention" and rng.random() < 0.25 else "query"
        flops = ops.attention_flops(b, hq, s, d, causal)
        if flops > 0.6 * ops.attention_flops(1, 32, 8192, 128, True) or b * hq * s * d > 2 ** 26:
            continue
        layers = 8 if flops < 6e9 and api in ("launch", "factored", "fused") and rng.random() < 0.7 else 0
        return _case(None, api, model, b, s, causal=causal, style=style, mode=mode, rope=rope, layers=layers)


def _tables(s, d, device):
    pos = torch.arange(s, dtype=torch.float32, device=device)
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, dtype=torch.float32, device=device) / d))
    ang = torch.cat([pos[:, None] * inv[None, :]] * 2, dim=1)
    return ang.cos().to(torch.bfloat16).contiguous(), ang.sin().to(torch.bfloat16).contiguous()


def _inputs(case, seed):
    """Per layer (q, k, v, gq, gk), and the rotary tables (None without RoPE)."""
    hq, hkv, d = ops.MODELS[case["model"]]
    b, s = case["b"], case["s"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    xs = []
    for _ in range(max(1, case["layers"])):
        q, k, v = (normal(b, h, s, d).to(torch.bfloat16) for h in (hq, hkv, hkv))
        gq, gk = ((1 + 0.1 * normal(d)).to(torch.bfloat16) for _ in range(2))
        xs.append((q, k, v, gq, gk))
    return xs, _tables(s, d, "cuda") if case["rope"] else (None, None)


def _call(case, x, tables, kept):
    q, k, v, gq, gk = x
    cos, sin = tables
    api, causal = case["api"], case["causal"]
    if api == "attention":
        return ops.optimized_attention(q, k, v, gq, gk, cos, sin, causal=causal, mode=case["mode"],
                                       norm_style=case["style"])
    if api == "launch":
        rope = cos is not None
        ops.launch_attention((q, k, v, gq, gk, cos if rope else q, sin if rope else k), kept["out"], causal=causal,
                             mode="query", bm=128, rope=rope, kn=kept["kn"], norm_style=case["style"])
        return kept["out"]
    if api in ("fused", "separate"):
        fn = ops.fused if api == "fused" else ops.separate
        return fn(q, k, v, gq, gk, cos, sin, causal, scale=ops.model_scale(case["model"], q.shape[-1]))
    if api == "factored":
        ops.launch_factored_attention(x, kept["out"], kept["inv"], kept["kn"], causal=causal)
        return kept["out"], kept["inv"], kept["kn"]
    return ops.norm_rope(q, k, gq, gk, cos, sin, norm_style=case["style"])


def prepare(case, seed):
    xs, tables = _inputs(case, seed)
    kept = [{"out": torch.empty_like(q), "kn": torch.empty_like(k),
             "inv": torch.empty(q.shape[:-1], device="cuda", dtype=torch.float32)}
            if case["api"] in ("launch", "factored") else None for q, k, *_ in xs]
    state = {"case": case, "xs": xs, "tables": tables, "kept": kept}
    if case["layers"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # warm up outside the capture, as programs that capture do
            _call(case, xs[0], tables, kept[0])
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["outs"] = [_call(case, x, tables, kp) for x, kp in zip(xs, kept)]
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return _call(state["case"], state["xs"][0], state["tables"], state["kept"][0])


def work(case):
    hq, hkv, d = ops.MODELS[case["model"]]
    b, s, n = case["b"], case["s"], max(1, case["layers"])
    q, kv = 2 * b * hq * s * d, 2 * b * hkv * s * d  # bytes of a Q- and of a K-shaped tensor
    tables = 4 * s * d if case["rope"] else 0
    if case["api"] == "norm_rope":
        return {"bytes": 2 * (q + kv) + tables + 4 * d, "flops": 8 * b * s * (hq + hkv) * d}
    extra = 4 * b * hq * s + kv if case["api"] == "factored" else 0  # inv and kn are outputs there
    return {"bytes": n * (2 * q + 2 * kv + 4 * d + extra) + tables, "flops": n * ops.attention_flops(b, hq, s, d, case["causal"])}


def tolerance(case):
    if case["api"] == "norm_rope":
        return {"rel": 0.01, "max": 0.05}
    return {"rel": 0.012, "max": 0.2}


def _norm64(x, gamma):
    x = x.double()
    inv = torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return x * inv * gamma.double(), inv


def _rope64(x, tables):
    cos, sin = tables
    if cos is None:
        return x
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos.double() + turned * sin.double()


def _attention64(q, k, v, causal, scale):
    """softmax(q k^T * scale) v in 64 bits, one sequence and a block of query rows at a time."""
    b, hq, s, d = q.shape
    g = hq // k.shape[1]
    out = torch.empty_like(q)
    rows = max(1, min(s, (1 << 28) // (hq * s)))
    for i in range(b):
        ki = k[i].repeat_interleave(g, dim=0).transpose(1, 2).contiguous()
        vi = v[i].double().repeat_interleave(g, dim=0)
        for r in range(0, s, rows):
            e = min(s, r + rows)
            n = e if causal else s
            scores = torch.matmul(q[i, :, r:e], ki[:, :, :n].contiguous()) * scale
            if causal:
                above = torch.arange(n, device=q.device)[None, :] > torch.arange(r, e, device=q.device)[:, None]
                scores.masked_fill_(above, -math.inf)
            out[i, :, r:e] = torch.matmul(torch.softmax(scores, dim=-1), vi[:, :n])
    return out


def exact(case, seed):
    xs, tables = _inputs(case, seed)
    api, d = case["api"], ops.MODELS[case["model"]][2]
    scale = ops.model_scale(case["model"], d) if api in ("fused", "separate") else d ** -0.5
    outs = []
    for q, k, v, gq, gk in xs:
        qn, inv = _norm64(q, gq)
        kn, inv_k = _norm64(k, gk)
        qn, kn = _rope64(qn, tables), _rope64(kn, tables)
        if api == "norm_rope":
            return qn, kn
        out = _attention64(qn, kn, v, case["causal"], scale)
        # the factored path's kn carries Q's gamma as well
        outs.append((out, inv[..., 0], k.double() * inv_k * gk.double() * gq.double()) if api == "factored" else out)
    return outs if case["layers"] else outs[0]
