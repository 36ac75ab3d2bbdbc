"""Mode 'query' on grids of few workgroups prepares Q with K in its first launch,
into `out`, and attention reads it there: on both sides of each bound (D, with and
without RoPE) the launch records show which way the call went, and the output is
that of mode 'unfused' on a scratch buffer of its own, bit for bit, whole."""
import pytest
import torch

import oracle
from helpers import announce
from kernelfuser_amd import fused, launch_attention, make_inputs

pytestmark = pytest.mark.gpu

# geometry, B, S, RoPE, Q prepared in the first launch (256 CUs; "causal": only then)
CASES = [((16, 8, 128), 1, 1, True, True), ((16, 8, 128), 1, 130, True, True), ((32, 8, 128), 2, 128, True, True),
         ((32, 8, 128), 1, 257, True, False), ((32, 8, 128), 1, 100, False, True), ((3, 1, 128), 11, 65, False, False),
         ((8, 4, 256), 1, 33, True, True), ((16, 8, 256), 1, 1020, True, True), ((16, 8, 256), 1, 1030, True, "causal"),
         ((16, 8, 256), 1, 1270, True, "causal"), ((16, 8, 256), 1, 1290, True, False),
         ((8, 4, 256), 1, 700, False, True), ((8, 4, 256), 1, 1025, False, False)]


def _launch(xs, causal, rope, style, mode, out=None, qn=None):
    out = torch.full_like(xs.q, float("nan")) if out is None else out
    kn = torch.empty_like(xs.k)
    recs = list(launch_attention(xs.reference7, out, causal=causal, mode=mode, rope=rope, qn=qn, kn=kn,
                                 norm_style=style))
    return out, kn, recs


@pytest.mark.parametrize("geom,b,s,rope,prepared", CASES)
@pytest.mark.parametrize("style", ["hf", "fp32"])
def test_query_prepares_q_on_small_grids(gpu, geom, b, s, rope, prepared, style):
    xs = make_inputs(b, s, geom, 9100 + s, rope=rope).to(gpu)
    bound = prepared
    for causal in (True, False):
        announce(f"query {geom} B={b} S={s} rope={rope} {style} causal={causal}")
        prepared = causal if bound == "causal" else bound
        out, kn, recs = _launch(xs, causal, rope, style, "query")
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            # the prologue is the attention instance's fourth argument: 0 for prepared Q
            assert (recs[1]["kernel"].split(", ")[3] == "0") == prepared, recs
        ref, kref, _ = _launch(xs, causal, rope, style, "unfused", qn=torch.empty_like(xs.q))
        torch.cuda.synchronize()
        assert torch.equal(kn, kref)
        if prepared:
            assert torch.equal(out, ref)
        else:  # the prologue's arithmetic, at most an ulp of Q apart
            assert oracle.attention_gate(out.cpu(), ref.cpu().float())["pass"]


@pytest.mark.parametrize("d", [128, 256])
def test_query_out_may_reuse_q_or_k(gpu, d):
    """`out` may be q itself, or k (dead after the preparation), as on larger grids."""
    xs = make_inputs(1, 96, (4, 4, d), 9300).to(gpu)
    announce(f"query D={d} out = q, out = k")
    ref, _, _ = _launch(xs, True, True, "hf", "query")
    torch.cuda.synchronize()
    for name in ("q", "k"):
        ys = make_inputs(1, 96, (4, 4, d), 9300).to(gpu)
        got, _, _ = _launch(ys, True, True, "hf", "query", out=getattr(ys, name))
        torch.cuda.synchronize()
        assert oracle.attention_gate(got.cpu(), ref.cpu().float())["pass"], name


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("name", ["gk", "v", "kn", "gq", "cos", "sin", "q"])
def test_query_out_overlapping_an_operand(gpu, d, name):
    """`out` over gk (dead after the preparation), over each head's own v or kn
    (equal head counts, one block per head) and, on a grid of one workgroup, over
    gamma, the tables or shifted q: Q is not prepared in `out` then."""
    heads, s = (4, 96) if name in ("gk", "v", "kn") else (1, 64)
    xs = make_inputs(1, s, (heads, heads, d), 9350).to(gpu)
    announce(f"query D={d} out over {name}")
    ref, _, recs = _launch(xs, True, True, "hf", "query")
    prologue = lambda r: r[1]["kernel"].split(", ")[3]
    assert prologue(recs) == "0"
    buf = torch.empty(2 * xs.q.numel(), dtype=torch.bfloat16, device=gpu)
    out = buf[:xs.q.numel()].view_as(xs.q)
    ops = dict(zip(("q", "k", "v", "gq", "gk", "cos", "sin"), xs.reference7), kn=torch.empty_like(xs.k))
    shift = {"gk": 5 * d, "gq": 5 * d, "q": 16 * d}.get(name, 0)
    over = buf[shift:shift + ops[name].numel()].view_as(ops[name])
    over.copy_(ops[name])
    ops[name] = over
    kn = ops.pop("kn")
    recs = list(launch_attention(tuple(ops.values()), out, causal=True, mode="query", rope=True, kn=kn,
                                 norm_style="hf"))
    torch.cuda.synchronize()
    assert prologue(recs) == "2", recs
    assert oracle.attention_gate(out.cpu(), ref.cpu().float())["pass"]


def test_fused_small_grid_eps_and_scale(gpu):
    """The older API's explicit eps and scale reach the preparation of Q."""
    xs = make_inputs(1, 70, (8, 4, 256), 9400, qkv_std=0.02).to(gpu)
    announce("fused small grid eps=1e-3 scale=0.05")
    got = fused(xs.q, xs.k, xs.v, xs.gq, xs.gk, xs.cos, xs.sin, True, eps=1e-3, scale=0.05)
    torch.cuda.synchronize()
    ref = oracle.oracle_fp32(*(t.cpu() for t in xs.astuple()), True, scale=0.05, eps=1e-3)
    assert oracle.attention_gate(got.cpu(), ref)["pass"]
    with pytest.raises(ValueError, match="eps must be >= 0"):
        fused(xs.q, xs.k, xs.v, xs.gq, xs.gk, xs.cos, xs.sin, True, eps=-1.0)
