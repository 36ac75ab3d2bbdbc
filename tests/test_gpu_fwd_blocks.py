"""The general attention kernel at the sizes where its block pipeline can go
wrong: one to ten 32-key blocks (the K/V rings of two and four tiles wrap, a
sweep ends on either buffer and either half of a 64-key tile), ragged last
blocks and rows, waves with no block at all, and both causal modes, for one,
two and four heads per workgroup (GQA ratios 3, 2 and 4) and every way Q
reaches the matrix cores (prepared, normalised, rotated, factored).
Whole output against the FP32 oracle; and the exact redo of the same shapes,
started by one key far above the first block's row maximum."""
import pytest
import torch

import oracle
from helpers import announce
from kernelfuser_amd import (_lib, attention_prefill, factored_attention, make_inputs, prepare_attention,
                             prepare_factored)

pytestmark = pytest.mark.gpu

# B, S: rows and keys per case
SIZES = [1, 31, 33, 64, 65, 96, 127, 129, 160, 193, 225, 257, 288, 320]


def _expect(xs, causal, rope):
    q, k, v, gq, gk, cos, sin = (None if t is None else t.cpu() for t in xs.astuple())
    return oracle.oracle_fp32(q, k, v, gq, gk, cos if rope else None, sin if rope else None, causal)


@pytest.mark.parametrize("geom", [(3, 1, 128), (4, 2, 128), (8, 2, 128), (3, 1, 256), (4, 2, 256), (8, 2, 256)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("path", ["plain", "norm", "rope", "factored"])
def test_block_counts_whole_output(gpu, geom, causal, path):
    for s in SIZES:
        announce(f"general kernel {geom} S={s} causal={causal} {path}")
        xs = make_inputs(2, s, geom, 7000 + s, rope=path != "factored").to(gpu)
        out = torch.full_like(xs.q, float("nan"))
        kn = torch.empty_like(xs.k)
        rope = path in ("plain", "rope")
        with _lib.tuning(attn_kernel="general"):
            if path == "factored":
                inv = torch.empty(xs.q.shape[:-1], device=gpu)
                prepare_factored((xs.q, xs.k, xs.v, xs.gq, xs.gk), inv, kn)
                factored_attention(xs.q, kn, xs.v, inv, out, causal=causal)
            else:
                qn = torch.empty_like(xs.q)
                prepare_attention(xs.reference7, qn, kn, rope=rope, norm_style="fp32")
                if path == "plain":
                    attention_prefill(qn, kn, xs.v, out, causal=causal, fuse_q=False)
                else:
                    attention_prefill(xs.q, kn, xs.v, out, gq=xs.gq, cos=xs.cos if rope else None,
                                      sin=xs.sin if rope else None, causal=causal, norm_style="fp32")
        torch.cuda.synchronize()
        gate = oracle.attention_gate(out.cpu(), _expect(xs, causal, rope))
        assert gate["pass"], (s, gate)


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("where", ["score", "value"])
def test_redo_whole_output(gpu, d, where):
    """``score``: the last key's logits lie ~150 (log2) above the first
    block's, so every row that sees it overflows the shift; ``value``: values
    near the end of the BF16 range with logits ~20 above, so that only O
    overflows.  Both leave the lean sweep for the exact softmax."""
    for s in (40, 65, 130, 290):
        announce(f"redo D={d} S={s} {where}")
        g = torch.Generator().manual_seed(s)
        q = torch.randn((1, 4, s, d), generator=g).bfloat16()
        k = (0.01 * torch.randn((1, 2, s, d), generator=g)).bfloat16()
        v = torch.randn((1, 2, s, d), generator=g).bfloat16()
        # one key along the queries' common direction
        u = torch.ones(d) / d ** 0.5
        size = 105.0 if where == "score" else 14.0  # logit = size in natural units: 151 or 20 in log2
        q += (4.0 * u).bfloat16()
        k[:, :, s - 1] = (size * d ** 0.5 / 4.0 * u).bfloat16()
        if where == "value":  # 2^20 * 2^115 overflows FP32, 2^8 (the exact path's slack) * 2^115 does not
            v = (v.sign() * 2.0 ** 115).bfloat16()
        out = torch.empty((1, 4, s, d), dtype=torch.bfloat16, device=gpu)
        qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
        with _lib.tuning(attn_kernel="general"):
            attention_prefill(qd, kd, vd, out, causal=False, fuse_q=False)
        torch.cuda.synchronize()
        scale = 2.0 ** -115 if where == "value" else 1.0  # exact in every step
        w = torch.softmax(torch.matmul(q.double(), k.double().repeat_interleave(2, 1).transpose(2, 3)) * d ** -0.5, -1)
        ref = torch.matmul(w, v.double().repeat_interleave(2, 1)) * scale
        got = out.cpu().double() * scale
        assert bool(torch.isfinite(got).all())
        # P and O are each rounded to BF16 (2^-9 relative): within 2^-7 of the largest value
        assert float((got - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max()), (s, float((got - ref).abs().max()))


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("causal", [True, False])
def test_redo_when_o_is_nan_and_never_inf(gpu, d, causal):
    """Values of +-2^100 at probabilities of 2^60, in two 16-key steps: O becomes
    inf and then NaN beside a finite row sum, where the result is finite."""
    s = 150
    q = torch.zeros(1, 4, s, d, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, s, d, dtype=torch.bfloat16)
    v = torch.zeros(1, 2, s, d, dtype=torch.bfloat16)
    q[..., 0] = 8.0
    k[:, :, [40, 60], 0] = 60.0 / (8.0 * d ** -0.5 * 1.4426950408889634)
    v[:, :, 40], v[:, :, 60] = 2.0 ** 100, -(2.0 ** 100)
    announce(f"redo on NaN D={d} causal={causal}")
    out = torch.empty_like(q, device=gpu)
    with _lib.tuning(attn_kernel="general"):
        attention_prefill(q.to(gpu), k.to(gpu), v.to(gpu), out, causal=causal, fuse_q=False)
    torch.cuda.synchronize()
    want = torch.zeros(s)  # the two keys cancel in every row that sees both
    if causal:
        want[40:60] = 1.0
    got = out.cpu().double() * 2.0 ** -100
    assert float((got - want.double()[None, None, :, None]).abs().max()) <= 2.0 ** -8


@pytest.mark.parametrize("geom,b,s", [((8, 2, 128), 64, 257), ((6, 2, 128), 80, 260), ((4, 2, 256), 128, 250)])
@pytest.mark.parametrize("causal", [True, False])
def test_head_major_grid_whole_output(gpu, geom, b, s, causal):
    """Grids of four or more workgroups per CU, which list the query blocks of
    one KV head after the other."""
    announce(f"head-major grid {geom} B={b} S={s} causal={causal}")
    xs = make_inputs(b, s, geom, 7777).to(gpu)
    out = torch.full_like(xs.q, float("nan"))
    kn = torch.empty_like(xs.k)
    prepare_attention(xs.reference7, None, kn, only_k=True, norm_style="fp32")
    with _lib.tuning(attn_kernel="general"):
        attention_prefill(xs.q, kn, xs.v, out, gq=xs.gq, cos=xs.cos, sin=xs.sin, causal=causal, norm_style="fp32")
        grid = [r["grid"] for r in _lib.last_launches()][-1]
    torch.cuda.synchronize()
    assert grid >= 1024, grid  # 4 x 256 CUs
    assert oracle.attention_gate(out.cpu(), _expect(xs, causal, True))["pass"]
