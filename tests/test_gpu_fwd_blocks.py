"""The general attention kernel at the sizes where its block pipeline can go
wrong: one to ten 32-key blocks (the K/V rings of two and four tiles wrap, a
sweep ends on either buffer and either half of a 64-key tile), ragged last
blocks and rows, waves with no block at all, and both causal modes, for every
way Q reaches the matrix cores (prepared, normalised, rotated, factored) and
one, two and four heads per workgroup (GQA ratios 3, 2 and 4: with RoPE on any
grid, the other ways on grids of more workgroups than CUs).  The launch record
says how many heads a workgroup took.  Whole output against the FP32 oracle;
and the exact redo, started by one key far above the first tile's row maximum."""
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


def _heads(geom, path, workgroups):
    """Heads per workgroup: as many as divide the GQA group, up to four at D = 128
    and two at D = 256; one without rotary tables on grids of up to 256."""
    group = geom[0] // geom[1]
    if path != "rope" and workgroups <= 256:
        return 1
    return 4 if geom[2] == 128 and group % 4 == 0 else 2 if group % 2 == 0 else 1


def _check(gpu, geom, b, s, causal, path):
    announce(f"general kernel {geom} B={b} S={s} causal={causal} {path}")
    xs = make_inputs(b, s, geom, 7000 + s, rope=path != "factored").to(gpu)
    out = torch.full_like(xs.q, float("nan"))
    kn = torch.empty_like(xs.k)
    rope = path in ("plain", "rope")
    no_split = torch.empty(0, dtype=torch.uint8, device=gpu)
    with _lib.tuning(attn_kernel="general"):
        if path == "factored":
            inv = torch.empty(xs.q.shape[:-1], device=gpu)
            prepare_factored((xs.q, xs.k, xs.v, xs.gq, xs.gk), inv, kn)
            factored_attention(xs.q, kn, xs.v, inv, out, causal=causal, work=no_split)
        else:
            qn = torch.empty_like(xs.q)
            prepare_attention(xs.reference7, qn, kn, rope=rope, norm_style="fp32")
            if path == "plain":
                attention_prefill(qn, kn, xs.v, out, causal=causal, fuse_q=False, work=no_split)
            else:
                attention_prefill(xs.q, kn, xs.v, out, gq=xs.gq, cos=xs.cos if rope else None,
                                  sin=xs.sin if rope else None, causal=causal, norm_style="fp32", work=no_split)
        plan = [r["plan"] for r in _lib.last_launches()][-1]
    torch.cuda.synchronize()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        heads = _heads(geom, path, b * geom[0] * -(-s // 128))
        assert f"heads={heads}" in plan.split(), (plan, heads)
    gate = oracle.attention_gate(out.cpu(), _expect(xs, causal, rope))
    assert gate["pass"], (s, gate)


GEOMS = [(3, 1, 128), (4, 2, 128), (8, 2, 128), (3, 1, 256), (4, 2, 256), (8, 2, 256)]


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("path", ["plain", "norm", "rope", "factored"])
def test_block_counts_whole_output(gpu, geom, causal, path):
    for s in SIZES:
        _check(gpu, geom, 2, s, causal, path)


@pytest.mark.parametrize("geom", [(4, 2, 128), (8, 2, 128), (4, 2, 256), (8, 2, 256)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("path", ["plain", "norm", "factored"])
def test_shared_workgroups_whole_output(gpu, geom, causal, path):
    """Several heads per workgroup without rotary tables: more than one workgroup
    per CU, ragged rows that leave waves without any."""
    for s in (1, 33, 65, 129, 161):
        _check(gpu, geom, 264 // geom[0], s, causal, path)


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


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("causal", [True, False])
def test_redo_of_rotated_rows_whole_output(gpu, geom, causal):
    """The redo behind the fused prologue (Q normalised and rotated in place), with
    and without a causal mask, for one, two and four heads per workgroup: one key
    whose logits lie ~150 (log2) above the others', along the queries' first component."""
    b, s, d = 3, 150, geom[2]
    xs = make_inputs(b, s, geom, 7600)
    key = 100
    xs.q[..., 0] = 4 * d ** 0.5  # after the norm 4 / sqrt(17) * sqrt(d), times gamma
    xs.cos[:, 0] = 1.0  # and the rotation leaves it in place
    xs.cos[:, d // 2] = 1.0
    xs.sin[:, 0] = 0.0
    xs.sin[:, d // 2] = 0.0
    xs = xs.to(gpu)
    kn = torch.empty_like(xs.k)
    prepare_attention(xs.reference7, None, kn, only_k=True, norm_style="fp32")
    kn[:, :, key] = 0.0
    kn[:, :, key, 0] = 110.0
    announce(f"redo of rotated rows {geom} causal={causal}")
    out = torch.full_like(xs.q, float("nan"))
    with _lib.tuning(attn_kernel="general"):
        attention_prefill(xs.q, kn, xs.v, out, gq=xs.gq, cos=xs.cos, sin=xs.sin, causal=causal, norm_style="fp32")
        plan = [r["plan"] for r in _lib.last_launches()][-1]
    torch.cuda.synchronize()
    assert f"heads={_heads(geom, 'rope', 0)}" in plan.split(), plan
    q = oracle.norm_rope_fp32(*(t.cpu() for t in (xs.q, xs.gq, xs.cos, xs.sin)))
    logits = torch.matmul(q.bfloat16().float()[:, :, key:], kn.cpu().float()[:, :, key, :, None].repeat_interleave(
        geom[0] // geom[1], 1)) * d ** -0.5 * 1.4426950408889634
    assert float(logits.min()) > 100.0  # far above the redo's bound in every row that sees the key
    ref = oracle.attention_fp32(q.bfloat16(), kn.cpu(), xs.v.cpu(), causal)
    assert oracle.attention_gate(out.cpu(), ref)["pass"]


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
