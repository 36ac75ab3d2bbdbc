"""The general attention kernel's lean softmax and its exact redo.

After the first KV tile of a work item the kernel takes p = exp2(logit -
m_run) with no per-tile max; a lane whose share of a row sum reaches 2^64 makes
the whole workgroup redo the item with the exact online softmax.  These inputs
put one key's logit so far above the first tile's row max (up to 163 in log2
units, where exp2 overflows) that only the redo gives finite, correct rows;
the FP32 oracle (softmax attention on the same prepared Q/K) is the check.
"""
import pytest
import torch

import oracle
from helpers import announce
from kernelfuser_amd import _lib, anchor, attention_prefill

pytestmark = pytest.mark.gpu


def _spiked(b, hq, hkv, s, d, key, seed):
    g = torch.Generator().manual_seed(seed)
    q = 0.1 * torch.randn(b, hq, s, d, generator=g)
    k = 0.1 * torch.randn(b, hkv, s, d, generator=g)
    v = torch.randn(b, hkv, s, d, generator=g)
    q[..., 0] = 8.0          # every query leans along e0
    k[:, :, key, 0] = 160.0  # one key far along e0: logit 1280/sqrt(D)
    return tuple(t.to(torch.bfloat16) for t in (q, k, v))


@pytest.mark.parametrize("d,hq,hkv,s,causal", [(128, 8, 2, 700, True), (128, 8, 2, 700, False),
                                               (256, 4, 2, 640, True), (256, 4, 2, 640, False)])
def test_lean_overflow_takes_exact_redo(gpu, d, hq, hkv, s, causal):
    q, k, v = _spiked(1, hq, hkv, s, d, 300, 4242)
    announce(f"lean redo D={d} Hq={hq} Hkv={hkv} S={s} causal={causal}")
    out = anchor(q.to(gpu), k.to(gpu), v.to(gpu), None, None, causal)
    torch.cuda.synchronize()
    out = out.cpu()
    assert torch.isfinite(out.float()).all()
    ref = oracle.attention_fp32(q, k, v, causal)
    m = oracle.attention_gate(out, ref)
    assert m["pass"], m
    # rows that see the spiked key are its value row
    first = 300 if causal else 0
    kv_of = torch.arange(hq) // (hq // hkv)
    want = v[0, kv_of, 300].float()[:, None, :].expand(hq, s - first, d)
    assert (out[0, :, first:].float() - want).abs().max() <= 2e-2


def test_lean_matches_exact_on_ordinary_inputs(gpu):
    """Without a spike no redo happens and the result is the same softmax."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, h, 900, 128, generator=g).to(torch.bfloat16) for h in (8, 2, 2))
    announce("lean ordinary D=128 S=900 causal")
    out = anchor(q.to(gpu), k.to(gpu), v.to(gpu), None, None, True)
    torch.cuda.synchronize()
    m = oracle.attention_gate(out.cpu(), oracle.attention_fp32(q, k, v, True))
    assert m["pass"], m


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("keys", [(40, 44), (40, 41), (40,), (70, 76, 81)])
@pytest.mark.parametrize("causal", [True, False])
def test_row_sums_near_overflow(gpu, d, keys, causal):
    """Spikes 60 to 130 (log2) above the first block's maximum, small values:
    the row sum reaches 2^128 and more while O stays finite.  Keys 40 and 44 (mod
    8 below 4, and 4 or above) are summed by different lanes, so at 127.5 both
    lanes' sums are finite and only their total is not."""
    s = 150
    g = torch.Generator().manual_seed(11)
    v = (torch.rand(1, 2, s, d, generator=g) - 0.5).bfloat16()
    unit = 8.0 * d ** -0.5 * 1.4426950408889634  # log2 logit of a key whose component along the queries is 1
    for level in (60.0, 63.5, 64.5, 120.0, 126.5, 127.25, 127.5, 127.75, 128.5, 130.0):
        q = torch.zeros(1, 4, s, d, dtype=torch.bfloat16)
        k = torch.zeros(1, 2, s, d, dtype=torch.bfloat16)
        q[..., 0] = 8.0
        c0 = torch.tensor(level / unit).bfloat16().float()  # the level to 2^-16, in two components
        q[..., 1] = 8.0
        for key in keys:
            k[:, :, key, 0] = c0
            k[:, :, key, 1] = level / unit - c0
        announce(f"row sum near overflow D={d} keys={keys} level={level} causal={causal}")
        out = torch.empty_like(q, device=gpu)
        with _lib.tuning(attn_kernel="general"):
            attention_prefill(q.to(gpu), k.to(gpu), v.to(gpu), out, causal=causal, fuse_q=False)
        torch.cuda.synchronize()
        ref = oracle.attention_fp32(q, k, v, causal)
        err = float((out.cpu().float() - ref).abs().max())
        # P and the result are each rounded to BF16 (2^-9 relative), |V| <= 0.5
        assert err <= 2.0 ** -9, (level, err)


def test_first_tile_sets_the_shift(gpu):
    """D = 128: the shift is the maximum of the first 64 keys.  Of two keys that
    count, the larger is in the second 32: its probability is 1 exactly and its
    weight 1 / (1 + 2^-2.05).  Relative to the first 32 keys' maximum it would be
    BF16(2^2.05) / (1 + 2^2.05), 0.0037 above, on the other side of a rounding tie that lies 0.3
    spacings off on either side."""
    s, x = 64, 2.05
    exact, other = 1 / (1 + 2.0 ** -x), float(torch.tensor(2.0 ** x).bfloat16()) / (1 + 2.0 ** x)
    want = torch.tensor(exact).bfloat16()
    assert want != torch.tensor(other).bfloat16()
    unit = 8.0 * 128 ** -0.5 * 1.4426950408889634
    q = torch.zeros(1, 2, s, 128, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, s, 128, dtype=torch.bfloat16)
    v = torch.zeros(1, 2, s, 128, dtype=torch.bfloat16)
    q[..., :2] = 8.0
    level = torch.full((s,), -60.0)
    level[5], level[50] = 0.0, x
    c0 = (level / unit).bfloat16()
    k[..., 0], k[..., 1] = c0, (level / unit - c0.float()).bfloat16()
    v[:, :, 50] = 1.0
    announce("shift of the first tile")
    out = torch.empty_like(q, device=gpu)
    with _lib.tuning(attn_kernel="general"):
        attention_prefill(q.to(gpu), k.to(gpu), v.to(gpu), out, causal=False, fuse_q=False)
    torch.cuda.synchronize()
    assert bool((out.cpu() == want).all()), (out.unique(), want)


@pytest.mark.parametrize("d", [128, 256])
def test_row_sums_of_long_rows(gpu, d):
    """One key of probability 1 and 30187 of 2^-24.4, too small to change 1.0 one by
    one in FP32.  Summed by tile first they all count; in a chain over a quarter
    of the keys that starts at 1.0 a quarter of them would be lost, 3.4e-4 of the
    sum.  The result lies 1.3e-4 below a tie of BF16 rounding, which that crosses."""
    s, n = 30188, 30187
    p = 2.0 ** -24.4
    exact = n * float(torch.tensor(p).bfloat16()) / (1 + n * p)  # P is BF16 in the product, FP32 in the sum
    want = torch.tensor(exact, dtype=torch.float64).bfloat16().double()
    lossy = exact * (1 + n * p) / (1 + 0.75 * n * p)
    tie = float(want) + 0.5 * 2.0 ** -17  # the spacing of BF16 at 2^-9.5
    assert exact * (1 + 1e-4) < tie < lossy * (1 - 1e-4)
    unit = 8.0 * d ** -0.5 * 1.4426950408889634
    q = torch.zeros(1, 1, s, d, dtype=torch.bfloat16, device=gpu)
    k = torch.zeros_like(q)
    v = torch.ones_like(q)
    q[..., :2] = 8.0
    c0 = torch.tensor(-24.4 / unit).bfloat16().float()
    k[:, :, 1:, 0] = c0
    k[:, :, 1:, 1] = -24.4 / unit - c0
    v[:, :, 0] = 0.0
    announce(f"long row sums D={d}")
    out = torch.empty_like(q)
    with _lib.tuning(attn_kernel="general"):
        attention_prefill(q, k, v, out, causal=False, fuse_q=False)
    torch.cuda.synchronize()
    assert bool((out == want.bfloat16().item()).all()), (out.unique(), want)
