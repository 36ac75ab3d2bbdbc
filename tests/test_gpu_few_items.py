"""Causal D = 128 grids from 24 query blocks of 128 rows: with fewer than 1.5
ping-pong items per compute unit the general kernel runs."""
import pytest
import torch

import oracle
from kernelfuser_amd import _lib, launch_attention, make_inputs


@pytest.mark.parametrize("b,hq,hkv,s,kernel", [
    (1, 16, 8, 2944, "general"),    # 23 blocks
    (1, 16, 8, 2945, "general"),    # 24 blocks: 192 items on 256 CUs
    (1, 16, 8, 4096, "general"),    # 256 items
    (1, 16, 8, 6016, "general"),    # 376 items
    (1, 16, 8, 6017, "pingpong"),   # 384 items
    (1, 16, 8, 8192, "pingpong"),   # paired
    (1, 32, 4, 3008, "general"),    # four heads per item: 47 blocks of 64 rows, 376 items
    (1, 32, 4, 3009, "pingpong"),   # 48 blocks, 384 items
    (2, 8, 2, 3200, "general"),     # 200 items, heads in plain order
    (1, 8, 2, 8192, "general"),     # 256 items, heads in plain order
])
def test_kernel_choice(b, hq, hkv, s, kernel):
    assert _lib.attention_kernel(b, hq, hkv, s, 128, True, 0) == kernel


@pytest.mark.gpu
@pytest.mark.parametrize("geom,b,s", [((16, 8, 128), 1, 2945), ((16, 8, 128), 1, 6016), ((8, 2, 128), 2, 3200),
                                      ((32, 4, 128), 1, 3008)])
@pytest.mark.parametrize("style", ["fp32", "hf"])
def test_general_kernel_rows(gpu, geom, b, s, style):
    """Two rows of every query block and the last row pass the oracle gate."""
    xs = make_inputs(b, s, geom, 6161)
    g = xs.to(gpu)
    out, kn = torch.full_like(g.q, float("nan")), torch.empty_like(g.k)
    print(f"attention query {style} geometry={geom} B={b} S={s} causal (few items)", flush=True)
    recs = list(launch_attention(g.reference7, out, causal=True, mode="query", kn=kn, norm_style=style))
    torch.cuda.synchronize()
    assert any(r["kernel"].startswith("attn_fwd_kernel") for r in recs), recs
    rows = torch.unique(torch.cat([torch.arange(0, s, 128), torch.arange(77, s, 128), torch.tensor([s - 1])]))
    m = oracle.attention_gate(out.cpu()[:, :, rows], oracle.oracle_rows_fp32(*xs.astuple(), rows, True))
    assert m["pass"], m
    assert not out.isnan().any()
