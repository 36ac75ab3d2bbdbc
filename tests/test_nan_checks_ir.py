"""The attention kernels' inf/NaN checks survive their build flags (no GPU).

The ping-pong and wide kernels' files are built without NaN semantics
(-fno-honor-nans, so max trees map onto v_max3_f32).  A test of the exponent bits of a value produced
by floating-point arithmetic is then rewritten by the compiler as a class
test, an unordered compare of fabs(x) with +inf whose operand is marked as
never NaN, and a NaN passes it.  The wide kernel's row-sum check was
rewritten that way, so a NaN row sum did not start the exact redo.  The checks
now pass the bits through an empty asm (`opaque_bits`).  One test compiles
these files to device LLVM IR with the build's own flags and checks that no
such compare is left.  The general kernel's check of O keeps a NaN through
floating-point maxima (`pack_rows`), so its files must have NaN semantics: the
other test pins their flags.
"""
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from kernelfuser_amd import build as B

FILES = ["attn_pp.hip", "attn_wide.hip"]
NAN_FILES = ["attn_fwd128.hip", "attn_fwd256.hip"]
INF_COMPARE = re.compile(r"fcmp [a-z ]*ueq float %\S+, 0x7FF0000000000000")


def _device_ir(name, out_dir):
    out = out_dir / (name + ".ll")
    cmd = [B.hipcc(), *B.COMMON, *B.DEVICE_FLAGS, *B.FILE_FLAGS.get(name, []), "--cuda-device-only", "-S",
           "-emit-llvm", str(B.CSRC / name), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    assert res.returncode == 0, res.stderr[-2000:]
    return out.read_text()


def test_no_inf_class_compares_in_attention_ir(tmp_path):
    try:
        B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    assert all(B.FILE_FLAGS.get(f) == ["-fno-honor-nans"] for f in FILES)  # the flags this guards against
    with ThreadPoolExecutor(len(FILES)) as ex:
        irs = dict(zip(FILES, ex.map(lambda f: _device_ir(f, tmp_path), FILES)))
    found = {f: INF_COMPARE.findall(ir)[:3] for f, ir in irs.items() if INF_COMPARE.search(ir)}
    assert not found, found
    assert "define" in irs["attn_wide.hip"] and "attn_ww_kernel" in irs["attn_wide.hip"]


def test_general_kernel_is_built_with_nan_semantics():
    for f in NAN_FILES:
        assert '#include "attn_fwd.h"' in (B.CSRC / f).read_text()
        flags = " ".join([*B.COMMON, *B.DEVICE_FLAGS, *B.FILE_FLAGS.get(f, [])])
        assert not re.search(r"honor-nans|fast-math|finite-math|honor-infinities|-Ofast", flags), (f, flags)
    # and nothing else instantiates pack_rows
    users = [p.name for p in B.CSRC.iterdir() if "pack_rows(" in p.read_text()]
    assert sorted(users) == ["attn_fwd.h", "attn_mfma.h"], users
