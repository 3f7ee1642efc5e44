"""Code-generation guard for the pooled means (CPU: hipcc cross-compiles to
gfx950 assembly): a block mean goes fp64 -> fp32 -> 16 bits, two roundings, as
the oracle's does. Left alone the compiler merges the two conversions of some
instantiations into one fp64 -> bf16 rounding (recognisable by the
v_cmp_nlg_f64 of its round-to-odd step), which differs where the fp32 value is
a tie: a mean 1.5e-8 above 0.556640625 rounds to 0.5546875 in two steps and to
0.55859375 in one."""

import os
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(shutil.which(HIPCC) is None and not Path(HIPCC).exists(),
                    reason="hipcc not available")
def test_pooled_means_round_twice():
    src = ROOT / "flashprefill_amd" / "csrc" / "fp_plan_pool.hip"
    with tempfile.TemporaryDirectory() as td:
        out = Path(td) / "fp_plan_pool.s"
        cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--offload-device-only", "-S",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               f"-I{ROOT / 'include'}", f"-I{src.parent}", str(src), "-o", str(out)]
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
        assert r.returncode == 0, r.stderr[-2000:]
        asm = out.read_text()
    assert "v_cvt_f32_f64" in asm and "v_cvt_pk_bf16_f32" in asm
    assert "v_cmp_nlg_f64" not in asm
