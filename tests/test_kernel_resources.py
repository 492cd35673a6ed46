"""Registers of the vocabulary projection's kernels (csrc/gemm_mid.hip), from the compiler's resource
report with the build's own flags (cross-compiled, no GPU): waves per SIMD and no spilled registers.
"""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nki-moe-megakernel_amd")


def _report(source, tmp_path):
    """{mangled kernel name: (waves per SIMD, spilled vector registers)}"""
    spec = importlib.util.spec_from_file_location("mkd_build", os.path.join(PKG, "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not shutil.which(b.HIPCC):
        pytest.skip("hipcc not available")
    r = subprocess.run([b.HIPCC, *b.COMMON_FLAGS, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                        os.path.join(PKG, "csrc", source), "-o", str(tmp_path / "k.o")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = {}
    for part in r.stderr.split("Function Name: ")[1:]:
        num = {k: int(re.search(re.escape(k) + r": (\d+)", part).group(1)) for k in
               ("Occupancy [waves/SIMD]", "VGPRs Spill")}
        out[part.split()[0]] = tuple(num.values())
    return out


def test_vocabulary_projection_waves(tmp_path):
    """The forms of up to 32 / 64 / 128 tokens keep 4 / 3 / 2 waves per SIMD: they stream weights, and
    the waves are what keeps loads in flight while one multiplies."""
    rep = {k: v for k, v in _report("gemm_mid.hip", tmp_path).items() if "gemm_kloop_kernel" in k}
    assert len(rep) == 3
    for name, (waves, spilled) in rep.items():
        tokens = 16 * int(re.search(r"kernelILi(\d+)E", name).group(1))
        assert waves >= {32: 4, 64: 3, 128: 2}[tokens] and spilled == 0, (name, waves, spilled)
