"""Compiler resource reports of kernels whose registers are tight (CPU only:
the kernel is compiled, not run)."""

from __future__ import annotations

import importlib.util
import re
import subprocess
from pathlib import Path

PKG = Path(__file__).resolve().parent.parent / "topk-tarmac_amd"


def _build():
    spec = importlib.util.spec_from_file_location("tarmac_build", PKG / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_dense_backward_at_d64_uses_no_scratch(tmp_path):
    """The d = 64 instantiations of the split-operand dense backward fill the
    register file of two waves a SIMD; none may spill a register to memory."""
    b = _build()
    cmd = [b.hipcc(), *b.HIPCC_FLAGS, "--cuda-device-only", "-c",
           "-Rpass-analysis=kernel-resource-usage", str(b.CSRC / "backward_split.hip"),
           "-o", str(tmp_path / "backward_split.o")]
    run = subprocess.run(cmd, capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    scratch = {}
    for name, size in re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)",
                                 run.stderr, flags=re.S):
        scratch[name] = int(size)
    wide = {n: s for n, s in scratch.items() if "dense_bwd_split_kernelILi64E" in n}
    assert len(wide) >= 3, sorted(scratch)
    assert not any(wide.values()), wide
