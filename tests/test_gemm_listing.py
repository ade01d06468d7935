"""The 256x256 products keep their accumulators in AGPRs between runs of the
loop text, where the compiler cannot see them; this checks on the compiled
listing that it uses no AGPR, and no scratch memory, of its own there."""

import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parents[1] / "voodoo-dyn-quant_amd"


def test_compiler_leaves_the_accumulators_alone(tmp_path):
    sys.path.insert(0, str(PKG))
    import build

    hipcc = build._hipcc()
    if shutil.which(hipcc) is None:
        pytest.skip("hipcc not found")
    out = tmp_path / "vq_gemm.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([hipcc, *flags, "-S", "--offload-device-only", str(PKG / "csrc" / "vq_gemm.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    kernel, in_text, checked, bad = None, False, set(), []
    for line in out.read_text().splitlines():
        m = re.match(r"(_Z\S+):", line)
        if m:
            kernel = m.group(1)
        if "ASMSTART" in line:
            in_text = True
            if kernel and "st_" in kernel:
                checked.add(kernel)
        elif "ASMEND" in line:
            in_text = False
        elif kernel in checked and not in_text and not line.strip().startswith((";", ".")):
            if re.search(r"\ba\d+\b|\ba\[|accvgpr|scratch_", line):
                bad.append((kernel[:60], line.strip()))
    assert len(checked) >= 9, sorted(checked)  # forward, dX, gate (2), parts, duals (3), routed
    assert not bad, bad[:10]
