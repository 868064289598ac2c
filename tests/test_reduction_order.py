"""Compiles the step kernels to gfx950 assembly and checks the order the pressure
range rests on: a workgroup's partial result, an agent-scope store (it bypasses
the caches that are not coherent between XCDs), has completed before the
workgroup is counted as finished.  The C++ memory model does not give that order
to relaxed atomics; the wait between them does, so it has to be there."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "opensayal_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not installed")
def test_partial_results_complete_before_the_count(tmp_path):
    out = tmp_path / "ks.s"
    subprocess.run([HIPCC, "-O3", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                    "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-fno-gpu-rdc", "-x", "hip", "-S", "--cuda-device-only",
                    str(CSRC / "kernels_step.hip"), "-o", str(out)],
                   check=True, capture_output=True, cwd=tmp_path)
    text = out.read_text()
    body = re.search(r"^_Z\w*k_minmax\w*:.*?s_endpgm", text, re.M | re.S).group(0)
    code = [line.strip() for line in body.split("\n")]
    counts = [i for i, line in enumerate(code) if re.match(r"global_atomic_(add|inc)", line)]
    assert len(counts) == 1
    stores = [i for i, line in enumerate(code[:counts[0]]) if line.startswith("global_store_")]
    assert stores and "sc1" in code[stores[-1]]
    between = code[stores[-1] + 1:counts[0]]
    assert any(re.match(r"s_waitcnt .*vmcnt\(0\)", line) for line in between), between
