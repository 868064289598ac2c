"""The quotient of the register and resident projection kernels
(projection_device.hpp: any_quotient, quotient_class, and the lines of
kind_quotient that use them), taken from the header and run over all 2^32 binary32 inputs for every number of open
faces against IEEE division (tests/csrc/any_quotient_check.cpp).  A table with
one digit changed has to be noticed."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "opensayal_amd" / "csrc" / "projection_device.hpp"
CHECK = Path(__file__).resolve().parent / "csrc" / "any_quotient_check.cpp"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def shipped():
    text = HEADER.read_text()
    parts = []
    for name in ("any_quotient", "quotient_class"):
        found = re.findall(rf"^__device__ inline [\w ]+ {name}\(.*?^}}\n", text, re.M | re.S)
        assert len(found) == 1, name
        parts.append(found[0])
    used = re.findall(r"^    const float s = \(float\)\(c & 255u\), y = .*?"
                      r"^    float q = any_quotient\(div, y, s\);\n", text, re.M | re.S)
    assert len(used) == 1 and used[0].count("\n") == 2
    parts.append("static float class_quotient(float div, uint32_t c) {\n" + used[0] +
                 "    return q;\n}\n")
    return "".join(parts)


def run(tmp_path, text, step=1):
    (tmp_path / "shipped.inc").write_text(text)
    exe = tmp_path / "check"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-fopenmp", f"-I{tmp_path}", "-o",
                    str(exe), str(CHECK)], check=True)
    res = subprocess.run([str(exe), str(step)], capture_output=True, text=True, timeout=600)
    return dict(line.rsplit(" ", 1) for line in res.stdout.strip().splitlines()), res.returncode


def test_shipped_quotient_is_exact(tmp_path):
    lines, rc = run(tmp_path, shipped())
    assert set(lines) == {f"class {s}:" for s in range(5)} | {"wall 3:", "wall 4:"}
    assert set(lines.values()) == {"0"} and rc == 0, lines


def test_a_wrong_table_is_noticed(tmp_path):
    text = shipped()
    assert "0x346C0u" in text
    lines, rc = run(tmp_path, text.replace("0x346C0u", "0x356C0u"), step=4099)
    assert rc != 0 and lines["class 3:"] != "0" and lines["class 4:"] == "0", lines
