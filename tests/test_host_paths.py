"""The solver's host code on a runtime in host memory
(tests/csrc/host_paths.cpp): failed allocations, launches on several streams,
timed-out waits, captured projections, what memory a handle holds.  One
scenario per test."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "opensayal_amd" / "csrc"
HERE = ROOT / "tests" / "csrc"
ROCM = Path("/opt/rocm/include")

SCENARIOS = [
    "exchange_out_of_memory",
    "autotune_fails",
    "autotune_without_exchange",
    "autotune_times_out",
    "batch_autotune_times_out",
    "cleaned_in_stream_order",
    "captured_projection",
    "exchange_is_counted",
    "exchange_in_a_budget",
    "resident_says_what_runs",
    "dividing_is_resident",
    "staging_is_bounded",
    "staging_shares_the_link",
    "batch_division",
    "project_shape_follows_sweeps",
    "launches_are_counted",
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None or not ROCM.exists():
        pytest.skip("needs g++ and the HIP headers")
    out = tmp_path_factory.mktemp("host_paths")
    sources = [CSRC / n for n in ("fluid_host.cpp", "batch_host.cpp", "staging.cpp", "config.cpp",
                                  "json_value.cpp")] + [HERE / "fake_hip.cpp",
                                                        HERE / "host_paths.cpp"]
    jobs = [(subprocess.Popen(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                               f"-I{ROCM}", "-c", str(s), "-o", str(out / (s.stem + ".o"))]))
            for s in sources]
    assert all(j.wait() == 0 for j in jobs)
    exe = out / "host_paths"
    subprocess.run(["g++", "-pthread", "-o", str(exe),
                    *[str(out / (s.stem + ".o")) for s in sources]], check=True)
    return exe


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_host_path(program, scenario):
    res = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout + res.stderr
