"""Host-side checks of the multi-step plan of the explicit kernel (no GPU)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_refused_threads_and_memory(tmp_path):
    """The planner runs inside a C call: a system that refuses its threads or their memory must not end the
    process (tests/capi/multi_plan_check.cpp)."""
    exe = tmp_path / "multi_plan_check"
    csrc = ROOT / "svl_amd" / "csrc"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", str(csrc), str(ROOT / "tests" / "capi" / "multi_plan_check.cpp"),
                    str(csrc / "svlg_tiles.cpp"), "-o", str(exe), "-lpthread", "-ldl"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
