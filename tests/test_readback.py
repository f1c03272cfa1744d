"""Image read-back through pinned staging (csrc/readback.cpp) on the CPU: the
class itself, compiled over a stand-in HIP runtime whose one stream can be
held as if a frame were still rendering, and whose calls can fail."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_readback_over_a_stand_in_runtime(tmp_path):
    exe = tmp_path / "readback_check"
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-I", str(ROOT / "tests" / "fake_hip"),
           str(ROOT / "tests" / "readback_check.cpp"), str(ROOT / "lavaframe_amd" / "csrc" / "readback.cpp"),
           "-o", str(exe), "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok"), r.stdout + r.stderr
