"""The waits of the flash prefill's direct global -> LDS loads (powerinfer_x64_amd/csrc/
prefill_loads.hpp) walked on the host: at every barrier the loads of the next step's tiles have
arrived (tests/cpp/test_prefill_loads.cpp).  No GPU is used."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "cpp", "_build", "test_prefill_loads")


def test_prefill_load_waits_host_walk():
    assert os.path.exists(EXE), "tests/cpp not built (python -m powerinfer_x64_amd.build)"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("0 failures"), r.stdout + r.stderr
