"""The relaxed Poseidon permutations flag no rare case on random states
(tests/native/poseidon_rare_test.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_random_states_are_not_rare(tmp_path):
    exe = str(tmp_path / "poseidon_rare_test")
    src = os.path.join(ROOT, "tests", "native", "poseidon_rare_test.cpp")
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                        src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok, 2000 states, 0 rare"), r.stdout + r.stderr[-2000:]
