"""The 9-bit and 8-bit forms of the 16-element NTT pass (zeknox_amd/csrc/ntt_pass.hpp),
their per-thread code run on the host under AddressSanitizer and UBSan, against
the general pass: as first, middle and last pass, forward, inverse and LDE (0
to 6 skipped bits), with and without the coset, the twiddle table, a scratch
buffer and the forced exact path."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_small_forms_equal_general_pass(tmp_path):
    exe = str(tmp_path / "ntt_r9_test")
    src = os.path.join(ROOT, "tests", "native", "ntt_r9_test.cpp")
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                        "-Xarch_host", "-fsanitize=address", "-Xarch_host", "-fsanitize=undefined", "-o", exe, src],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr[-2000:]
