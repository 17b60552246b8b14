"""Transforms through the forms of the 16-element NTT pass that the library
picks (10, 9 and 8 bits), run on the host with the library's dispatch
(tests/native/ntt_forms_test.cpp), against the oracle; each pass must have run
the form named here."""
import os
import re
import subprocess

import numpy as np
import pytest

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ntt_forms") / "ntt_forms_test")
    src = os.path.join(ROOT, "tests", "native", "ntt_forms_test.cpp")
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
                        "-I" + os.path.join(ROOT, "include"), src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


def plan_args(bits, k16=None):
    """A plan of these pass bits, the most groups, the 16-element kernel allowed (k16: per pass)."""
    pad = [0] * (3 - len(bits))
    return [str(v) for v in [len(bits)] + list(bits) + pad + [-1] * 3 + list(k16 or [1] * len(bits)) + pad]


def forms(out):
    return re.findall(r"form=(\w+)", out)


CASES = [  # lg, lg_in, columns, inverse, coset, force_exact, twiddle table, plan bits (None: default), forms
    (19, 19, 1, 0, 0, 0, 1, None, ["r10", "r9"]),
    (19, 16, 2, 0, 1, 0, 0, (10, 9), ["r10", "r9"]),
    (19, 19, 1, 1, 1, 1, 1, (9, 10), ["r9", "r10"]),
    (18, 15, 3, 0, 1, 0, 1, None, ["r9", "r9"]),
    (18, 18, 1, 1, 0, 1, 0, None, ["r9", "r9"]),
    (18, 18, 16, 0, 0, 0, 1, (8, 10), ["r8", "r10"]),
    (18, 18, 16, 1, 1, 1, 0, (8, 10), ["r8", "r10"]),
    (18, 14, 16, 0, 1, 1, 1, (8, 10), ["r8", "r10"]),
    (17, 14, 2, 0, 1, 0, 1, None, ["r9", "general"]),
]


@pytest.mark.parametrize("lg,lg_in,C,inv,coset,force,table,bits,want", CASES)
def test_forms_equal_oracle(harness, tmp_path, lg, lg_in, C, inv, coset, force, table, bits, want):
    x = O.random(C << lg_in, 6000 + 16 * lg + lg_in + 3 * inv + 5 * coset + 7 * force)
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    x.tofile(fin)
    r = subprocess.run([harness] + [str(v) for v in (lg, lg_in, C, inv, coset, force, table)] + [fin, fout] +
                       (plan_args(bits) if bits else []), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert forms(r.stdout) == want, r.stdout
    # every tile of the 16-element passes took the exact path, or none did (twiddles computed
    # without a table pass through small powers, whose products a column's first tile redoes)
    for tiles, exact, form in re.findall(r"tiles=(\d+) exact=(\d+) form=(\w+)", r.stdout):
        if form != "general" and (force or table):
            assert exact == (tiles if force else "0"), r.stdout
    got = np.fromfile(fout, dtype=np.uint64)
    if lg_in == lg:
        ref = O.ntt(x, lg, C, inverse=bool(inv), with_coset=bool(coset))
    else:
        ref = O.lde(x, lg_in, lg - lg_in, C, inverse=bool(inv), with_coset=bool(coset))
    assert (got == ref).all(), r.stdout


@pytest.mark.parametrize("bits,C,want", [
    ((8, 10), 15, "general"), ((8, 10), 16, "r8"),          # 512 workgroups
    ((8, 7, 7), 1, "r8"),                                   # 2^22: no other 8-bit pass
    ((8, 5, 8), 11, "general"), ((8, 5, 8), 12, "r8"),      # 3072 workgroups where a later pass has 8 bits
    ((8, 8, 7), 2, "general"), ((8, 8, 7), 3, "r8"),
    ((8, 8, 8), 1, "general"), ((8, 8, 8), 2, "r8"),
    ((8, 8), 400, "general"),                               # 2^16
])
def test_where_a_first_8bit_pass_takes_its_form(harness, bits, C, want):
    """An 8-bit first pass beside another 8-bit pass stays on the general
    kernel, whose code that pass runs too, until the launch is large."""
    lg = sum(bits)
    r = subprocess.run([harness, str(lg), str(lg), str(C), "0", "0", "0", "0", "-", "-"] + plan_args(bits),
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    got = forms(r.stdout)
    assert got[0] == want and "r8" not in got[1:], r.stdout
