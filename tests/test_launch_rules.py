"""The host-side launch rules of leapquant_amd/csrc/lq_rules.h, compiled for the CPU and evaluated over their whole range."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RULES = os.path.join(ROOT, "leapquant_amd", "csrc", "lq_rules.h")

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="needs a host C++ compiler")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = d / "rules.cpp", d / "rules.so"
    src.write_text('#include "%s"\nextern "C" int kda_decode_heads(int N, int HV, int H, int L, int cus) '
                   '{ return lq_kda_decode_heads(N, HV, H, L, cus); }\n' % RULES)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("cus", [256, 304])
def test_kda_one_launch_workgroups_hold_whole_key_heads(rules, cus):
    """A key head's value heads share its key window, of which the first one appends the token's key; the flush of each
    reads it in the same launch, so all of them sit in one workgroup: W heads hv0 = 0, W, 2 W, ... of a row."""
    chosen = set()
    for H in (1, 2, 3, 4, 5, 8, 16, 32):
        for G in (1, 2, 3, 4, 8):
            HV = H * G
            for N in (1, 2, 3, 9, 31, 32, 33, 64, 100, 128, 256, 1024):
                for L in (1, 16, 31, 32, 33, 64):
                    W = rules.kda_decode_heads(N, HV, H, L, cus)
                    chosen.add((W, G))
                    if W == 0:
                        continue
                    assert HV % W == 0, (N, HV, H, L)
                    assert all(hv // W == hv // G * G // W for hv in range(HV)), (N, HV, H, L, W)
    assert {(1, 1), (2, 1), (2, 2), (0, 2), (0, 4)} <= chosen     # every form is reached
