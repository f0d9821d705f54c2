"""The host-side launch rules of leapquant_amd/csrc/lq_rules.h, compiled for the CPU and evaluated over their range."""
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
    src.write_text('#include "%s"\nextern "C" {\nint kda_decode_heads(int N, int HV, int H, int L, int cus) '
                   '{ return lq_kda_decode_heads(N, HV, H, L, cus); }\n'
                   'int gdn_decode_form(int N, int HV, int H, int K, int V, int R, int L, int conv, int deferred, int cus) '
                   '{ return lq_gdn_decode_form(N, HV, H, K, V, R, L, conv != 0, deferred != 0, cus); }\n}\n' % RULES)
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


TWO, ONE, HELPERS = 0, 1, 2


def test_gdn_forms_have_kernels(rules):
    """Over heads, dims, ranks and sizes: a form is chosen only where its kernels exist (one launch: HV / H of 1 with an even
    H and R <= 4, 2 or 4; helper waves: R <= 4, V = 128 or HV = H, workgroups that are all resident)."""
    seen = set()
    for K, V in ((128, 128), (64, 128), (64, 64)):
        for R in (1, 4) + ((5, 8) if K == 128 else ()):
            for H in (1, 2, 3, 4, 8, 16, 32):
                for G in (1, 2, 3, 4):
                    for N in (1, 4, 5, 8, 16, 24, 32, 64, 100, 256, 1000):
                        for L in (1, 16, 33, 64):
                            for conv in (0, 1):
                                for deferred in (0, 1):
                                    f = rules.gdn_decode_form(N, H * G, H, K, V, R, L, conv, deferred, 256)
                                    seen.add((f, G, V, R > 4, conv, deferred))
                                    if f != TWO:
                                        assert G in (2, 4) or (G == 1 and H % 2 == 0 and R <= 4)
                                    if f == HELPERS:
                                        assert R <= 4 and (V == 128 or G == 1) and N * H * G <= 4 * 256
    assert {(HELPERS, 4, 128, False, c, 0) for c in (0, 1)} <= seen and (HELPERS, 4, 128, False, 0, 1) not in seen


@pytest.mark.parametrize("N,H,conv,deferred,form", [
    # four value heads a key head: two workgroups without conv, helpers between two and four heads per CU in step
    (8, 4, 0, 0, ONE), (32, 4, 0, 0, ONE), (33, 4, 0, 0, HELPERS), (64, 4, 0, 0, HELPERS), (65, 4, 0, 0, ONE),
    (8, 4, 1, 0, HELPERS), (64, 4, 1, 0, HELPERS), (65, 4, 1, 0, ONE),
    # rows at different fills: a flush launch where a row is often due and heads are few
    (4, 4, 0, 1, ONE), (5, 4, 0, 1, TWO), (16, 4, 0, 1, TWO), (17, 4, 0, 1, ONE), (64, 4, 0, 1, ONE),
    (3, 4, 1, 1, HELPERS), (4, 4, 1, 1, TWO), (32, 4, 1, 1, TWO), (33, 4, 1, 1, HELPERS), (65, 4, 1, 1, TWO)])
def test_gqa4_lines(rules, N, H, conv, deferred, form):
    for K in (128, 64):
        assert rules.gdn_decode_form(N, 4 * H, H, K, 128, 4, 16, conv, deferred, 256) == form


def test_wide_ranks_defer_to_a_flush_launch_at_gqa4(rules):
    assert rules.gdn_decode_form(32, 64, 16, 128, 128, 8, 16, 0, 1, 256) == TWO
    assert rules.gdn_decode_form(32, 64, 16, 128, 128, 8, 16, 0, 0, 256) == ONE
    assert rules.gdn_decode_form(32, 32, 16, 128, 128, 8, 16, 0, 1, 256) == ONE


@pytest.mark.parametrize("N,HV,H,L,heads", [
    (32, 32, 32, 16, 1), (33, 32, 32, 16, 2), (64, 32, 32, 64, 2), (65, 32, 32, 64, 0), (65, 32, 32, 33, 0),
    (256, 32, 32, 32, 2), (1024, 32, 32, 16, 2), (60, 17, 17, 16, 1), (61, 17, 17, 16, 0), (9, 32, 16, 16, 2), (9, 32, 8, 16, 0)])
def test_kda_lines(rules, N, HV, H, L, heads):
    assert rules.kda_decode_heads(N, HV, H, L, 256) == heads
