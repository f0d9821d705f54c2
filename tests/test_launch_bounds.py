"""Launch geometry of every kernel of the built liblq.so against its compiled metadata (CPU; reads the library's own
gfx950 code objects, tests/lq_codeobj.py).

  * the workgroup size each launch site uses (tests/lq_codeobj.LAUNCH_BLOCK, from leapquant_amd/csrc/*.hip) equals the
    kernel's compiled maximum (__launch_bounds__): a kernel is never launched with more threads than its registers
    were allocated for;
  * its static LDS fits a workgroup on a CU (160 KiB), and the workgroups per CU that LDS and registers allow are at
    least one, so every launch can make progress;
  * the kernels of the benchmark's hot path (the one-launch GDN decode, the four-wave GDN and KDA flushes, the KDA
    step) keep the residency they are tuned for (four workgroups per CU for the 256-thread ones, eight for the KDA
    step);
  * so do the other one-launch decodes (GDN and KDA) and the rank-8 flush, whose register spills are bounded.
"""
import os
import shutil

import pytest

from tests import lq_codeobj as C

pytestmark = pytest.mark.skipif(not os.path.exists(C.LIB) or not os.path.exists(C.READELF) or not shutil.which("c++filt"),
                                reason="needs the built liblq.so, llvm-readelf and c++filt")


@pytest.fixture(scope="module")
def kernels():
    ks = C.kernels()
    assert ks, "no gfx950 code object found in liblq.so"
    return ks


def _per_cu(k):
    """Workgroups of kernel k that fit one CU at once (LDS and registers; wave64, four SIMDs)."""
    waves = k["block"] // 64
    regs = -(-(k["vgpr"] + k["agpr"]) // 8) * 8                     # allocation granule of 8
    waves_per_simd = min(8, C.VGPRS_PER_SIMD_LANE // max(regs, 1))
    by_regs = (4 * waves_per_simd) // waves
    by_lds = C.LDS_PER_CU // k["lds"] if k["lds"] else 64
    return min(by_regs, by_lds)


def test_every_kernel_has_a_known_launch_site(kernels):
    fams = {C.family(k["name"]) for k in kernels}
    assert fams <= set(C.LAUNCH_BLOCK), fams - set(C.LAUNCH_BLOCK)


def test_launch_block_equals_the_compiled_bound(kernels):
    bad = [(k["name"], k["block"], C.launch_block(k)) for k in kernels if C.launch_block(k) != k["block"]]
    assert not bad, bad


def test_lds_and_registers_fit(kernels):
    for k in kernels:
        assert k["lds"] <= C.LDS_PER_CU, (k["name"], k["lds"])
        assert k["vgpr"] + k["agpr"] <= C.VGPRS_PER_SIMD_LANE, k["name"]
        assert _per_cu(k) >= 1, k["name"]


def test_hot_kernels_keep_their_residency(kernels):
    def find(pattern):
        hit = [k for k in kernels if pattern in k["name"]]
        assert hit, pattern
        return hit
    for k in find("gdn_step_kernel<128, 128, 2, false, true, 4, false>") + find("flush4_kernel<128, 128, 1, false>"):
        assert _per_cu(k) >= 4 and k["scratch"] <= 8, (k["name"], _per_cu(k), k["scratch"])
    for k in find("flush4_kernel<128, 128, 1, true>"):        # KDA: a few loop-invariant values spilled per head
        assert _per_cu(k) >= 4 and k["scratch"] <= 64, (k["name"], _per_cu(k), k["scratch"])
    for k in find("kda_step_kernel"):
        assert _per_cu(k) >= 8 and k["scratch"] == 0, (k["name"], _per_cu(k), k["scratch"])


# (kernel, workgroups per CU it is launched for, scratch bytes per lane at most)
ONE_LAUNCH = ([("gdn_decode_pair_kernel<%s>" % d, 4, 0) for d in ("128, 128, false", "128, 128, true", "64, 128, false",
                                                                 "64, 128, true", "64, 64, false", "64, 64, true")]
              + [("gdn_decode_split_kernel<%s>" % d, 4, 0) for d in ("128, 128", "64, 128", "64, 64")]
              + [("gdn_decode_wide_kernel<%s, %d, %s>" % (d, g, c), 4 // g, 0) for d in ("128, 128", "64, 128")
                 for g in (1, 2, 4) for c in ("false", "true")]
              + [("gdn_step_kernel<%s, %d, %s, true, 4, false>" % (d, g, c), 8 // g, 0) for d in ("128, 128", "64, 128")
                 for g, c in ((2, "false"), (2, "true"), (4, "true"))]
              + [("gdn_step_kernel<128, 128, 2, %s, true, 4, true>" % c, 4, 0) for c in ("false", "true")]   # deferred
              + [("gdn_step_kernel<128, 128, %d, %s, true, 16, false>" % (g, c), 8 // g, 48) for g in (2, 4)   # rank 8
                 for c in ("false", "true")]
              + [("flush8_kernel<%d>" % m, 4, 48) for m in (0, 1, 2)]
              + [("kda_decode_kernel<%d>" % w, 4, 32) for w in (1, 2)])


@pytest.mark.parametrize("name,per_cu,scratch", ONE_LAUNCH)
def test_one_launch_kernels_keep_their_residency(kernels, name, per_cu, scratch):
    """The one-launch decodes and the rank-8 flush: the residency their launch rules are drawn for, and no more register
    spills than they were measured with."""
    hit = [k for k in kernels if name + "(" in k["name"]]
    assert hit, name
    for k in hit:
        assert _per_cu(k) >= per_cu and k["scratch"] <= scratch, (k["name"], _per_cu(k), k["scratch"])
