"""GPU: the one-launch decodes (lq_gdn_decode, lq_kda_decode: the step's workgroups flush the heads whose window they
fill) against the step followed by the standalone flush on a copy of the state, byte for byte: every head-dim pair and
GQA factor, window lengths on both sides of a staged half (32 entries), rows whose heads are due together and rows where
they stand at different fills (one head of a pair due, a head found full, none due), padding rows; launches of up to two
and up to four heads per CU, some of whose workgroups have helper waves, and larger ones; the same with the conv1d update
in the step."""
import ctypes

import pytest
import torch

from leapquant_amd import _lib
from leapquant_amd import kernels as KN
from tests import lqgpu as G

pytestmark = pytest.mark.gpu


def _state(g, NS, HV, H, K, V, L, R, qmax, kda=False, glb=0.0):
    ssm = torch.zeros(NS, HV, V, K, device=G.DEV).normal_(0.0, 0.02, generator=g)
    lq = G.LeapQuantState(ssm, H, kda=kda, gate_lower_bound=glb, L=L, R=R, qmax=qmax)
    lq.quantize(ssm, torch.arange(1, NS, device=G.DEV))
    # fills: slot 1 all heads L - 1, slot 2 all full but one, slot 3 none due, the others any mix over the key heads, with
    # some heads full.  The value heads of a key head share one fill, as their buffered keys do (include/lq.h); full heads
    # beside others only where one workgroup steps the whole key head, on both sides of the comparison (GDN at GQA 1 and
    # 2): elsewhere a head appends over a row that another one, with another fill after the first call, is reading
    fill = torch.randint(max(0, L - 3), L, (NS, H, 1), generator=g, device=G.DEV).expand(NS, H, HV // H).reshape(NS, HV)
    full = torch.rand(NS, HV, device=G.DEV, generator=g) < 0.25
    if HV // H == 4 or (kda and HV > H):
        full = full.view(NS, H, HV // H)[:, :, :1].expand(NS, H, HV // H).reshape(NS, HV)
    fill = torch.where(full, L, fill).int()
    fill[1] = L - 1
    fill[2] = L
    fill[2, HV - HV // H:] = max(0, L - 2)
    fill[3] = max(0, L - 2)
    lq.hcnt.copy_(fill)
    j = torch.arange(L, device=G.DEV)
    lq.Wbuf.copy_(torch.rand(NS, HV, L, device=G.DEV, generator=g) * (j < fill[..., None]))
    lq.Pbuf.copy_(torch.rand(lq.Pbuf.shape, device=G.DEV, generator=g) * (-1.0 if kda else 1.0))
    if kda:                                             # decays below 1, 1 past the fill
        e = 0.8 + 0.2 * torch.rand(lq.Gbuf.shape, device=G.DEV, generator=g)
        lq.Gbuf.copy_(torch.where((j < fill[..., None])[..., None], e, torch.ones_like(e)))
    lq.Kbuf.copy_(torch.randn(lq.Kbuf.shape, device=G.DEV, generator=g) * 0.09)
    lq.Ubuf.copy_(torch.randn(lq.Ubuf.shape, device=G.DEV, generator=g) * 0.5)
    return ssm, lq


def _step(lq, ssm, mixed, a, b, A_log, dt_bias, idx, out, conv):
    """The step alone, with the conv update in it if conv = (conv_state, weight, bias)."""
    if conv is None:
        v = lq.views(ssm)
        lq.kstep(v["q32"], v["Sk"], v["Sv"], v["skv"], lq.Kbuf, lq.Ubuf, lq.Wbuf, lq.Pbuf,
                 *((lq.Gbuf,) if lq.kda else ()), lq.hcnt, mixed, a, b, A_log, dt_bias, v["uq"], idx, out)
        return
    st, cv = lq._struct(ssm), KN.conv_struct(*conv)
    io = KN._step_io(mixed, a, b, A_log, dt_bias, idx, out, lq.kstep_scale)
    _lib.check(_lib.lib().lq_gdn_step_conv(ctypes.byref(st), ctypes.byref(io), ctypes.byref(cv), KN._stream(mixed)),
               "lq_gdn_step_conv")


def _check(g, lq, ssm, H, N, rest, with_conv=False):
    """Two decode calls (the second steps the windows that the first has reset) of N rows, padding rows among them,
    against step + flush on a copy of the state; with_conv: decode_conv, the conv states compared as well."""
    NS, HV, K, V, L = lq.NS, lq.HV, lq.K, lq.V, lq.L
    ssm2 = ssm.clone()
    lq2 = G.LeapQuantState(ssm2, H, L=L, **rest)
    bufs = ("hcnt", "Wbuf", "Pbuf", "Kbuf", "Ubuf") + (("Gbuf",) if lq.kda else ())
    for k in bufs:
        getattr(lq2, k).copy_(getattr(lq, k))
    idx = (torch.randperm(NS - 1, device=G.DEV, generator=g)[:N] + 1).int()
    idx[:5] = torch.tensor([3, 0, 1, -1, NS + 3], device=G.DEV)
    idx[5:] = idx[5:][torch.randperm(N - 5, device=G.DEV, generator=g)]
    idx[5:] = torch.where((idx[5:] == 3) | (idx[5:] == 1), torch.zeros_like(idx[5:]), idx[5:])
    bf = lambda *s: torch.randn(*s, device=G.DEV, generator=g).bfloat16()
    KA = K if lq.kda else 1
    A_log, dt_bias = torch.zeros(HV, device=G.DEV), torch.zeros(HV * KA, device=G.DEV)
    C = 2 * H * K + HV * V
    conv = conv2 = None
    if with_conv:                                       # [NS, C, 3] as vLLM's transposed layout holds it
        conv = (bf(NS, 3, C).transpose(1, 2), bf(C, 4) * 0.5, bf(C) * 0.1)
        conv2 = (conv[0].clone(),) + conv[1:]
    for _ in range(2):
        mixed, a, b = bf(N, C), bf(N, HV, KA), bf(N, HV)
        o1 = torch.empty(N, HV, V, device=G.DEV, dtype=torch.bfloat16)
        o2 = torch.empty_like(o1)
        if with_conv:
            lq.decode_conv(ssm, mixed, *conv, True, a, b, A_log, dt_bias, idx, o1)
        else:
            lq.decode(ssm, mixed, a, b, A_log, dt_bias, idx, o1)
        _step(lq2, ssm2, mixed, a, b, A_log, dt_bias, idx, o2, conv2)
        lq2.flush(ssm2, idx)
        torch.cuda.synchronize()
        assert torch.equal(o1, o2)
        assert not with_conv or torch.equal(conv[0], conv2[0])
        assert torch.equal(ssm.view(torch.int32), ssm2.view(torch.int32))
        for k in bufs:
            assert torch.equal(getattr(lq, k), getattr(lq2, k)), k
        assert int((lq.hcnt[idx[(idx > 0) & (idx < NS)].long()] >= L).sum()) == 0


@pytest.mark.parametrize("K,V", [(128, 128), (64, 128), (64, 64)])
@pytest.mark.parametrize("GQA", [1, 2, 4])
@pytest.mark.parametrize("L,R,qmax", [(16, 4, 127.0), (33, 3, 31.0), (64, 4, 127.0), (1, 1, 127.0)])
@pytest.mark.parametrize("heads", [100, 700, 1100])
def test_gdn_one_launch_equals_step_then_flush(K, V, GQA, L, R, qmax, heads):
    g = torch.Generator(device=G.DEV)
    g.manual_seed(K + V + GQA + L + heads)
    H = 3 if (GQA, heads) == (1, 100) else 4            # an odd number of key heads at GQA 1
    N = max(9, heads // (H * GQA) + 1)
    ssm, lq = _state(g, N + 4, H * GQA, H, K, V, L, R, qmax)
    _check(g, lq, ssm, H, N, dict(R=R, qmax=qmax))


@pytest.mark.parametrize("K,V", [(128, 128), (64, 128), (64, 64)])
@pytest.mark.parametrize("GQA", [1, 2, 4])
@pytest.mark.parametrize("L,R,qmax", [(16, 4, 127.0), (33, 3, 31.0)])
@pytest.mark.parametrize("heads", [100, 700, 1100])
def test_gdn_one_launch_with_conv_equals_step_then_flush(K, V, GQA, L, R, qmax, heads):
    g = torch.Generator(device=G.DEV)
    g.manual_seed(K + V + GQA + L + heads + 1)
    H = 3 if (GQA, heads) == (1, 100) else 4
    N = max(9, heads // (H * GQA) + 1)
    ssm, lq = _state(g, N + 4, H * GQA, H, K, V, L, R, qmax)
    _check(g, lq, ssm, H, N, dict(R=R, qmax=qmax), with_conv=True)


@pytest.mark.parametrize("conv", [False, True])
@pytest.mark.parametrize("R,V,heads", [(4, 128, 100), (4, 128, 700), (4, 128, 1100), (4, 64, 1100), (8, 128, 400)])
def test_deferred_entry_at_gqa4(R, V, heads, conv):
    """HV = 4 H: the deferred entry leaves no head full; its calls, in one launch or two, equal step then flush."""
    g = torch.Generator(device=G.DEV)
    g.manual_seed(R + V + heads)
    H, N, K = 4, heads // 16 + 1, 64 if V == 64 else 128
    ssm, lq = _state(g, N + 4, 4 * H, H, K, V, 16, R, 127.0)
    lq.defer_flush = True
    _check(g, lq, ssm, H, N, dict(R=R), with_conv=conv)


@pytest.mark.parametrize("conv", [False, True])
@pytest.mark.parametrize("GQA,L,R", [(1, 16, 8), (2, 16, 8), (2, 33, 8), (2, 64, 8), (4, 16, 8), (4, 64, 8)])
def test_rank8_one_launch_equals_step_then_flush(GQA, L, R, conv):
    g = torch.Generator(device=G.DEV)
    g.manual_seed(GQA + L + R)
    H, N = 3, 30
    ssm, lq = _state(g, N + 4, H * GQA, H, 128, 128, L, R, 127.0)
    _check(g, lq, ssm, H, N, dict(R=R), with_conv=conv)


@pytest.mark.parametrize("L,R,glb", [(16, 4, 0.0), (33, 2, -5.0), (64, 4, 0.0), (1, 1, 0.0)])
@pytest.mark.parametrize("HV,H,heads", [(3, 3, 100), (8, 4, 1100), (5, 5, 1100), (16, 16, 4200),
                                        # value heads sharing a key head, on both sides of four heads per CU
                                        (8, 4, 100), (6, 2, 100), (6, 2, 1100), (8, 2, 100), (8, 2, 1100)])
def test_kda_one_launch_equals_step_then_flush(HV, H, heads, L, R, glb):
    g = torch.Generator(device=G.DEV)
    g.manual_seed(HV + L + heads)
    N = heads // HV + 1
    ssm, lq = _state(g, N + 4, HV, H, 128, 128, L, R, 127.0, kda=True, glb=glb)
    _check(g, lq, ssm, H, N, dict(R=R, kda=True, gate_lower_bound=glb))


@pytest.mark.parametrize("N", [64, 70, 130])
def test_kda_rows_rotated(N):
    """Two heads per workgroup and 16 workgroups a row at a window of 16: the rounds of 256 workgroups take their rows
    rotated, with whole and partial rounds."""
    g = torch.Generator(device=G.DEV)
    g.manual_seed(N)
    ssm, lq = _state(g, N + 4, 32, 32, 128, 128, 16, 4, 127.0, kda=True)
    _check(g, lq, ssm, 32, N, dict(R=4, kda=True))


def test_deferred_decode_of_a_large_batch():
    """More than a round of 256 workgroups at a window whose rows are taken rotated: the deferred decode's outputs are the
    immediate one's, and the states agree once the deferred heads are flushed."""
    g = torch.Generator(device=G.DEV)
    g.manual_seed(70)
    NS, HV, H, L, N = 75, 8, 4, 16, 70
    ssm, lq = _state(g, NS, HV, H, 128, 128, L, 4, 127.0)
    lq.hcnt.copy_((torch.arange(NS, device=G.DEV) % L)[:, None].expand(NS, HV))
    ssm2 = ssm.clone()
    lq2 = G.LeapQuantState(ssm2, H, L=L, defer_flush=True)
    for k in ("hcnt", "Wbuf", "Pbuf", "Kbuf", "Ubuf"):
        getattr(lq2, k).copy_(getattr(lq, k))
    idx = (torch.randperm(NS - 1, device=G.DEV, generator=g)[:N] + 1).int()
    bf = lambda *s: torch.randn(*s, device=G.DEV, generator=g).bfloat16()
    A_log, dt_bias = torch.zeros(HV, device=G.DEV), torch.zeros(HV, device=G.DEV)
    for _ in range(4):
        mixed, a, b = bf(N, 2 * H * 128 + HV * 128), bf(N, HV), bf(N, HV)
        o1 = torch.empty(N, HV, 128, device=G.DEV, dtype=torch.bfloat16)
        o2 = torch.empty_like(o1)
        lq.decode(ssm, mixed, a, b, A_log, dt_bias, idx, o1)
        lq2.decode(ssm2, mixed, a, b, A_log, dt_bias, idx, o2)
        torch.cuda.synchronize()
        assert torch.equal(o1, o2)
    lq2.flush(ssm2, idx)
    torch.cuda.synchronize()
    assert torch.equal(ssm.view(torch.int32), ssm2.view(torch.int32)) and torch.equal(lq.hcnt, lq2.hcnt)
