"""GPU: the one-launch GDN decode (lq_gdn_decode: the step's workgroups flush the heads whose window they fill) against
the step followed by the standalone flush on a copy of the state, byte for byte: every head-dim pair and GQA factor,
window lengths on both sides of a staged half (32 entries), rows whose heads are due together and rows where they stand
at different fills (one head of a pair due, a head found full, none due), padding rows."""
import numpy as np
import pytest
import torch

from tests import lqgpu as G

pytestmark = pytest.mark.gpu


def _state(g, NS, HV, H, K, V, L, R, qmax):
    ssm = torch.zeros(NS, HV, V, K, device=G.DEV).normal_(0.0, 0.02, generator=g)
    lq = G.LeapQuantState(ssm, H, L=L, R=R, qmax=qmax)
    lq.quantize(ssm, torch.arange(1, NS, device=G.DEV))
    # fills: slot 1 all heads L - 1, slot 2 all full but one, slot 3 none due, the others any mix per head
    fill = torch.randint(max(0, L - 3), L + 1, (NS, HV), generator=g, device=G.DEV, dtype=torch.int32)
    fill[1] = L - 1
    fill[2] = L
    fill[2, HV - 1] = max(0, L - 2)
    fill[3] = max(0, L - 2)
    lq.hcnt.copy_(fill)
    j = torch.arange(L, device=G.DEV)
    lq.Wbuf.copy_(torch.rand(NS, HV, L, device=G.DEV, generator=g) * (j < fill[..., None]))
    lq.Pbuf.copy_(torch.rand(lq.Pbuf.shape, device=G.DEV, generator=g))
    lq.Kbuf.copy_(torch.randn(lq.Kbuf.shape, device=G.DEV, generator=g) * 0.09)
    lq.Ubuf.copy_(torch.randn(lq.Ubuf.shape, device=G.DEV, generator=g) * 0.5)
    return ssm, lq


@pytest.mark.parametrize("K,V", [(128, 128), (64, 128), (64, 64)])
@pytest.mark.parametrize("GQA", [1, 2, 4])
@pytest.mark.parametrize("L,R,qmax", [(16, 4, 127.0), (33, 3, 31.0), (64, 4, 127.0), (1, 1, 127.0)])
def test_one_launch_equals_step_then_flush(K, V, GQA, L, R, qmax):
    g = torch.Generator(device=G.DEV)
    g.manual_seed(K + V + GQA + L)
    NS, H = 9, 4
    HV = H * GQA
    ssm, lq = _state(g, NS, HV, H, K, V, L, R, qmax)
    ssm2 = ssm.clone()
    lq2 = G.LeapQuantState(ssm2, H, L=L, R=R, qmax=qmax)
    for k in ("hcnt", "Wbuf", "Pbuf", "Kbuf", "Ubuf"):
        getattr(lq2, k).copy_(getattr(lq, k))
    lq2.ctl[0] = 1                                      # heads found full are due too (the scan's flag is theirs)
    idx = torch.tensor([3, 1, 0, 8, 2, -1, 5, 4, 7, NS + 3], device=G.DEV, dtype=torch.int32)
    N = len(idx)
    bf = lambda *s: torch.randn(*s, device=G.DEV, generator=g).bfloat16()
    for _ in range(2):                                  # the second call steps the windows the first has reset
        mixed, a, b = bf(N, 2 * H * K + HV * V), bf(N, HV), bf(N, HV)
        A_log, dt_bias = torch.zeros(HV, device=G.DEV), torch.zeros(HV, device=G.DEV)
        o1 = torch.empty(N, HV, V, device=G.DEV, dtype=torch.bfloat16)
        o2 = torch.empty_like(o1)
        lq.decode(ssm, mixed, a, b, A_log, dt_bias, idx, o1)
        v = lq2.views(ssm2)
        lq2.kstep(v["q32"], v["Sk"], v["Sv"], v["skv"], lq2.Kbuf, lq2.Ubuf, lq2.Wbuf, lq2.Pbuf, lq2.hcnt, mixed, a, b,
                  A_log, dt_bias, v["uq"], idx, o2)
        lq2.flush(ssm2, idx)
        torch.cuda.synchronize()
        assert torch.equal(o1, o2)
        assert torch.equal(ssm.view(torch.int32), ssm2.view(torch.int32))
        for k in ("hcnt", "Wbuf", "Pbuf", "Kbuf", "Ubuf"):
            assert torch.equal(getattr(lq, k), getattr(lq2, k)), k
        assert int((lq.hcnt[idx[(idx > 0) & (idx < NS)].long()] >= L).sum()) == 0
