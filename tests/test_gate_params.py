"""Gate parameters (A_log, dt_bias) in any float dtype: what reaches a decode call is the parameter's present value, in
place updates included, and the outputs are those of the same values in fp32."""
import ctypes

import pytest
import torch

from leapquant_amd import _lib
from leapquant_amd import kernels as KN
from leapquant_amd.state import LeapQuantState

DTYPES = [torch.float32, torch.bfloat16, torch.float16, torch.float64]


class _Recorder:
    """Stands for liblq on the host: reads the gate parameters that a decode call was given at their addresses."""

    def _take(self, st, io, KA):
        st, io = st._obj, io._obj
        def val(p, n, bf):
            if bf:
                raw = torch.tensor(list((ctypes.c_int16 * n).from_address(p)), dtype=torch.int16)
                return raw.view(torch.bfloat16).float()
            return torch.tensor(list((ctypes.c_float * n).from_address(p)))

        self.got = (val(io.A_log, st.HV, io.gate_bf16 & 1), val(io.dt_bias, st.HV * KA, io.gate_bf16 & 2))
        return 0

    def lq_gdn_decode(self, st, io, cv, Q0, stream):
        return self._take(st, io, 1)

    def lq_kda_decode(self, st, io, glb, Q0, stream):
        return self._take(st, io, 128)


def _inputs(N, H, HV, KA, dev):
    bf = lambda *s: torch.randn(*s, device=dev).bfloat16()
    return bf(N, 2 * H * 128 + HV * 128), bf(N, HV, KA), bf(N, HV)


@pytest.mark.parametrize("kda", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
def test_a_decode_call_is_given_the_present_values(monkeypatch, kda, dtype):
    monkeypatch.setattr(KN, "_dev", lambda t: t.data_ptr())
    monkeypatch.setattr(KN, "_raw_stream", lambda t: 0)
    HV, H, KA = 4, 4 if kda else 2, 128 if kda else 1
    lq = LeapQuantState(torch.zeros(3, HV, 128, 128), H, kda=kda)
    lq._lib = rec = _Recorder()
    ssm = torch.zeros(3, HV, 128, 128)
    mixed, a, b = _inputs(2, H, HV, KA, "cpu")
    out = torch.empty(2, HV, 128, dtype=torch.bfloat16)
    idx = torch.tensor([1, 2], dtype=torch.int32)
    A_log, dt = torch.randn(HV).to(dtype), torch.randn(HV * KA).to(dtype)

    def check(A_log, dt):
        lq.decode(ssm, mixed, a, b, A_log, dt, idx, out)
        assert torch.equal(rec.got[0], A_log.float().reshape(-1)) and torch.equal(rec.got[1], dt.float().reshape(-1))

    check(A_log, dt)
    A_log.data.copy_(torch.randn(HV))                  # a weight reload in place
    dt.add_(0.5)
    check(A_log, dt)
    for _ in range(3):                                 # other parameters at an address that the allocator hands out again
        t = torch.randn(HV * KA).to(dtype)
        check(A_log, t)
        del t
    check(A_log.view(1, 1, HV, 1), dt.view(HV, KA))    # as the engine's layers hold them
    check(torch.randn(2 * HV).to(dtype)[::2], torch.randn(HV * KA + 1).to(dtype)[1:])


@pytest.mark.gpu
@pytest.mark.parametrize("kda", [False, True])
@pytest.mark.parametrize("dtype", DTYPES[1:])
@pytest.mark.parametrize("off", [0, 1])
def test_outputs_equal_those_of_fp32_parameters(kda, dtype, off):
    torch.manual_seed(3)
    dev, N, NS, HV = "cuda:0", 3, 5, 6
    H, KA = HV if kda else HV // 2, 128 if kda else 1
    ssm = torch.randn(NS, HV, 128, 128, device=dev) * 0.02
    lq = LeapQuantState(ssm, H, kda=kda, L=2)
    lq.quantize(ssm, torch.arange(1, NS, device=dev))
    ssm2 = ssm.clone()
    lq2 = LeapQuantState(ssm2, H, kda=kda, L=2)
    idx = torch.tensor([2, 1, 4], device=dev, dtype=torch.int32)
    A_log = torch.randn(HV + off, device=dev).to(dtype)[off:]
    dt = torch.randn(HV * KA + off, device=dev).to(dtype)[off:]
    for _ in range(3):
        mixed, a, b = _inputs(N, H, HV, KA, dev)
        o1 = torch.empty(N, HV, 128, device=dev, dtype=torch.bfloat16)
        o2 = torch.empty_like(o1)
        lq.decode(ssm, mixed, a, b, A_log, dt, idx, o1)
        lq2.decode(ssm2, mixed, a, b, A_log.float(), dt.float(), idx, o2)
        torch.cuda.synchronize()
        assert torch.equal(o1, o2) and torch.equal(ssm.view(torch.int32), ssm2.view(torch.int32))
        A_log.data.copy_(torch.randn(HV, device=dev))
        dt.mul_(0.5)


def test_gate_bf16_is_checked():
    """lq_step_io's last field; a value outside its two bits is refused."""
    assert _lib.LqStepIO._fields_[-1][0] == "gate_bf16"
    lib = _lib.lib()
    st = _lib.LqState(ssm=16, slot_stride=4 * 128 * 128, Kbuf=32, Ubuf=48, Wbuf=64, Pbuf=80, Gbuf=96, hcnt=112,
                      NS=8, HV=4, H=2, K=128, V=128, L=16, R=4)
    for bits, rc in ((0, 0), (3, 0), (4, -1), (-1, -1)):
        io = _lib.LqStepIO(mixed=16, a=32, b=48, A_log=64, dt_bias=80, idx=96, out=112, N=0, scale=1.0, gate_bf16=bits)
        assert lib.lq_gdn_step(ctypes.byref(st), ctypes.byref(io), None) == rc
