"""State set from and read into device arrays: one launch where the arrays are
the handle's device's memory on 16 bytes and apart, the runtime's copies
elsewhere; both the same bits as through the host."""
import ctypes as C

import numpy as np
import pytest
import torch

import utc_amd as U
from tests.nbcases import plummer

pytestmark = pytest.mark.gpu
HANDLES = [(U.PREC_MIXED, U.F64), (U.PREC_FP32, U.F32), (U.PREC_FP64, U.F64), (U.PREC_REFERENCE, U.F32),
           (U.PREC_REFERENCE, U.F64)]


def ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("prec,state", HANDLES)
@pytest.mark.parametrize("n", [1, 255, 256, 257, 3000])
@pytest.mark.parametrize("io", [U.F32, U.F64])
@pytest.mark.parametrize("off", [0, 1])
def test_device_arrays(prec, state, n, io, off):
    """off: one element past 16 bytes, which the copies serve."""
    c = plummer(max(n, 2), eps=0.005)
    dt, tt = (np.float32, torch.float32) if io == U.F32 else (np.float64, torch.float64)
    pos, vel = (np.ascontiguousarray(c[k][:n]).astype(dt) for k in ("pos", "vel"))
    print(f"case: device state prec={prec} n={n} io={io} off={off}", flush=True)
    L = U.lib()
    kick = U.KICK_REFERENCE if prec == U.PREC_REFERENCE else U.KICK_PHYSICAL

    def dev(a):
        t = torch.empty(4 * n + off, dtype=tt, device="cuda")
        t[off:].copy_(torch.from_numpy(a.reshape(-1)))
        return t[off:]

    with U.System(n, prec, c["eps"] ** 2, c["dt"], state_dtype=state, kick=kick) as s:
        U.check(L.utcnb_set_state(s.h, pos.ctypes.data_as(C.c_void_p), vel.ctypes.data_as(C.c_void_p), io, U.HOST), "set")
        s.step(2)
        want, wantv = np.empty_like(pos), np.empty_like(vel)
        U.check(L.utcnb_get_state(s.h, want.ctypes.data_as(C.c_void_p), wantv.ctypes.data_as(C.c_void_p), io, U.HOST),
                "get")
        x, v = dev(pos), dev(vel)
        torch.cuda.synchronize()
        U.check(L.utcnb_set_state(s.h, ptr(x), ptr(v), io, U.DEVICE), "set")
        s.step(2)
        x.zero_(), v.zero_()
        torch.cuda.synchronize()
        for both in (True, False):
            U.check(L.utcnb_get_state(s.h, ptr(x), ptr(v) if both else None, io, U.DEVICE), "get")
            s.sync()
            assert np.array_equal(x.cpu().numpy().reshape(n, 4), want)
            assert np.array_equal(v.cpu().numpy().reshape(n, 4), wantv)


def test_own_buffer_as_input():
    """The handle's own position buffer as the positions: the other buffer
    (one step in) or the one the state is set into (two)."""
    n = 3000
    c = plummer(n, eps=0.005)
    with U.System(n, U.PREC_FP32, c["eps"] ** 2, c["dt"]) as s:
        for steps in (1, 2):
            s.set_state(c["pos"], c["vel"])
            s.step(steps)
            want, wantv = s.get_state(np.float32)
            v = torch.from_numpy(wantv).cuda()
            torch.cuda.synchronize()
            p, dtype = s.position_buffer(0)
            assert dtype == U.F32
            U.check(U.lib().utcnb_set_state(s.h, C.c_void_p(p), ptr(v), U.F32, U.DEVICE), "set")
            got, gotv = s.get_state(np.float32)
            assert np.array_equal(got, want) and np.array_equal(gotv, wantv)
