"""utcnb_accel_noalloc on the small-system tiles reads the caller's bodies
without a padded copy: bitwise the field of a handle at the edges of a wave's
load and of the padding, and where the copy is still needed (a result over its
own input, bodies off 16 bytes)."""
import ctypes as C

import numpy as np
import pytest
import torch

import utc_amd as U
from tests.nbcases import plummer

pytestmark = pytest.mark.gpu


def field(pos_ptr, n, eps2, prec, tile, acc_ptr):
    U.check(U.lib().utcnb_accel_noalloc(C.c_void_p(pos_ptr), n, eps2, prec, tile, 0, C.c_void_p(acc_ptr), None), "field")
    torch.cuda.synchronize()


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("tile", [k + 1 for k, t in enumerate(U.tiles()) if t.startswith("sm")])
def test_bitwise_the_handle_field(tile, prec):
    cap = int(U.tiles()[tile - 1].split("n")[1][:-1]) * 1024
    for n in (1, 2, 63, 64, 65, 1000, 1023, 1024, 1025, cap - 1, cap):
        print(f"case: noalloc tile={U.tiles()[tile - 1]} prec={prec} n={n}", flush=True)
        c = plummer(max(n, 2), eps=0.005)
        pos = c["pos"][:n].astype(np.float32)
        with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=tile) as s:
            s.set_state(pos.astype(np.float64), c["vel"][:n])
            want = s.accel()
        # NaN beyond the n bodies: nothing of it may be read
        buf = torch.full((4 * n + 5,), float("nan"), device="cuda")
        acc = torch.empty((n, 3), dtype=torch.float64, device="cuda")
        for off in (0, 1):  # on and off 16 bytes
            x = buf[off:off + 4 * n]
            x.copy_(torch.from_numpy(pos.reshape(-1)))
            field(x.data_ptr(), n, c["eps"] ** 2, prec, tile, acc.data_ptr())
            assert np.array_equal(acc.cpu().numpy(), want), (n, off)
        # the result over its own input
        over = torch.empty((n, 3), dtype=torch.float64, device="cuda")
        over.view(torch.float32).reshape(-1)[2 * n:].copy_(torch.from_numpy(pos.reshape(-1)))
        start = over.data_ptr() + 8 * n
        if start % 16 == 0:
            field(start, n, c["eps"] ** 2, prec, tile, over.data_ptr())
            assert np.array_equal(over.cpu().numpy(), want), n
