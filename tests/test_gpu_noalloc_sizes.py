"""utcnb_accel_noalloc at the largest sizes of its symmetric tiles: sym8r64, which
the default is there, is divided up to 46080 bodies and fits the 64 MiB scratch
undivided up to 49152; bitwise the field of a handle, refused above.  The default
beyond: bitwise the slice of all bodies of a symmetric handle, and k2s8 once
those sums no longer fit."""
import ctypes as C

import numpy as np
import pytest
import torch

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [46080, 46081, 49152])
@pytest.mark.parametrize("tile_name", ["default", "sym8r64"])
def test_largest_symmetric_fields(n, tile_name):
    tile = 0 if tile_name == "default" else U.tiles().index(tile_name) + 1
    pos = plummer(n, eps=0.005)["pos"].astype(np.float32)
    x = torch.from_numpy(pos).cuda()
    for prec in (U.PREC_MIXED, U.PREC_FP32):
        print(f"case: noalloc {tile_name} n={n} prec={prec}", flush=True)
        acc = torch.empty((n, 3), dtype=torch.float64, device="cuda")
        U.check(U.lib().utcnb_accel_noalloc(C.c_void_p(x.data_ptr()), n, 2.5e-5, prec, tile, 0,
                                            C.c_void_p(acc.data_ptr()), None), "field")
        torch.cuda.synchronize()
        with U.System(n, prec, 2.5e-5, 1e-3, tile=tile) as s:
            assert s.tile()[1] == "sym8r64"
            s.set_state(pos.astype(np.float64))
            assert np.array_equal(acc.cpu().numpy(), s.accel())


def test_refused_above():
    n, tile = 49153, U.tiles().index("sym8r64") + 1
    x = torch.zeros((n, 4), device="cuda")
    acc = torch.empty((n, 3), dtype=torch.float64, device="cuda")
    assert U.lib().utcnb_accel_noalloc(C.c_void_p(x.data_ptr()), n, 2.5e-5, U.PREC_MIXED, tile, 0,
                                       C.c_void_p(acc.data_ptr()), None) == U.EINVAL
    assert b"64 MiB" in U.lib().utcnb_last_error()


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n", [49153, 85000, 90001])
def test_default_beyond_the_symmetric_sizes(n, prec):
    pos = plummer(n, eps=0.005)["pos"].astype(np.float32)
    x = torch.from_numpy(pos).cuda()
    acc = torch.empty((n, 3), dtype=torch.float64, device="cuda")
    print(f"case: noalloc default n={n} prec={prec}", flush=True)
    U.check(U.lib().utcnb_accel_noalloc(C.c_void_p(x.data_ptr()), n, 2.5e-5, prec, 0, 0, C.c_void_p(acc.data_ptr()),
                                        None), "field")
    torch.cuda.synchronize()
    got = acc.cpu().numpy()
    k2s8 = U.tiles().index("k2s8") + 1
    with U.System(n, prec, 2.5e-5, 1e-3, tile=0 if n < 86000 else k2s8) as s:
        s.set_state(pos.astype(np.float64))
        if n < 86000:
            assert s.slice_tile(n)[1] == "k2p64"
        assert np.array_equal(got, s.accel_slice(0, n))
    rows = np.sort(np.random.default_rng(5).choice(n, 512, replace=False))
    want = O.accel_rows_f64(pos.astype(np.float64), 2.5e-5, rows, nthreads=16)
    # FP32 pair terms at FP32 positions
    assert np.linalg.norm(got[rows] - want) <= 2e-6 * np.linalg.norm(want)
