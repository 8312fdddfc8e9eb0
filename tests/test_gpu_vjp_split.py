"""The symmetric adjoint pair sum with its sub-units shared in chunks of the
rotation (sym_vjp.hip): from two wave blocks to the sizes where the number of
waves per block changes, equal and unequal masses, against the FP64 adjoint."""
import numpy as np
import pytest

import utc_amd as U
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 512, 1024, 1025, 2049, 5000, 8193, 16385, 38913, 39937])
@pytest.mark.parametrize("masses", ["equal", "loguniform"])
def test_against_fp64(n, masses):
    c = plummer(n, eps=0.05, dt=1e-3)
    pos, vel = c["pos"].copy(), c["vel"]
    if masses == "loguniform":
        pos[:, 3] *= 10.0 ** np.random.default_rng(3).uniform(-2, 0, n)
    tgt = np.random.default_rng(5).normal(0, 0.5, (n, 3))
    print(f"case: vjp split n={n} {masses}", flush=True)
    out = {}
    for prec in (U.PREC_MIXED, U.PREC_FP64):
        with U.System(n, prec, c["eps"] ** 2, c["dt"]) as s:
            s.set_state(pos, vel)
            out[prec] = s.adjoint(2, 2, tgt)
    loss, dx, dv, dm = out[U.PREC_MIXED]
    loss64, dx64, dv64, dm64 = out[U.PREC_FP64]
    # the bounds of the symmetric VJP at N = 5000 (test_gpu_adjoint.py): every
    # pair term is FP32 and the mass gradients cancel
    assert abs(loss - loss64) <= 1e-9 * abs(loss64)
    assert relnorm(dx, dx64) <= 1e-5
    assert relnorm(dv, dv64) <= 1e-5
    assert relnorm(dm, dm64) <= 1e-5
