"""FP64 steps with 4 to 64 targets per workgroup: sizes on both sides of the
lines between them against the CPU FP64 oracle; slices keep the bits."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 63, 65, 1023, 1024, 1025, 2048, 2049, 3000, 4097, 6001, 8192, 8193, 10000])
def test_field_and_slices(n):
    c = plummer(max(n, 2), eps=0.005)
    pos, vel = c["pos"][:n], c["vel"][:n]
    print(f"case: fp64 n={n}", flush=True)
    with U.System(n, U.PREC_FP64, c["eps"] ** 2, c["dt"]) as s:
        s.set_state(pos, vel)
        full = s.accel()
        if n == 1:
            assert not full.any()
        else:
            # sums of n FP64 terms on both sides, the oracle's uncompensated
            assert relnorm(full, O.accel_f64(pos, c["eps"] ** 2)) <= 1e-13
        for start, count in {(0, 1), (n - 1, 1), (n // 3, n - n // 3), (n // 2, max(1, n // 5))}:
            assert np.array_equal(s.accel_slice(start, count), full[start:start + count]), (start, count)


def test_tiny_and_huge_distances():
    """Distances outside the short inverse-distance form's range."""
    g = np.random.default_rng(3)
    pos = np.ones((700, 4))
    pos[:, :3] = g.normal(0, 1, (700, 3)) * 10.0 ** g.uniform(-120, 120, (700, 1))
    with U.System(700, U.PREC_FP64, 1e-190, 1e-3) as s:  # self pairs: d2 below 2^-600
        s.set_state(pos, np.zeros((700, 4)))
        a = s.accel()
    want = O.accel_f64(pos, 1e-190)
    r = pos[None, :, :3] - pos[:, None, :3]
    inv = 1.0 / np.sqrt((r * r).sum(2) + 1e-190)
    with np.errstate(under="ignore"):
        size = np.abs(r * (inv * inv * inv)[:, :, None]).sum(1)
    assert np.isfinite(a).all() and np.isfinite(size).all()
    # 700 terms, each of a few roundings, added without compensation by the oracle
    assert (np.abs(a - want) <= 710 * 2.0 ** -52 * size).all()
