"""One-pass tiles with the sources in parts over separate waves (force_part.h):
sizes below one wave, at its edges, with fewer 64-source chunks than parts
(empty parts) and ragged ones, against the CPU FP64 oracle; slices of every
kind of start give the full field's bits; the default slice tile."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


def tile_id(name):
    return U.tiles().index(name) + 1


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 1023, 1025, 8193, 9001])
@pytest.mark.parametrize("name", ["k1p128", "k2p64"])
def test_field_and_slices(name, n, prec):
    c = plummer(max(n, 2), eps=0.005)
    pos, vel = c["pos"][:n], c["vel"][:n]
    print(f"case: part tile {name} n={n} prec={prec}", flush=True)
    with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=tile_id(name)) as s:
        s.set_state(pos, vel)
        full = s.accel()
        if n == 1:
            assert not full.any()
        else:
            # the FP32 positions alone perturb close pairs by ~u|x|/r
            assert relnorm(full, O.accel_f64(pos, c["eps"] ** 2)) <= 2e-6
        for start, count in {(0, 1), (n - 1, 1), (n // 3, n - n // 3), (n // 2, max(1, n // 5))}:
            assert np.array_equal(s.accel_slice(start, count), full[start:start + count]), (start, count)


def test_default_slice_tile_of_a_symmetric_system():
    """A symmetric handle's slices take the part tiles while its target-side
    partials can hold their records (64 rows: 128 parts for up to half the
    bodies), whatever the count, and agree with the whole symmetric field."""
    n = 9001
    c = plummer(n, eps=0.005)
    with U.System(n, U.PREC_MIXED, c["eps"] ** 2, c["dt"]) as s:
        assert s.tile()[1].startswith("sym")
        assert s.slice_tile(1)[1] == s.slice_tile(n // 2)[1] == "k1p128"
        assert s.slice_tile(n)[1] == "k2p64"
        s.set_state(c["pos"], c["vel"])
        full = s.accel()
        for start, count in U.partition(n, 3) + [(0, n)]:
            assert relnorm(s.accel_slice(start, count), full[start:start + count]) <= 1e-6
        assert np.array_equal(s.accel(), full)  # the slices leave nothing behind
