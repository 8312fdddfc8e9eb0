"""One-pass tiles with the sources in parts over separate waves (force_part.h):
sizes below one wave, at its edges, with fewer 64-source chunks than parts
(empty parts) and ragged ones, against the CPU FP64 oracle; a body's bits do
not depend on the slice; the default slice tile."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 1023, 1025, 8193, 9001])
def test_slices_of_a_symmetric_system(n, prec):
    c = plummer(max(n, 2), eps=0.005)
    pos, vel = c["pos"][:n], c["vel"][:n]
    want = O.accel_f64(pos, c["eps"] ** 2)
    with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=U.tiles().index("sym8r64") + 1) as s:
        s.set_state(pos, vel)
        seen = {}
        for start, count in sorted({(0, n), (0, 1), (n - 1, 1), (0, max(1, n // 2)), (n // 3, n - n // 3),
                                    (n // 2, max(1, n // 5))}):
            name = s.slice_tile(count)[1]
            print(f"case: part tile {name} n={n} prec={prec} slice {start}+{count}", flush=True)
            assert name in ("k1p128", "k2p64")
            got = s.accel_slice(start, count)
            # the FP32 positions alone perturb close pairs by ~u|x|/r
            assert np.linalg.norm(got - want[start:start + count]) <= 2e-6 * np.linalg.norm(want)
            # a body's bits depend on the tile, not on the slice
            have = seen.setdefault(name, np.full((n, 3), np.nan))[start:start + count]
            old = ~np.isnan(have)
            assert np.array_equal(got[old], have[old])
            have[:] = got


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
