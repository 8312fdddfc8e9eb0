"""Slices of a symmetric system: a body's bits depend neither on the slice's size
nor on which of the two slice tiles its size selects, across 65536 targets."""
import numpy as np
import pytest

import utc_amd as U
from tests.nbcases import plummer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n", [2, 65, 1025, 9001, 140001])
def test_any_slicing_gives_the_same_bits(n, prec):
    c = plummer(n, eps=0.005)
    tile = 0 if n > 8192 else U.tiles().index("sym8r64") + 1
    with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=tile) as s:
        s.set_state(c["pos"], c["vel"])
        whole = s.accel_slice(0, n)
        for shares in (2, 5):
            names = set()
            for start, count in U.partition(n, shares):
                if count == 0:
                    continue
                names.add(s.slice_tile(count)[1])
                print(f"case: slice bits n={n} prec={prec} {start}+{count} {names}", flush=True)
                assert np.array_equal(s.accel_slice(start, count), whole[start:start + count])
            assert names == {"k1p128"} and s.slice_tile(n)[1] == "k2p64" or n < 128
