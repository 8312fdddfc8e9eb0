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


def test_slices_in_the_partial_sums_of_few_waves():
    """sym4r4 has 4 rows of target-side partials, which hold the slice tiles'
    records of a 16th of the bodies: the same bits, in several launches, and no
    device memory for slices beyond those rows in a large system."""
    import torch
    n = 100001
    c = plummer(n, eps=0.005)
    names = ("sym8r64", "sym4r4")
    fields, n_pad = [], (n + 1023) // 1024 * 1024
    for name in names:
        k, rows = int(name[3]), int(name[5:])
        free = torch.cuda.mem_get_info()[0]
        with U.System(n, U.PREC_MIXED, c["eps"] ** 2, c["dt"], tile=U.tiles().index(name) + 1) as s:
            used = free - torch.cuda.mem_get_info()[0]
            blocks = n_pad // (64 * k)
            partials = 12 * (rows * n_pad + blocks * (blocks // 2) * 64 * k)
            # the states (64 n), two snapshots (32 n), scratch (24 n), staging (64 n)
            assert used <= partials + 200 * n_pad + (32 << 20), (used, partials)
            s.set_state(c["pos"], c["vel"])
            print(f"case: slices of {name} n={n}", flush=True)
            fields.append(s.accel_slice(0, n))
            for start, count in U.partition(n, 3):
                assert np.array_equal(s.accel_slice(start, count), fields[-1][start:start + count])
    assert np.array_equal(*fields)
