"""The default tiles' field is no further from FP64 than that of tiles with
shorter chains of plain FP32 additions: 128 source splits up to 2048 bodies,
2 and 4 targets per lane from 8193 to 24575.

The bound: both errors are root mean squares over the 3 components of at least
1025 bodies in 5 systems, nearly independent, each good to
1/sqrt(2 * 3 * 1025 * 5) = 0.6%, so 1.04 leaves five standard deviations of
their ratio."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n,tile", [(1025, "sm1t8w16n8k"), (1500, "sm1t8w16n8k"), (2048, "sm1t8w16n8k"),
                                    (8193, "sym2r32"), (12288, "sym2r32"), (16384, "sym4r64x2"),
                                    (24575, "sym4r64x2")])
def test_default_against_shorter_chains(n, tile, prec):
    err = {"default": 0.0, tile: 0.0}
    for seed in range(5):
        g = np.random.default_rng(seed)
        pos = np.empty((n, 4), np.float32)
        pos[:, :3] = g.uniform(-1.0, 1.0, (n, 3))
        pos[:, 3] = np.exp(g.uniform(-0.7, 0.7, n)) / n
        rows = np.sort(g.choice(n, min(n, 2048), replace=False))
        want = O.accel_rows_f64(pos.astype(np.float64), 1e-4, rows, nthreads=16)
        for name in err:
            with U.System(n, prec, 1e-4, 1e-3, tile=0 if name == "default" else U.tiles().index(name) + 1) as s:
                s.set_state(pos.astype(np.float64))
                err[name] += float(np.sum((s.accel()[rows] - want) ** 2) / np.sum(want ** 2))
    err = {k: (v / 5) ** 0.5 for k, v in err.items()}
    print(f"case: default error n={n} prec={prec} {err}", flush=True)
    assert err["default"] <= 1.04 * err[tile]
