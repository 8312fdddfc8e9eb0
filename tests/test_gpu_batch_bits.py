"""A system's bits in a symmetric batch are those it has alone, forward and
adjoint, in batches and groups of any size: around 65536 and 131072 bodies, where
the reductions' lanes change, and above."""
import numpy as np
import pytest

import utc_amd as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [4, 5])
@pytest.mark.parametrize("sizes", [[8192] * 15 + [7900], [8192] * 17 + [300], [40000, 3000] + [8192] * 26, [257] * 300])
def test_as_alone(sizes, tile):
    eps2, dt, steps = 1e-4, 1e-3, 3
    both = [U.generate(U.GEN_PLUMMER, n, 3 + k) for k, n in enumerate(sizes)]
    pos, vel = (np.concatenate([b[k] for b in both]) for k in (0, 1))
    tgt = U.generate(U.GEN_TARGETS, len(pos), 5, 0.5)
    print(f"case: batch bits tile={tile} systems={len(sizes)} bodies={len(pos)}", flush=True)
    with U.Batch(sizes, eps2, dt, tile=tile) as b:
        b.set_state(pos, vel)
        out = (*b.run(steps, 0, steps, tgt)[1:], *b.get_state())
    off = np.concatenate([[0], np.cumsum(sizes)])
    for k in sorted({0, 1, len(sizes) // 2, len(sizes) - 1}):
        a, e = off[k], off[k + 1]
        with U.Batch([sizes[k]], eps2, dt, tile=tile) as b:
            b.set_state(pos[a:e], vel[a:e])
            one = (*b.run(steps, 0, steps, tgt[a:e])[1:], *b.get_state())
        assert out[0][k] == one[0][0]
        for x, y in zip(out[1:], one[1:]):
            assert np.array_equal(x[a:e], y), (k, sizes[k])
