"""The symmetric batch's items shrink with the batch (one sub-unit below 131072
bodies in all, 6 below 262144, else 8) and one stream serves it below 65536: a
batch on each side of each line against the one-pass kernels, one system too
large for single sub-units among them, and a batch of up to 131072 bodies
bitwise the systems alone."""
import numpy as np
import pytest

import utc_amd as U

pytestmark = pytest.mark.gpu


def systems(sizes):
    both = [U.generate(U.GEN_PLUMMER, n, 3 + k) for k, n in enumerate(sizes)]
    pos, vel = (np.concatenate([b[k] for b in both]) for k in (0, 1))
    return pos, vel, U.generate(U.GEN_TARGETS, len(pos), 5, 0.5)


@pytest.mark.parametrize("tile", [4, 5])
@pytest.mark.parametrize("sizes", [[1], [255, 257], [8192] * 7 + [7900], [8192] * 8, [8192] * 15 + [7000, 900],
                                   [8192] * 16, [20000] + [4096] * 40, [40000], [1000] * 300])
def test_against_one_pass(tile, sizes):
    eps2, dt, steps = 1e-4, 1e-3, 2
    pos, vel, tgt = systems(sizes)
    print(f"case: batch items tile={tile} total={len(pos)}", flush=True)
    out = {}
    for t in (tile, 2):
        with U.Batch(sizes, eps2, dt, tile=t) as b:
            b.set_state(pos, vel)
            r = b.run(steps, mode=0, ckpt_every=1, target3=tgt)
            out[t] = (*b.get_state(), *r[2:])
    # each is within 1e-9 (positions) and 1e-5 (gradients) of FP64
    # (test_gpu_batch.py); in product form, as a lone body sits at 0
    for k, tol in ((0, 2e-9), (2, 2e-5), (3, 2e-5), (4, 2e-5)):
        a, b = out[tile][k], out[2][k]
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), k


def test_systems_keep_their_bits():
    sizes = [8192, 300, 5000, 1024, 8000, 1, 700]
    pos, vel, _ = systems(sizes)
    with U.Batch(sizes, 1e-4, 1e-3, tile=5) as b:
        b.set_state(pos, vel)
        b.run(3)
        p, v = b.get_state()
    o = 0
    for n in sizes:
        with U.Batch([n], 1e-4, 1e-3, tile=5) as b:
            b.set_state(pos[o:o + n], vel[o:o + n])
            b.run(3)
            p1, v1 = b.get_state()
        assert np.array_equal(p[o:o + n], p1) and np.array_equal(v[o:o + n], v1), n
        o += n
