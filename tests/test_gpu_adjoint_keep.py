"""The adjoint keeps every step's positions while they fit 1 GiB and recomputes
segments beyond that: a trajectory just past it (4200 steps of 8192 bodies,
32 bytes each) gives the same bits with recomputed segments (an uneven last
one among them) as with the whole trajectory kept, which a checkpoint interval
of all steps asks for."""
import numpy as np
import pytest

import utc_amd as U

pytestmark = pytest.mark.gpu

STEPS = 4200


def case(n):
    pos, vel = U.generate(U.GEN_PLUMMER, n, 3)
    return pos, vel, U.generate(U.GEN_TARGETS, n, 5, 0.5)


@pytest.mark.parametrize("kick", [U.KICK_PHYSICAL, U.KICK_REFERENCE])
def test_single_system(kick):
    n = 8192
    assert n * 32 * STEPS > 1 << 30
    pos, vel, tgt = case(n)
    outs = []
    with U.System(n, U.PREC_MIXED, 1e-3, 1e-5, kick=kick, flags=U.FLAG_NO_NEWTON) as s:
        for ckpt in (STEPS, 1300):
            print(f"case: adjoint {STEPS} steps checkpoint every {ckpt} kick={kick}", flush=True)
            s.set_state(pos, vel)
            outs.append(s.adjoint(STEPS, ckpt, tgt))
    assert np.isfinite(outs[0][1]).all()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_batch():
    sizes = [5000, 3001, 250]
    assert sum(sizes) * 32 * STEPS > 1 << 30
    both = [U.generate(U.GEN_PLUMMER, n, 3 + n) for n in sizes]
    pos, vel = (np.concatenate([b[k] for b in both]) for k in (0, 1))
    tgt = U.generate(U.GEN_TARGETS, len(pos), 5, 0.5)
    outs = []
    with U.Batch(sizes, 1e-3, 1e-5, tile=5) as b:
        for ckpt in (STEPS, 1300):
            print(f"case: batch adjoint {STEPS} steps checkpoint every {ckpt}", flush=True)
            b.set_state(pos, vel)
            outs.append(b.run(STEPS, 2, ckpt, tgt)[1:])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
