"""Adjoints in recomputed segments: the same bits as with every step's positions
kept, on every path that has segments (MIXED and FP64 handles, both kicks; the
symmetric, one-pass and per-system batches, eager and as a replayed graph), and
no more device memory than the checkpoint interval asks for."""
import numpy as np
import pytest
import torch

import utc_amd as U

pytestmark = pytest.mark.gpu


def segmented(nsteps, ckpt, buffers, row_bytes):
    """Whether positions of row_bytes for each step exceed the checkpoints (64
    bytes) and the segments' buffers (32 a step) of that interval."""
    nck = -(-nsteps // ckpt)
    return row_bytes * nsteps > 64 * nck + 32 * ckpt * buffers


def case(n):
    pos, vel = U.generate(U.GEN_PLUMMER, n, 3)
    return pos, vel, U.generate(U.GEN_TARGETS, n, 5, 0.5)


@pytest.mark.parametrize("kick", [U.KICK_PHYSICAL, U.KICK_REFERENCE])
@pytest.mark.parametrize("prec,n,steps,ckpts", [(U.PREC_MIXED, 700, 100, (10, 7)), (U.PREC_MIXED, 9001, 100, (10, 7)),
                                                (U.PREC_FP64, 700, 41, (5, 6))])
def test_handle(prec, n, steps, ckpts, kick):
    pos, vel, tgt = case(n)
    with U.System(n, prec, 1e-3, 1e-4, kick=kick) as s:
        want = None
        for ckpt in (steps, *ckpts, steps):
            print(f"case: adjoint segments prec={prec} n={n} kick={kick} {steps}/{ckpt}", flush=True)
            assert segmented(steps, ckpt, 2, 16 if prec == U.PREC_MIXED else 32) == (ckpt != steps)
            s.set_state(pos, vel)
            got = s.adjoint(steps, ckpt, tgt)
            want = want or got
            assert np.isfinite(got[1]).all()
            for a, b in zip(got, want):
                assert np.array_equal(a, b), ckpt


@pytest.mark.parametrize("tile,mode", [(5, 0), (4, 0), (5, 2), (2, 0), (2, 2), (2, 1)])
def test_batch(tile, mode):
    sizes, steps = [700, 1024, 250, 1], 100
    both = [U.generate(U.GEN_PLUMMER, n, 3 + n) for n in sizes]
    pos, vel = (np.concatenate([b[k] for b in both]) for k in (0, 1))
    tgt = U.generate(U.GEN_TARGETS, len(pos), 5, 0.5)
    with U.Batch(sizes, 1e-3, 1e-4, tile=tile) as b:
        want = None
        # the second of two equal graph runs replays it; others make the workspace grow in between
        for ckpt in (steps, steps, 10, 10, 7, steps, 10):
            print(f"case: batch adjoint segments tile={tile} mode={mode} {steps}/{ckpt}", flush=True)
            assert segmented(steps, ckpt, 1, 16) == (ckpt != steps)
            b.set_state(pos, vel)
            got = (*b.run(steps, mode, ckpt, tgt)[1:], *b.get_state())
            want = want or got
            for x, y in zip(got, want):
                assert np.array_equal(x, y), ckpt


def test_memory_is_what_the_interval_asks_for():
    n, steps, ckpt = 32768, 100, 10
    pos, vel, tgt = case(n)
    with U.System(n, U.PREC_MIXED, 1e-3, 1e-4) as s:
        s.set_state(pos, vel)
        s.adjoint(1, 1, tgt)  # what does not depend on the steps
        free = torch.cuda.mem_get_info()[0]
        s.adjoint(steps, ckpt, tgt)
        used = free - torch.cuda.mem_get_info()[0]
    # 10 checkpoints of 64 bytes and two buffers of 10 steps of 32 bytes a body;
    # all positions in FP64 would take 3200 bytes a body, 63 MB more
    assert used <= (64 * 10 + 32 * 20) * n + (16 << 20), used
