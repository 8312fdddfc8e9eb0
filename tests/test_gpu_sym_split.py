"""Symmetric tiles whose waves share the sub-units in chunks (SymSplit,
sym_reduce.h): from two wave blocks with more waves than chunks to ragged
sizes, equal and unequal masses, against the CPU FP64 oracle; the default
tiles; shares of a default system, whose wave blocks are another tile's."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("n", [2, 513, 1024, 1025, 3000, 8193, 9001])
@pytest.mark.parametrize("name", ["sym8r128", "sym8r64", "sym4r128x4", "sym2r64x2"])
def test_field(name, n, prec):
    c = plummer(n, eps=0.005)
    print(f"case: split tile {name} n={n} prec={prec}", flush=True)
    for seed in (None, 3):
        pos = c["pos"].copy()
        if seed is not None:
            pos[:, 3] *= 10.0 ** np.random.default_rng(seed).uniform(-2, 0, n)
        for flags in (0, U.FLAG_NO_NEWTON):
            with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=U.tiles().index(name) + 1, flags=flags) as s:
                s.set_state(pos, c["vel"])
                # the FP32 positions alone perturb close pairs by ~u|x|/r
                assert relnorm(s.accel(), O.accel_f64(pos, c["eps"] ** 2)) <= 2e-6


@pytest.mark.parametrize("n,name", [(8193, "sym8r128"), (39936, "sym8r128"), (39937, "sym8r64"), (65536, "sym8r64")])
def test_default_tile(n, name):
    """sym8r128 is divided below 40960 bodies (padded), sym8r64 below 65536."""
    for prec in (U.PREC_MIXED, U.PREC_FP32):
        with U.System(n, prec, 1e-4, 1e-3) as s:
            assert s.tile()[1] == name


@pytest.mark.parametrize("n,blocks", [(9001, 72), (16384, 64), (30000, 60)])
def test_shares_of_a_default_system(n, blocks):
    """As many shares as wave blocks of 128 (N < 16384), 256 (< 24576) or 512
    bodies, which add up to the whole step."""
    import torch
    G = blocks
    c = plummer(n, eps=0.005, dt=5e-4)
    with U.System(n, U.PREC_MIXED, c["eps"] ** 2, c["dt"]) as s, \
            U.System(n, U.PREC_MIXED, c["eps"] ** 2, c["dt"]) as full:
        s.set_state(c["pos"], c["vel"])
        full.set_state(c["pos"], c["vel"])
        with pytest.raises(U.UtcnbError):
            s.share_range(G + 1, 0)
        reacts = torch.zeros((G, n, 3), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        for g in range(G):
            s.share_pairs(G, g, reacts[g].data_ptr())
        s.sync()
        total = reacts.sum(0)
        torch.cuda.synchronize()
        for g in range(G):
            start, cnt = s.share_range(G, g)
            if cnt > 0:
                s.share_finish(G, g, total[start:].data_ptr())
        s.sync()
        s.commit_step()
        full.step(1)
        ps, vs = s.get_state()
        pf, vf = full.get_state()
    dv = vf[:, :3] - c["vel"][:, :3]
    # each body's kick is two FP32 evaluations of one sum: 2e-6 as in test_field
    assert np.linalg.norm(vs[:, :3] - vf[:, :3]) <= 2e-6 * np.linalg.norm(dv)
    assert relnorm(ps[:, :3], pf[:, :3]) <= 1e-10
