"""Symmetric launches of few waves carry the sources round in registers, others
through LDS: tiles on both sides of the line (1024 waves, 2048 with 2 targets per
lane), whole and divided sub-units, equal and unequal masses, against the CPU FP64
oracle; and shares of few wave blocks against the whole step."""
import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [U.PREC_MIXED, U.PREC_FP32])
@pytest.mark.parametrize("name,sizes", [("sym2r32", (2, 1025, 8192, 8193)), ("sym4r4", (2, 1025, 8193)),
                                        ("sym4r64", (1, 4096, 4097)), ("sym8r32", (1025, 8193)),
                                        ("sym2r64x2", (2, 4096, 4097)), ("sym4r64x2", (2, 4096, 4097))])
def test_field(name, sizes, prec):
    for n in sizes:
        c = plummer(max(n, 2), eps=0.005)
        pos = c["pos"][:n].copy()
        for masses in ("equal", "unequal"):
            if masses == "unequal":
                pos[:, 3] *= 10.0 ** np.random.default_rng(3).uniform(-2, 0, n)
            # of the positions the kernels read: their rounding alone moves the field of the 4096 by 2.1e-6
            want = O.accel_f64(pos.astype(np.float32).astype(np.float64), c["eps"] ** 2)
            for flags in (0, U.FLAG_NO_NEWTON):
                print(f"case: registers {name} n={n} prec={prec} {masses} flags={flags}", flush=True)
                with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=U.tiles().index(name) + 1, flags=flags) as s:
                    s.set_state(pos, c["vel"][:n])
                    assert np.linalg.norm(s.accel() - want) <= 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("n,G", [(8193, 64), (16384, 32), (30000, 30)])
def test_shares_of_few_waves(n, G):
    import torch
    c = plummer(n, eps=0.005, dt=5e-4)
    pos = c["pos"].copy()
    pos[:, 3] *= 10.0 ** np.random.default_rng(3).uniform(-2, 0, n)
    print(f"case: shares of few waves n={n} G={G}", flush=True)
    with U.System(n, U.PREC_MIXED, c["eps"] ** 2, c["dt"]) as s:
        s.set_state(pos, c["vel"])
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
        _, v = s.get_state()
    kick = (v[:, :3] - c["vel"][:, :3]) / c["dt"]
    assert relnorm(kick, O.accel_f64(pos.astype(np.float32).astype(np.float64), c["eps"] ** 2)) <= 2e-6
