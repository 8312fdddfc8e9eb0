"""Small-system tiles take sources up to a whole number of their splits' root
groups (256 to 1024 bodies): sizes around those ends against the CPU FP64
oracle, and the default tiles."""
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import plummer, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 255, 256, 257, 511, 512, 513, 768, 769, 1023, 1024, 1025, 1536, 1537, 2047, 2048, 2561,
                               4095, 4097, 4608, 4865, 6145, 7937, 8192])
def test_field(n):
    c = plummer(n, eps=0.005)
    want = O.accel_f64(c["pos"], c["eps"] ** 2)
    for k, name in enumerate(U.tiles()):
        if not name.startswith("sm") or (n + 1023) // 1024 > int(name.split("n")[1][:-1]):
            continue
        for prec in (U.PREC_MIXED, U.PREC_FP32):
            print(f"case: {name} n={n} prec={prec}", flush=True)
            with U.System(n, prec, c["eps"] ** 2, c["dt"], tile=k + 1) as s:
                s.set_state(c["pos"], c["vel"])
                # the FP32 positions alone perturb close pairs by ~u|x|/r
                assert relnorm(s.accel(), want) <= 2e-6


@pytest.mark.parametrize("n,name", [(1024, "sm1t4w8n2k"), (1025, "sm1t8w8n2k"), (2048, "sm1t8w8n2k"),
                                    (2049, "sm1t16w16n4k"), (4097, "sm1t8w16n8k"), (6144, "sm1t8w16n8k"), (6145, "sm2t16w16n8k")])
def test_default_tile(n, name):
    with U.System(n, U.PREC_MIXED, 1e-4, 1e-3) as s:
        assert s.tile()[1] == name
