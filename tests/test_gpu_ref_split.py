"""Reference arithmetic with the terms by many waves and the sums by one
(ref_split_kernel) against the oracle, bit for bit: sizes at the edges of the
16- and 32-target workgroups, of the batches of sources (128, 192 and 96 for
FP32; 96 and 48 for FP64) and of the size classes; slices; squared distances
that are powers of four, infinite and NaN; and the group inverse distance on
every float."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import utc_amd as U
from oracle import oracle as O
from tests.nbcases import cube4096

pytestmark = pytest.mark.gpu


def system(n, T, eps2, dt=1e-3):
    return U.System(n, U.PREC_REFERENCE, float(eps2), float(T(dt)), 1.0, kick=U.KICK_REFERENCE,
                    state_dtype=U.F32 if T == np.float32 else U.F64)


def rows_want(pos, eps2, T):
    return O.gravitation_f32(pos, eps2) if T == np.float32 else O.gravitation_f64(pos, eps2)


def test_group_inverse_distance_exhaustive():
    exe = Path(__file__).resolve().parent / "device" / "_bin" / "probe_invdist_group"
    assert exe.exists(), "build first: python -m utc_amd.build"
    print("case: probe_invdist_group (all floats 2^-96..inf)", flush=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    out = r.stdout.split()
    print(r.stdout, flush=True)
    assert r.returncode == 0
    v = dict(zip(out[::2], out[1::2]))
    assert v["mismatches"] == "0" and v["group_mismatches"] == "0"
    assert int(v["checked"]) == 0x7F800000 - 0x0F800000 + 1


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 47, 48, 49, 95, 97, 127, 128, 129, 191, 193, 383, 385, 4097])
def test_steps_bit_exact(n, T):
    c = cube4096(n=n)
    pos, vel = c["pos"].astype(T), c["vel"].astype(T)
    eps2 = T(c["eps"]) * T(c["eps"])
    print(f"case: ref split n={n} {np.dtype(T).name}", flush=True)
    with system(n, T, eps2, c["dt"]) as s:
        s.set_state(pos, vel)
        s.step(2)
        gp, gv = s.get_state(T)
    run = O.run_f32 if T == np.float32 else O.run_f64
    op, ov = run(pos, vel, 2, eps2, 1.0, T(c["dt"]), nthreads=8)
    assert np.array_equal(gp, op) and np.array_equal(gv, ov)


@pytest.mark.parametrize("T,n", [(np.float32, 8193), (np.float32, 16385), (np.float64, 8193)])
def test_size_classes_and_slices_bit_exact(T, n):
    """A size of each class (the whole system) and slices that take the others:
    every slice gives the whole field's rows, and 64 of them the oracle's."""
    c = cube4096(n=n)
    pos = c["pos"].astype(T)
    eps2 = T(c["eps"]) * T(c["eps"])
    print(f"case: ref split classes n={n} {np.dtype(T).name}", flush=True)
    with system(n, T, eps2) as s:
        s.set_state(pos, np.zeros_like(pos))
        full = s.accel()
        for start, count in ((0, 1), (n - 17, 17), (5, 4096), (3, 4097), (0, n - 1)):
            assert np.array_equal(s.accel_slice(start, count), full[start:start + count]), (start, count)
    if T == np.float32:
        for i0 in (0, n - 32):
            want = O.gravitation_rows_f32(pos, eps2, i0, i0 + 32)[i0:i0 + 32]
            assert np.array_equal(full[i0:i0 + 32].astype(T), want)
    else:
        assert np.array_equal(full, O.gravitation_f64(pos, eps2))


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("what", ["lattice", "inf", "nan"])
def test_special_distances_bit_exact(what, T):
    """Integer coordinates with eps2 = 1 (many d2 are powers of four), and
    bodies at infinity or NaN."""
    n = 1000
    rng = np.random.default_rng(7)
    pos = np.zeros((n, 4), T)
    pos[:, :3] = rng.integers(-8, 9, (n, 3))
    pos[:, 3] = rng.uniform(0.5, 2.0, n)
    if what == "inf":
        pos[[3, 500, 998], [0, 1, 2]] = [np.inf, -np.inf, np.inf]
    if what == "nan":
        pos[501, 1] = np.nan
    print(f"case: ref split {what} {np.dtype(T).name}", flush=True)
    with system(n, T, T(1.0)) as s:
        s.set_state(pos, np.zeros_like(pos))
        a = s.accel().astype(T)
    assert np.array_equal(a, rows_want(pos, T(1.0), T), equal_nan=True)
