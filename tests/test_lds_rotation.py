"""CPU check of how a block of 64 sources rotates through a wave's LDS in the
symmetric kernels (utc_amd/csrc/sym.hip sym_rotate, sym_vjp.hip sym_vjp_block),
restated: source s lies in slots s and s + 64 of 128; at rotation step t lane l
reads slot l + t, adds its reactions to the sum in slot l + t, and reads slot
l + t + 1 ahead for the next step.  A chunk runs steps [t0, t0 + steps); the sum
of source s is that of slots s and s + 64."""
import numpy as np
import pytest


@pytest.mark.parametrize("chunks", [1, 2, 4, 8, 16])
def test_every_lane_meets_every_source_once(chunks):
    steps = 64 // chunks
    source = np.arange(128) % 64
    met = np.zeros((64, 64), int)       # lane, source
    reaction = np.zeros((64, 64), int)  # source, lane
    lanes = np.arange(64)
    for t0 in range(0, 64, steps):
        sums = np.zeros((128, 64), int)  # slot, lanes that added to it
        for t in range(steps):
            slot = lanes + t0 + t
            assert len(set(slot)) == 64          # no two lanes on one slot
            assert slot.max() + 1 < 128          # the read ahead stays inside
            met[lanes, source[slot]] += 1
            sums[slot, lanes] += 1
        reaction += sums[:64] + sums[64:]        # lane s takes home slots s, s + 64
    assert (met == 1).all() and (reaction == 1).all()
