"""The chunk ranges of the symmetric tiles (SymSplit, utc_amd/csrc/sym_reduce.h):
every chunk of a wave block's sub-units is taken by exactly one wave, and the
reduction reads exactly the reaction records that the waves write."""
import pytest


class Split:
    def __init__(self, NW, w, K, R, rs):
        self.chunks = (NW // 2 + (w < NW // 2)) * K * rs
        self.R, self.rs = min(R, self.chunks), rs

    def first(self, r):
        return self.chunks * r // self.R if r < self.R else self.chunks

    def wave(self, x):
        return ((x + 1) * self.R - 1) // self.chunks

    def records(self):
        return ((self.chunks + self.R - 1) // self.R + self.rs - 2) // self.rs + 1


@pytest.mark.parametrize("NW", [2, 4, 6, 12, 18, 26, 64])
@pytest.mark.parametrize("K", [2, 4, 8])
@pytest.mark.parametrize("R", [1, 2, 4, 16, 51, 64, 113, 128])
@pytest.mark.parametrize("rs", [2, 4, 8, 16])
def test_every_chunk_once_and_every_record_read(NW, K, R, rs):
    J, half = Split(NW, 0, K, R, rs).records(), NW // 2
    for w in {0, half - 1, half, NW - 1}:
        sp = Split(NW, w, K, R, rs)
        chunks, written = [], set()
        for r in range(R):  # sym_wave
            c0, c1 = sp.first(r), sp.first(r + 1)
            qf, ql = c0 // rs, (c1 + rs - 1) // rs
            for q in range(qf, ql):
                a = c0 - q * rs if q == qf else 0
                e = c1 - q * rs if q + 1 == ql else rs
                assert 0 <= a < e <= rs and q - qf < J
                chunks += range(q * rs + a, q * rs + e)
                written.add((r, q, q - qf))
        assert chunks == list(range(sp.chunks))
        read = set()
        for q in range(sp.chunks // rs):  # sym_split_sum
            for r in range(sp.wave(q * rs), sp.wave((q + 1) * rs - 1) + 1):
                read.add((r, q, q - sp.first(r) // rs))
        assert read == written
