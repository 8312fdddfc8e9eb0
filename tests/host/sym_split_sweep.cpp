// Sweeps SymSplit (utc_amd/csrc/sym_split.h): every chunk of a wave block goes to
// one wave, in order; a wave touches at most J sub-units; the reduction's first
// and last wave of a sub-unit (sym_split_sum) are those that take its chunks.
#include <cstdio>
#include <cstdlib>

#include "sym_split.h"

using utcnb::SymSplit;

static void check(bool ok, const char* what, int NW, int w, int K, int R, int rs, int r)
{
    if (ok)
        return;
    std::printf("%s: NW=%d w=%d K=%d R=%d rs=%d r=%d\n", what, NW, w, K, R, rs, r);
    std::exit(1);
}

static void sweep(int NW, int w, int K, int R, int rs)
{
    const SymSplit sp(NW, w, K, R, rs);
    const int J = SymSplit::records(NW, K, R, rs);
    int next = 0;
    for (int r = 0; r < R; ++r) {  // sym_wave
        const int c0 = sp.first(r), c1 = sp.first(r + 1);
        check(c0 == next && c1 >= c0, "chunks in a row", NW, w, K, R, rs, r);
        next = c1;
        check((c1 + rs - 1) / rs - c0 / rs <= J, "records", NW, w, K, R, rs, r);
        for (int x : {c0, (c0 + c1) / 2, c1 - 1})
            if (x >= c0 && x < c1)
                check(sp.wave(x) == r, "wave of a chunk", NW, w, K, R, rs, r);
    }
    check(next == sp.chunks && sp.chunks == (NW / 2 + (w < NW / 2)) * K * rs, "all chunks", NW, w, K, R, rs, R);
}

int main()
{
    for (int NW = 2; NW <= 66; NW += 2)
        for (int K : {2, 4, 8})
            for (int R : {1, 2, 3, 16, 32, 51, 64, 113, 128})
                for (int rs : {2, 4, 8, 16})
                    for (int w : {0, NW / 2 - 1, NW / 2, NW - 1})
                        sweep(NW, w, K, R, rs);
    // the most wave blocks whose partial sums fit 64 GiB: sym2r128x4, sym4r128x4
    // and the VJP (K = 4, 16 chunks, 32 waves, 16-byte records)
    sweep(9248, 0, 2, 128, 4);
    sweep(6534, 0, 4, 128, 4);
    sweep(5746, 0, 4, 32, 16);
    std::puts("ok");
    return 0;
}
