// sym_split.h -- how the waves of a wave block share its work in chunks (host and
// device; the symmetric kernels of sym.hip and sym_vjp.hip and their reductions).
#pragma once

#include <hip/hip_runtime.h>

namespace utcnb {

// How the R waves of wave block w of NW share its sub-units when each is cut
// into RS chunks (K sub-units for the own unit and each of the NW/2 after it,
// one less in the upper half, which skips the block half way round): wave r
// takes chunks [first(r), first(r + 1)) in a row, whole sub-units but for the
// first and the last, and leaves one reaction record for each of the at most
// J sub-units it touches.  Waves past the last chunk take none.  The products
// stay below 2^31: partial sums of at most 64 GiB hold some 180000 chunks per
// wave block, and R <= 128.
struct SymSplit {
    int chunks, R, rs;
    __host__ __device__ SymSplit(int NW, int w, int K, int R_, int rs_)
        : chunks((NW / 2 + (w < NW / 2)) * K * rs_), R(R_ < chunks ? R_ : chunks), rs(rs_)
    {
    }
    __host__ __device__ int first(int r) const { return r < R ? (int)((unsigned)(chunks * r) / (unsigned)R) : chunks; }
    // the wave that takes chunk x: the last r with first(r) <= x
    __host__ __device__ int wave(int x) const { return (int)((unsigned)((x + 1) * R - 1) / (unsigned)chunks); }
    __host__ __device__ int records() const { return ((chunks + R - 1) / R + rs - 2) / rs + 1; }
    // J: the lower half's waves touch the most
    __host__ __device__ static int records(int NW, int K, int R, int rs) { return SymSplit(NW, 0, K, R, rs).records(); }
};

}  // namespace utcnb
