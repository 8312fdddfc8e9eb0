// force_fp32.hip -- launchers of the FP32 pair kernels (plain and mixed steps,
// field-only evaluation).  The kernel itself is in force_tmpl.h.
#include <algorithm>

#include "force_tmpl.h"

namespace utcnb {

namespace {
const Tile kTiles[] = {
    {1, 1, "k1s1", false},  {2, 1, "k2s1", false},  {4, 1, "k4s1", false},
    {1, 2, "k1s2", false},  {2, 2, "k2s2", false},  {1, 4, "k1s4", false},
    {2, 4, "k2s4", false},  {1, 8, "k1s8", false},  {2, 8, "k2s8", false},
    {1, 16, "k1s16", false},
    // symmetric (sym.hip): K targets per lane, R waves per wave block (sym8r64 and
    // sym8r128 are divided up to 46080 and 39936 bodies: sym_tile_r, sym_tile_rs)
    {4, 4, "sym4r4", true}, {4, 8, "sym4r8", true}, {8, 4, "sym8r4", true},
    {8, 8, "sym8r8", true}, {8, 16, "sym8r16", true}, {4, 16, "sym4r16", true},
    {4, 32, "sym4r32", true}, {8, 32, "sym8r32", true}, {4, 64, "sym4r64", true},
    {4, 128, "sym4r128", true}, {2, 32, "sym2r32", true}, {2, 64, "sym2r64", true},
    {8, 64, "sym8r64", true}, {8, 128, "sym8r128", true},
    // symmetric with each sub-unit's rotation cut into RS chunks: symKrRxRS
    {2, 64, "sym2r64x2", true, 2}, {4, 64, "sym4r64x2", true, 2}, {2, 128, "sym2r128x4", true, 4},
    {4, 128, "sym4r128x4", true, 4},
    // one kernel per step for small systems (force_small.h): A targets per
    // lane, TL target lanes per wave, W waves, at most CAP bodies:
    // smAtTLwWnCAPk; k = A, s = W (sm1t8w16n8k has A = 3 from 4097 to 6144 bodies)
    {1, 8, "sm1t4w8n2k", false, 1, 4, 2048}, {1, 8, "sm1t8w8n2k", false, 1, 8, 2048},
    {1, 16, "sm1t8w16n8k", false, 1, 8, 8192}, {1, 16, "sm1t16w16n4k", false, 1, 16, 4096},
    {1, 16, "sm1t16w16n8k", false, 1, 16, 8192}, {2, 16, "sm2t16w16n8k", false, 1, 16, 8192},
    // more one-pass tiles (appended: ids are stable)
    {2, 16, "k2s16", false}, {4, 8, "k4s8", false}, {4, 16, "k4s16", false},
    // past the tiles a system can be given (tile_count): one-pass, the sources
    // in P parts over separate waves (force_part.h), for slices and the
    // handle-free field: kKpP, whose bits are the same
    {1, 1, "k1p128", false, 1, 0, 0, 128}, {2, 1, "k2p64", false, 1, 0, 0, 64},
};
}  // namespace

size_t part_floats(int tile, int64_t nt) { return (size_t)kTiles[tile].parts * nt * 3; }

int tile_count() { return kTilePart128; }
int tile_total() { return (int)(sizeof(kTiles) / sizeof(kTiles[0])); }
const Tile& tile_get(int id) { return kTiles[id]; }

// Default tile, from sweeps of every tile on MI355X (mixed precision, time per
// step, best three; equal masses; log-uniform masses and plain FP32 rank
// alike):
//   N = 131072: sym8r64 2.732, sym8r32 2.768, sym8r128 2.814 ms  (sym4r64 2.906)
//   N =  65536: sym8r16 0.716, sym8r64 0.720, sym8r32 0.737 ms  (sym4r64 0.743)
//   N =  49152: sym8r64 431, sym8r32 439, sym4r32 440 us  (divided sym8r64 406: sym_tile_rs)
//   N =  40960: sym8r64 295, sym4r64 317, sym8r128 319 us
//   N =  32768: sym8r128 195, sym8r64 198, sym8r32 201 us  (sym4r64 211)
//   N =  24576: sym8r128 122.5, sym8r64 123.5, sym4r64x2 127.8 us  (sym4r64 129.5)
//   N =  16384: sym8r64 61.5, sym8r128 61.5, sym4r64 67.5 us  (sym4r64x2 68.1)
//   N =  14336: sym4r128 52.6, sym8r128 53.6, sym8r64 55.0 us  (sym4r64 56.8)
//   N =  12288: sym4r64x2 42.6, sym8r128 43.7, sym4r64 44.3 us
//   N =   9001: sym8r128 33.2, sym4r128 35.0, sym2r64 36.0 us  (sym4r64x2 36.5)
//   N =   8192: sm2t16w16n8k 22.2, sm1t16w16n8k 24.9 us  (sym4r64x2 26.1)
//   N =   7168: sm2t16w16n8k 20.0, sm1t16w16n8k 22.4 us  (sym4r64 22.6)
//   N =   6144: sm1t8w16n8k 15.2, sm2t16w16n8k 17.5, sm1t16w16n8k 19.7 us  (sym2r64 20.7)
//   N =   5120: sm1t8w16n8k 13.4, sm2t16w16n8k 15.1, sm1t16w16n8k 17.2 us
//   N =   4096: sm1t16w16n8k 8.2, sm1t16w16n4k 8.2, sm1t8w16n8k 10.3 us  (sym2r64x2 13.8)
//   N =   2048: sm1t8w8n2k 4.6, sm1t8w16n8k 4.7, sm1t4w8n2k 5.0 us  (sym2r64x2 9.8)
//   N =   1024: sm1t4w8n2k 3.4, sm1t8w8n2k 3.6, sm1t8w16n8k 3.9 us  (sym2r64x2 9.1)
// (sym8r48, sym8r24, other R and chunk counts for K = 2, 4 and 8 and several
// other small-system shapes were swept and are not in the table: 4 to 8 targets
// per lane, 4 target lanes with 16 waves, 8 waves per workgroup.)  Up to 8192
// bodies the small-system kernels win: one launch per step against two, and
// their one-pass pair sums fill the chip where the symmetric kernels' 64-step
// rotations leave it waiting.  Above, K = 8, which has the least LDS traffic
// and the fewest reaction partials per pair.  Up to 160 bodies per CU the
// waves' unequal ends weigh most: two waves on every SIMD (2048) that start
// together and have equal shares of the work but for an eighth of a sub-unit.
// Longer runs drift apart over the chip and want shorter waves, several in
// turn; from 46081 bodies whole ones, without a second reaction record
// (sym_tile_rs).  The partial sums must fit the
// device's budget (sym_partial_budget); above it a one-pass tile is used (N =
// 262144: k2s8 19.1 ms, k2s16 21.1).
size_t sym_partial_budget(size_t device_bytes)
{
    if (device_bytes == 0)
        return (size_t)16 << 30;
    return std::min<size_t>((size_t)64 << 30, device_bytes / 4);
}

int tile_default(int64_t n, int cu_count, size_t partial_budget)
{
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    const int64_t n_pad = pad_j(n);
    const auto fits = [&](int tile) {
        const Tile& t = kTiles[tile];
        return n_pad <= (1 << 30) && n_pad % (128 * t.k) == 0 &&
               (sym_jpart_floats((int)n_pad, t) + sym_ipart_floats((int)n_pad, t.k, sym_tile_r(t, (int)n_pad))) * sizeof(float) <=
                   partial_budget;
    };
    // from the sweeps above: each choice within 3% of the fastest tile at its size
    if (n <= 1024)
        return 28;  // sm1t4w8n2k
    if (n <= 2048)
        return 29;  // sm1t8w8n2k
    if (n <= 4096)
        return 31;  // sm1t16w16n4k
    if (n <= 6144)
        return 30;  // sm1t8w16n8k, with 3 targets per lane: 24 for each of the 256 CUs at 6144
    if (n <= 8192)
        return 33;  // sm2t16w16n8k
    if (n_pad >= 160 * cus && fits(22))
        return 22;  // sym8r64
    if (n >= 8 * cus && fits(23))
        return 23;  // sym8r128
    if ((n + 127) / 128 * 8 >= cus * 16)
        return 8;   // k2s8
    return 9;       // k1s16
}

template <class Epi>
hipError_t launch_sym(const Tile& t, bool newton, bool comp, const float4* src, int n, int n_pad, float eps2,
                      float* ipart, float* jpart, const Epi& epi, hipStream_t st);
template <class Epi>
hipError_t launch_sym_chunked(const Tile& t, bool newton, const float4* src, int n, int n_pad, float eps2,
                              int chunks, int Rs, float* ipart, float* jchunk, double* react3, const Epi& epi,
                              hipStream_t st);

// Shares and chunks of a default system divide it by wave blocks of this
// tile, whatever tile its whole steps take: at most n_pad / (64 K) shares, so
// the smaller the system the smaller K.
int sym_share_tile_default(int64_t n, int cu_count)
{
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    return n >= 96 * cus ? 22 : (n >= 64 * cus ? 18 : 20);  // sym8r64, sym4r64, sym2r32
}

hipError_t launch_fp32_step(const StepArgs& a, const float4* pos_old, float4* pos_new,
                            float4* vel, hipStream_t st)
{
    EpiFP32 epi{pos_old, pos_new, vel, (float)a.dt, (float)a.damping, a.kick};
    if (tile_get(a.tile).sym)
        return launch_sym(tile_get(a.tile), a.newton, false, pos_old, a.n, a.n_pad, a.eps2f, a.ipart,
                          a.jpart, epi, st);
    if (a.newton)
        return launch_force<false, true>(a.tile, pos_old, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return launch_force<false, false>(a.tile, pos_old, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

hipError_t launch_mixed_step(const StepArgs& a, const float4* snap_old, float4* snap_new,
                             double4* pos, double4* vel, hipStream_t st, float4* keep)
{
    EpiMixed epi{pos, vel, snap_new, a.dt, a.damping, a.kick, keep};
    if (tile_get(a.tile).sym && a.chunks > 0)
        return launch_sym_chunked(tile_get(a.share_tile), a.newton, snap_old, a.n, a.n_pad, a.eps2f, a.chunks, a.chunk_r,
                                  a.cipart, a.cjpart, a.react, epi, st);
    if (tile_get(a.tile).sym)
        return launch_sym(tile_get(a.tile), a.newton, true, snap_old, a.n, a.n_pad, a.eps2f, a.ipart,
                          a.jpart, epi, st);
    if (a.newton)
        return launch_force<true, true>(a.tile, snap_old, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return launch_force<true, false>(a.tile, snap_old, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

// One-pass tile for a slice of nt targets against all sources (the
// symmetric tiles evaluate unordered pairs of the whole system and do not
// split by target); part_ws: floats of workspace for the tiles with source
// parts.  From sweeps on MI355X, ms per step:
//   N = 262145: nt = 32769 k1p256 2.106, k1p128 2.109, k2p128 2.168, k2p64
//               2.322   (k2s8 5.19, k2s16 5.50, k1s16 5.86)
//   N = 262144: nt =   8192 k1p256 0.545, k1p128 0.561, k2p64 0.683 (k1s16 1.97)
//               nt =  32768 k1p128 2.090, k1p256 2.108, k2p64 2.220 (k2s16 2.63)
//               nt = 131072 k2p64 8.057, k2p128 8.060, k1p128 8.122 (k2s8 10.0)
//   N =  32768: nt =   4096 k1p128 0.051, k2p64 0.056               (k1s16 0.237)
// Many small waves fill the chip whatever the number of targets; 256 parts
// gain at most 3% more and take twice the workspace, K = 4 (k4p32 ... k4p128)
// is slower throughout.  Which of the two it is does not change a bit of the
// result, nor does the slicing: where the workspace holds fewer targets than
// the slice has, it is evaluated in several launches (launch_part_tile).
int slice_tile_default(int64_t nt, size_t part_ws)
{
    return part_floats(kTilePart128, nt) <= part_ws ? kTilePart128 : kTilePart64;
}

hipError_t launch_fp32_step_slice(const StepArgs& a, int tile, int i0, int nt, const float4* pos_old,
                                  float4* pos_new, float4* vel, hipStream_t st)
{
    if (tile_get(tile).sym)
        return hipErrorInvalidValue;
    EpiFP32 epi{pos_old, pos_new, vel, (float)a.dt, (float)a.damping, a.kick};
    if (a.newton)
        return launch_force_range<false, true>(tile, pos_old, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return launch_force_range<false, false>(tile, pos_old, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

hipError_t launch_mixed_step_slice(const StepArgs& a, int tile, int i0, int nt, const float4* snap_old,
                                   float4* snap_new, double4* pos, double4* vel, hipStream_t st)
{
    if (tile_get(tile).sym)
        return hipErrorInvalidValue;
    EpiMixed epi{pos, vel, snap_new, a.dt, a.damping, a.kick};
    if (a.newton)
        return launch_force_range<true, true>(tile, snap_old, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return launch_force_range<true, false>(tile, snap_old, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

hipError_t launch_fp32_accel_slice(const StepArgs& a, int tile, int i0, int nt, const float4* src,
                                   bool compensated, double* acc3, hipStream_t st)
{
    if (tile_get(tile).sym)
        return hipErrorInvalidValue;
    EpiAccel epi{acc3, i0};
    if (compensated)
        return a.newton ? launch_force_range<true, true>(tile, src, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st)
                        : launch_force_range<true, false>(tile, src, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return a.newton ? launch_force_range<false, true>(tile, src, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st)
                    : launch_force_range<false, false>(tile, src, i0, nt, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

hipError_t launch_fp32_accel(const StepArgs& a, const float4* src, bool compensated,
                             double* acc3, hipStream_t st)
{
    EpiAccel epi{acc3};
    if (tile_get(a.tile).sym && a.chunks > 0) {
        if (!compensated)
            return hipErrorInvalidValue;  // the chunked step sums its partials in FP64
        return launch_sym_chunked(tile_get(a.share_tile), a.newton, src, a.n, a.n_pad, a.eps2f, a.chunks, a.chunk_r,
                                  a.cipart, a.cjpart, a.react, epi, st);
    }
    if (tile_get(a.tile).sym)
        return launch_sym(tile_get(a.tile), a.newton, compensated, src, a.n, a.n_pad, a.eps2f, a.ipart,
                          a.jpart, epi, st);
    if (compensated) {
        if (a.newton)
            return launch_force<true, true>(a.tile, src, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
        return launch_force<true, false>(a.tile, src, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    }
    if (a.newton)
        return launch_force<false, true>(a.tile, src, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
    return launch_force<false, false>(a.tile, src, a.n, a.n_pad, a.eps2f, a.part_ws, epi, st);
}

}  // namespace utcnb
