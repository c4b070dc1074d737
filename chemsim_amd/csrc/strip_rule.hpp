// Which lattices take the streaming temporally blocked step (lbm_ts.hpp) and
// how it splits them: host arithmetic on sizes and modes, without HIP, so that
// a test can ask it about any lattice.
#pragma once

#include <algorithm>
#include <cstdint>

#include "../../include/chemsim.h"

namespace cs {

// What the choice depends on.
struct StripCase {
    int w = 0, h = 0;
    int storage = CS_F32;     // cs_storage
    int cus = 256;            // compute units
    bool half = false;        // half-way boundary mode with flags
    bool zero_edge = false;   // zero edge, not periodic
    bool io = false;          // ... and inlet or outlet cells
    bool mask = false;        // reference boundary mode with flags
    bool stochastic = false;  // 16-bit storage: stochastic rounding
    bool kbc = false;
    bool walls() const { return half && zero_edge; }  // the lattice's own edge is a wall
};

// Waves are independent and all resident at once, two per SIMD; rows are
// split into as many runs as that allows, of at least 8 rows.  Where the
// lattice's own edge is a wall (half-way mode, zero edge), every row of the
// first and the last strip takes the geometry pulls and the edge masks, so
// these strips get more and shorter runs.
struct TsSplit {
    int strips, chunks, edge_chunks;
    int64_t waves() const { return (int64_t)std::max(0, strips - 2) * chunks + (int64_t)std::min(strips, 2) * edge_chunks; }
};
// v: columns per lane, k: steps per launch.
inline TsSplit ts_split(const StripCase& c, int v, int k)
{
    const int in = 64 * v - 2 * k;
    TsSplit s;
    s.strips = (c.w + in - 1) / in;
    const int waves = 2 * 4 * c.cus, most = (c.h + 7) / 8;
    // an edge strip's time per row in inner strips': cavity and channel 4096^2,
    // GLUPS with 1, 1.3, 1.6, 2: 206, 226, 243, 242 and 181, 195, 192, 188
    const double share = c.walls() ? 1.6 : 1.0;
    const int edges = std::min(s.strips, 2);
    const double unit = waves / (s.strips - edges + edges * share);
    s.chunks = std::clamp((int)unit, 1, most);
    s.edge_chunks = std::clamp((int)(unit * share), 1, most);
    return s;
}

// Cells computed per kept cell by the streaming kernel (two columns per lane)
// with the runs of inner strips, or those of edge strips.
inline double ts_computed(const StripCase& c, int k, bool edge_runs = false)
{
    const TsSplit s = ts_split(c, 2, k);
    const double rows = (double)c.h / (edge_runs ? s.edge_chunks : s.chunks);
    return (double)s.strips * 128 * (rows + k - 1) / ((double)c.w * rows);
}
// The device's wave slots over the waves that run in them: above 1 where the
// last (or only) round of waves leaves slots idle.
inline double ts_idle(const StripCase& c, int64_t waves)
{
    const int64_t slots = 2 * 4 * (int64_t)c.cus;
    return (double)((waves + slots - 1) / slots * slots) / (double)waves;
}

constexpr int TS_REGION_EDGE = 64;  // the region kernels' side above about 512^2 (lbm_tb.hpp, TB_EDGE)
inline double region_computed(const StripCase& c, int k)
{
    const int in = TS_REGION_EDGE - 2 * k;
    return (double)((c.w + in - 1) / in) * ((c.h + in - 1) / in) * TS_REGION_EDGE * TS_REGION_EDGE /
           ((double)c.w * c.h);
}

// A last strip that keeps at most K columns (K + 1 with walls, whose links reach
// one column further) leaves edge cells to the one before it as well, which has
// an inner strip's long runs: the launch waits for those.
inline bool ts_two_wall_strips(const StripCase& c)
{
    constexpr int K = 8, in = 128 - 2 * K;
    const int strips = (c.w + in - 1) / in;
    return c.walls() && strips > 2 && c.w - (strips - 1) * in <= K + (c.io ? 0 : 1);
}

// FP32 and FP32 deviations: strips against regions, cells computed by each.
inline bool ts_takes_32(const StripCase& c)
{
    constexpr int K = 8;
    const TsSplit s = ts_split(c, 2, K);
    const double stream = ts_computed(c, K), regions = region_computed(c, K);
    if ((c.half ? 1.0 : 1.12) * stream >= regions) return false;
    const double computed = s.strips <= 2 ? ts_computed(c, K, true) : stream;
    const double cost = !c.half ? 1.12 : c.io ? 1.19 : !c.walls() ? 1.0 : s.strips <= 2 ? 0.95 : s.strips <= 5 ? 1.1 : 1.0;
    const double two = !ts_two_wall_strips(c) ? 1.0 : c.io ? 1.3 : 1.2;
    const double idle = ts_idle(c, s.waves());
    return cost * two * computed * (s.waves() > 8 * (int64_t)c.cus ? 1 + 0.6 * (idle - 1) : 1) < regions;
}

// 16-bit storage: strips against the one-step kernels, whose geometry modes
// compute whole tiles of 256 columns.
inline bool ts_takes_16(const StripCase& c)
{
    constexpr int K = 8;
    const bool bf16 = c.storage == CS_BF16DEV, sr = c.stochastic;
    const double stream = ts_computed(c, K);
    const double most = c.half ? 1.65 : !sr ? 2.2 : bf16 ? 1.9 : 1.45;
    if (stream >= most) return false;
    if (!bf16 && !sr) return true;
    const double idle = ts_idle(c, ts_split(c, 2, K).waves());
    const double cost = stream * (1 + (bf16 || c.half ? 1.5 : 1.0) * std::max(0.0, idle - 1.05)) *
                        (ts_two_wall_strips(c) ? 1.3 : 1.0);
    const double tiles = (double)((c.w + 255) / 256 * 256) / c.w;
    if (c.io && sr) return cost / tiles < (bf16 ? 1.24 : 1.31);
    if (c.half) return cost < (sr ? most : 2.0);
    if (c.mask) return cost / tiles < (!sr ? 1.75 : bf16 ? 1.375 : 1.4);
    return cost < most;
}

// Whether the lattice takes 8 steps per launch in strips.  The figures behind
// the lines are in lattice_ts.hip.
inline bool ts_takes(const StripCase& c)
{
    constexpr int K = 8;
    if (c.kbc) return false;
    if (c.h < 2 * K) return false;  // the kernel wraps a row index once
    if (c.storage == CS_F64) return (int64_t)c.w * c.h >= (int64_t)1 << 20;
    // both waves of (nearly) every SIMD, or the region kernels' many small blocks win
    if (ts_split(c, 2, K).waves() < 6 * (int64_t)c.cus) return false;
    return c.storage == CS_BF16DEV || c.storage == CS_F16DEV ? ts_takes_16(c) : ts_takes_32(c);
}

// A lattice of 8 steps per launch in strips: whether its 4-step remainder
// launch goes in strips too, or (FP32) in regions.
inline bool ts_takes_remainder(const StripCase& c)
{
    if (c.storage == CS_F64) return true;
    const bool narrow = ts_split(c, 2, 4).strips <= 2;
    return ts_computed(c, 4) < (c.half ? 1.2 : narrow ? 1.1 : c.mask ? 0.907 : 0.96) * region_computed(c, 4);
}

}  // namespace cs
