// Launch of the streaming temporally blocked step kernel (lbm_ts.hpp), shared
// by the units that instantiate it.
#pragma once

#include <algorithm>
#include <type_traits>

#include "cs_internal.hpp"
#include "lbm_ts.hpp"

namespace cs {

// Columns per lane: two for 32-bit arithmetic, one for 64-bit (the kept rows of
// 8 levels take the same registers).
template <class T>
constexpr int ts_cells() { return sizeof(T) == 8 ? 1 : 2; }

// Waves are independent and all resident at once, two per SIMD; rows are
// split into as many runs as that allows, of at least 8 rows.  Where the
// lattice's own edge is a wall (half-way mode, zero edge), every row of the
// first and the last strip takes the geometry pulls and the edge masks, so
// these strips get more and shorter runs.
struct TsSplit {
    int strips, chunks, edge_chunks;
    int64_t waves() const { return (int64_t)std::max(0, strips - 2) * chunks + (int64_t)std::min(strips, 2) * edge_chunks; }
};
inline TsSplit ts_split(const cs_lattice* l, int v, int k)
{
    const int in = 64 * v - 2 * k;
    TsSplit s;
    s.strips = (l->w + in - 1) / in;
    const int waves = 2 * 4 * l->cus, most = (l->h + 7) / 8;
    const bool walls = l->has_flags && l->params.boundary == CS_BB_HALFWAY && l->params.edge == CS_EDGE_ZERO;
    // an edge strip's time per row in inner strips': cavity and channel 4096^2,
    // GLUPS with 1, 1.3, 1.6, 2: 206, 226, 243, 242 and 181, 195, 192, 188
    const double share = walls ? 1.6 : 1.0;
    const int edges = std::min(s.strips, 2);
    const double unit = waves / (s.strips - edges + edges * share);
    s.chunks = std::clamp((int)unit, 1, most);
    s.edge_chunks = std::clamp((int)(unit * share), 1, most);
    return s;
}

template <class St, int EDGE, int MODE, int K, int COLL, bool SR = false>
void ts_launch(cs_lattice* l)
{
    using T = typename St::T;
    constexpr int V = ts_cells<T>();
    const TsSplit sp = ts_split(l, V, K);
    TsArgs<T, K> A{};
    A.a.fin = l->buf[l->cur];
    A.a.fout = l->buf[l->cur ^ 1];
    A.a.node = MODE == MODE_FLUID ? nullptr : l->node;
    A.a.w = l->w;
    A.a.h = l->h;
    A.a.pitch = l->pitch;
    A.a.cpitch = l->cpitch;
    A.a.plane = l->plane;
    if constexpr (std::is_same_v<T, double>) A.a.k = l->k64;
    else A.a.k = l->k32;
    A.strips = sp.strips;
    A.chunks = sp.chunks;
    A.edge_chunks = sp.edge_chunks;
    if constexpr (SR)
        for (int s = 0; s < K; ++s) A.keys[s] = sr_key(l->params.seed, l->steps + (uint64_t)s);
    const unsigned blocks = (unsigned)((sp.waves() + TS_WAVES - 1) / TS_WAVES);
    hipLaunchKernelGGL((k_step_ts<St, EDGE, MODE, K, COLL, V, SR>), dim3(blocks), dim3(TS_THREADS), 0, l->stream, A);
    l->cur ^= 1;
    l->steps += K;
    for (int s = 0; s < K; ++s) l->time += l->params.delta_t;  // as step by step (lbm.rs:713)
}

// The units that instantiate it per storage: k = 8 or, for BGK, 4 steps.
void launch_ts_f64(cs_lattice* l, int k);
void launch_ts_16(cs_lattice* l);  // 8 steps

}  // namespace cs
