// Launch of the streaming temporally blocked step kernel (lbm_ts.hpp), shared
// by the units that instantiate it.
#pragma once

#include <type_traits>

#include "cs_internal.hpp"
#include "lbm_ts.hpp"
#include "strip_rule.hpp"

namespace cs {

// Columns per lane: two for 32-bit arithmetic, one for 64-bit (the kept rows of
// 8 levels take the same registers).
template <class T>
constexpr int ts_cells() { return sizeof(T) == 8 ? 1 : 2; }

inline StripCase strip_case(const cs_lattice* l)
{
    StripCase c;
    c.w = l->w;
    c.h = l->h;
    c.storage = l->storage;
    c.cus = l->cus;
    c.half = l->has_flags && l->params.boundary == CS_BB_HALFWAY;
    c.zero_edge = l->params.edge == CS_EDGE_ZERO;
    c.io = c.half && l->has_io;
    c.mask = l->has_flags && !c.half;
    c.stochastic = l->params.rounding == CS_ROUND_STOCHASTIC;
    c.kbc = l->params.collision == CS_COLL_KBC;
    return c;
}

template <class St, int EDGE, int MODE, int K, int COLL, bool SR = false>
void ts_launch(cs_lattice* l)
{
    using T = typename St::T;
    constexpr int V = ts_cells<T>();
    const TsSplit sp = ts_split(strip_case(l), V, K);
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
