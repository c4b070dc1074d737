// Temporally blocked fused step, streaming variant: K steps per launch, each
// wave marching down a strip of the lattice with all K time levels in flight.
//
// A wave owns a strip of 64 V columns (lane l the V columns V l .. V l + V-1)
// and a run ("chunk") of rows.  In iteration t it computes one row of every
// level: level 1 row r from the stored lattice, level 2 row r - 1 from level
// 1, ..., level K row r - K + 1, which it stores.  Level s needs rows r' - 1,
// r' and r' + 1 of level s - 1 for its row r': the last is the row level s - 1
// has just computed, the others are kept in registers -- only the populations
// that are still to be pulled: 0, 2, 4 of row r' and 3, 6, 7 of rows r' and
// r' - 1, nine values per cell and level.  Neighbouring columns come from the
// lane itself or from the next lane (ts_lane).  No barrier and no
// communication between waves; the per-cell arithmetic and pull order are the
// one-step kernels', so K steps equal K launches of k_step bit for bit.
//
// What is computed more than once: K columns on either side of the strip
// (64 V - 2 K of 64 V columns are kept) and (K - 1) / R of a chunk of R rows
// (level s starts 2 (s - 1) iterations after level 1).  The region variants
// (lbm_tb.hpp) recompute the halo on all four sides.
//
// Bound by VALU issue.  4096^2 FP32 Taylor-Green, 800 steps in a row: 51.8 us per
// step against 68.2 for the register regions (k_step_tbr), 153 against 201 VALU
// instructions per kept cell and step, 0.34 against 0.32 of them per SIMD and
// cycle at two waves per SIMD.  With DPP shifts and v_rcp_f32 instead of the
// LDS crossbar and recip_newton it ran at 0.27 per cycle, 63 us per step; with
// the row loop not unrolled by two, 58 us (the kept rows' registers are then
// copied at every iteration).  K = 4 with the same strips: 72 us.
//
// Cells outside a zero-edged lattice hold the outside value (f = 0, or
// g = -w_i rho0) at every level; a periodic lattice is unrolled by wrapping
// the loads.
//
// Geometry: the node words of a row are read once, when the row enters, and
// wait for the later levels in a ring of rows in LDS (each lane reads only
// what it wrote); a bit per row says whether any cell of the wave's row needs
// more than the plain pulls, and rows without one -- most rows of a lattice --
// take the fluid path.  In the half-way mode a special row's populations 1, 5
// and 8 (the only own values that are not in registers any more when the
// level above needs them for links and carried cells) wait in LDS as well.
#pragma once

#include "lbm_tb.hpp"

namespace cs {

constexpr int TS_WAVES = 4;                // waves per block (independent of each other)
constexpr int TS_THREADS = 64 * TS_WAVES;
constexpr int TS_RING = 16;                // rows of node words kept (>= K + 1, a power of two)

template <class T, int K>
struct TsArgs {
    StepArgs<T> a;
    int strips, chunks;   // waves: chunks per inner strip,
    int edge_chunks;      // and per first and last strip
    uint32_t keys[K];     // stochastic rounding keys of the K steps
};

// The value of the lane to the left or right (NEXT).  32-bit values go through
// the LDS crossbar (`from`: 4 x the lane): a DPP wave shift would do, but keeps
// the SIMD's two waves from issuing side by side (recip_newton's comment).
// 64-bit arithmetic issues from one wave at a time anyway and takes the DPP.
template <bool NEXT, class T>
__device__ __forceinline__ T ts_lane(int from, T v)
{
    if constexpr (sizeof(T) == 8) return lane_shift<T, NEXT>(v);
    else return __builtin_bit_cast(T, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, v)));
}
// y[j] = the value of the column to the left or right (NEXT) of lane cell j; e: the neighbouring lane's cell.
template <bool NEXT, class T, int V>
__device__ __forceinline__ void ts_shift(const T (&x)[V], T e, T (&y)[V])
{
#pragma unroll
    for (int j = 0; j < V; ++j) y[j] = NEXT ? (j + 1 < V ? x[j + 1 < V ? j + 1 : 0] : e) : (j > 0 ? x[j > 0 ? j - 1 : 0] : e);
}

// The nine values of a cell rounded to the 16-bit storage, with finish()'s
// random bits if SR.  For bf16 in the integer form (round to nearest even, or
// the top 16 random bits added below the kept ones and truncated): the
// conversions' NaN tests per value and v_cvt_sr_bf16_f32, which holds the
// SIMD's second wave back (recip_newton's comment), cost more -- 4096^2
// Taylor-Green, bf16 168 GLUPS to nearest and 157 stochastic with them.  A NaN
// takes them.  For f16, whose subnormal results would need more instructions
// than the conversion costs, the conversion itself.
template <class St, bool SR>
__device__ __forceinline__ void ts_round(float (&x)[9], uint32_t cell_key)
{
    uint32_t h = SR ? lowbias32(cell_key) : 0u;
    if constexpr (std::is_same_v<St, StBF16>) {
        bool nan = x[8] != x[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) nan = nan || __builtin_isunordered(x[2 * q], x[2 * q + 1]);
        if (!nan) {
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const uint32_t u = __builtin_bit_cast(uint32_t, x[i]);
                const uint32_t add = !SR ? 0x7fffu + ((u >> 16) & 1u) : (i & 1) ? (h & 0xffffu) : (h >> 16);
                x[i] = __builtin_bit_cast(float, (u + add) & 0xffff0000u);
                if (SR && (i & 1)) h = xorshift32(h);
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        x[i] = St::wid(SR ? St::nar_sr(x[i], (i & 1) ? h << 16 : h) : St::nar(x[i]));
        if (SR && (i & 1)) h = xorshift32(h);
    }
}

// Per-wave LDS of the geometry modes.
template <class T, int MODE, int K, int V>
struct TsLds {
    uint32_t ring[TS_RING][64 * V];
    T own[MODE == MODE_HALF ? K : 1][3][64 * V];  // populations 1, 5, 8 of a level's last row
};
template <class T, int K, int V>
struct TsLds<T, MODE_FLUID, K, V> {};

// One strip and chunk: output rows ra .. rb-1, columns c0 + K .. c0 + 64 V - K - 1.
template <class St, int EDGE, int MODE, int K, int COLL, int V, bool SR>
__device__ __forceinline__ void ts_strip(const TsArgs<typename St::T, K>& A, int c0, int ra, int rb,
                                         TsLds<typename St::T, MODE, K, V>* lds)
{
    using S = typename St::S;
    using T = typename St::T;
    constexpr bool HALF = MODE == MODE_HALF;
    constexpr int UNROLL = HALF ? 1 : 2;  // the half-way mode's loop is too long to repeat
    const StepArgs<T>& a = A.a;
    const int lane = (int)(threadIdx.x & 63);
    const int lprev = ((lane - 1) & 63) * 4, lnext = ((lane + 1) & 63) * 4;
    const S* __restrict__ fin = (const S*)a.fin;
    S* __restrict__ fout = (S*)a.fout;

    // this lane's columns in the lattice, and whether they lie inside it
    uint32_t col[V];
    bool cin[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        int c = c0 + lane * V + j;
        cin[j] = true;
        if (EDGE == CS_EDGE_PERIODIC) {
            c %= a.w;
            c += c < 0 ? a.w : 0;
        } else {
            cin[j] = c >= 0 && c < a.w;
            c = cin[j] ? c : 0;
        }
        col[j] = (uint32_t)c;
    }
    uint32_t inside[V];  // cin as a vector mask
#pragma unroll
    for (int j = 0; j < V; ++j) inside[j] = lane_mask(cin[j], 0);
    const bool edge_strip = EDGE == CS_EDGE_ZERO && (c0 < 0 || c0 + 64 * V > a.w);  // uniform over the wave
    const bool vec_out = V == 1 || c0 + 64 * V - K <= a.w || a.w % V == 0;  // the lane's cells stored as one vector
    const auto outside = [&](int i) -> T { return St::DEV ? -a.k.base(i) : T(0); };
    // wrapped or clamped row, and whether it lies inside the lattice
    const auto wrap_row = [&](int r, bool& in) -> int {
        in = true;
        if (EDGE == CS_EDGE_PERIODIC) return r < 0 ? r + a.h : (r >= a.h ? r - a.h : r);  // h > K
        in = r >= 0 && r < a.h;
        return in ? r : 0;
    };

    S P[9][V];           // stored values of the next row to enter (raw, as loaded)
    uint32_t Pn[V];      // its node words
    const auto load3 = [&](int r, const int (&dir)[3]) {
        bool in;
        const int g = wrap_row(r, in);
        const S* row = fin + (int64_t)g * a.pitch;
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int j = 0; j < V; ++j) P[dir[q]][j] = *at<uint32_t>(row + dir[q] * a.plane, col[j]);
    };
    constexpr int UP[3] = {1, 5, 8}, MID[3] = {0, 2, 4}, DN[3] = {3, 6, 7};
    // what iteration t's level 1 pulls for its row r (half-way mode: the row's
    // own 3, 6, 7, which the next row pulls; the previous ones are kept)
    const auto load_row = [&](int r) {
        load3(r + 1, UP);
        load3(r, MID);
        load3(HALF ? r : r - 1, DN);
        if (MODE != MODE_FLUID) {
            bool in;
            const int g = wrap_row(r, in);
#pragma unroll
            for (int j = 0; j < V; ++j) Pn[j] = a.node[(int64_t)g * a.cpitch + col[j]];
        }
    };
    // widened P[i] with the outside value where row r (of population i) or the column is outside
    const auto take = [&](int i, int r, T (&x)[V]) {
        bool in;
        wrap_row(r, in);
#pragma unroll
        for (int j = 0; j < V; ++j) x[j] = St::wid(P[i][j]);
        if (EDGE == CS_EDGE_ZERO && (edge_strip || !in)) {  // uniform over the wave
#pragma unroll
            for (int j = 0; j < V; ++j) x[j] = lane_select(in ? inside[j] : 0u, x[j], outside(i));
        }
    };

    T M[K][3][V], D0[K][3][V], D1[K][3][V];  // [level - 1 .. ]: mid (row r), down (rows r - 1, r) of each level's output
#pragma unroll
    for (int s = 0; s < K; ++s)
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int j = 0; j < V; ++j) M[s][q][j] = D0[s][q][j] = D1[s][q][j] = T(0);

    const int iters = (rb - ra) + 2 * (K - 1);
    int r1 = ra - (K - 1);  // level 1's row
    // bit s - 1: level s's row needs the geometry pulls; has a lid link; has an inlet or outlet cell
    uint32_t special = 0, lid_rows = 0, io_rows = 0;
    if constexpr (HALF) {
        // populations 3, 6, 7 of the row above the first, and 1, 5, 8 of the first row itself
        load3(r1 - 1, DN);
        load3(r1, UP);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            take(DN[q], r1 - 1, D0[0][q]);
            T u[V];
            take(UP[q], r1, u);
#pragma unroll
            for (int j = 0; j < V; ++j) lds->own[0][q][lane * V + j] = u[j];
        }
    }
    load_row(r1);

    // One iteration; FILL: level s runs from iteration 2 (s - 1) on, before that its rows are not there yet.
    const auto iteration = [&](auto fill, int t) {
        constexpr bool FILL = decltype(fill)::value;
        T N[9][V];  // the row the level below has just computed: up (row r + 1); for level 1 the loaded values
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            take(UP[q], r1 + 1, N[UP[q]]);
            take(MID[q], r1, N[MID[q]]);
            take(DN[q], HALF ? r1 : r1 - 1, N[DN[q]]);
        }
        if constexpr (MODE != MODE_FLUID) {
            bool in, need = false, lid = false, io = false;
            wrap_row(r1, in);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const uint32_t w = in && cin[j] ? Pn[j] : 0u;
                const int type = (int)(w >> NODE_TYPE_SHIFT);
                const bool solid = type == CS_WALL || type == CS_LID;
                need = need || solid || (HALF && ((w & 0x1FEu) != 0 || type != CS_FLUID));
                lid = lid || (w & 0x3FC00u) != 0;
                io = io || type == CS_INLET || type == CS_OUTLET;
                lds->ring[r1 & (TS_RING - 1)][lane * V + j] = w;
            }
            special = (special << 1) | (__any(need) ? 1u : 0u);
            if (HALF) {
                lid_rows = (lid_rows << 1) | (__any(lid) ? 1u : 0u);
                io_rows = (io_rows << 1) | (__any(io) ? 1u : 0u);
            }
        }
        load_row(r1 + 1);

        // what crosses the lanes on the way into level 1
        T e2 = ts_lane<false>(lprev, N[2][V - 1]), e4 = ts_lane<true>(lnext, N[4][0]);
        T e5 = ts_lane<false>(lprev, N[5][V - 1]), e8 = ts_lane<true>(lnext, N[8][0]);
        T e6 = ts_lane<false>(lprev, HALF ? D0[0][1][V - 1] : N[6][V - 1]);
        T e7 = ts_lane<true>(lnext, HALF ? D0[0][2][0] : N[7][0]);
#pragma unroll
        for (int s = 1; s <= K; ++s) {
            __builtin_amdgcn_sched_barrier(0);  // levels one after the other: overlapping them costs registers
            const int r = r1 - (s - 1);
            // pulls: up from N, mid and down from the kept rows of level s - 1
            T B[9][V], C[V][9];
            T um[3][V], dn[3][V], dc[3][V];  // mid of row r, down of rows r - 1 and r
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    if (s == 1) {  // level 0: the loaded rows themselves
                        um[q][j] = N[MID[q]][j];
                        dn[q][j] = HALF ? D0[0][q][j] : N[DN[q]][j];
                        dc[q][j] = N[DN[q]][j];
                        if (HALF) D0[0][q][j] = N[DN[q]][j];
                    } else {
                        um[q][j] = M[s - 1][q][j];
                        dn[q][j] = D0[s - 1][q][j];
                        dc[q][j] = D1[s - 1][q][j];
                        M[s - 1][q][j] = N[MID[q]][j];
                        D0[s - 1][q][j] = D1[s - 1][q][j];
                        D1[s - 1][q][j] = N[DN[q]][j];
                    }
                }
            T u1[3][V];  // half-way mode: the level's own up populations of row r
            const bool spec = MODE != MODE_FLUID && ((special >> (s - 1)) & 1u) != 0;
            if constexpr (HALF) {
                // level s - 1's row r + 1 is the own row of the next iteration
                if (spec) {
#pragma unroll
                    for (int q = 0; q < 3; ++q)
#pragma unroll
                        for (int j = 0; j < V; ++j) u1[q][j] = lds->own[s - 1][q][lane * V + j];
                }
                if (s == 1 || ((special >> (s >= 2 ? s - 2 : 0)) & 1u)) {
#pragma unroll
                    for (int q = 0; q < 3; ++q)
#pragma unroll
                        for (int j = 0; j < V; ++j) lds->own[s - 1][q][lane * V + j] = N[UP[q]][j];
                }
            }
            if (FILL && t < 2 * (s - 1)) continue;  // uniform
#pragma unroll
            for (int j = 0; j < V; ++j) {
                B[0][j] = um[0][j];
                B[1][j] = N[1][j];
                B[3][j] = dn[0][j];
            }
            ts_shift<false, T, V>(um[1], e2, B[2]);
            ts_shift<true, T, V>(um[2], e4, B[4]);
            ts_shift<false, T, V>(N[5], e5, B[5]);
            ts_shift<true, T, V>(N[8], e8, B[8]);
            ts_shift<false, T, V>(dn[1], e6, B[6]);
            ts_shift<true, T, V>(dn[2], e7, B[7]);
            if (s < K) {
                // the next level's kept populations start across the lanes while this level computes
                e2 = ts_lane<false>(lprev, M[s < K ? s : 0][1][V - 1]);
                e4 = ts_lane<true>(lnext, M[s < K ? s : 0][2][0]);
                e6 = ts_lane<false>(lprev, D0[s < K ? s : 0][1][V - 1]);
                e7 = ts_lane<true>(lnext, D0[s < K ? s : 0][2][0]);
            }
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int i = 0; i < 9; ++i) C[j][i] = B[i][j];

            uint32_t info[V];
            if constexpr (MODE != MODE_FLUID) if (spec) {  // uniform over the wave
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    info[j] = lds->ring[r & (TS_RING - 1)][lane * V + j];
                    const int type = (int)(info[j] >> NODE_TYPE_SHIFT);
                    const bool solid = type == CS_WALL || type == CS_LID;
                    if constexpr (MODE == MODE_REF) {
                        const uint32_t swap = lane_mask(solid, 0);
#pragma unroll
                        for (int i = 1; i < 9; ++i)
                            if (i < OPP[i]) {
                                const T x = C[j][i], y = C[j][OPP[i]];
                                C[j][i] = lane_select(swap, y, x);
                                C[j][OPP[i]] = lane_select(swap, x, y);
                            }
                    } else if constexpr (HALF) {
                        const T own[9] = {um[0][j], u1[0][j], um[1][j], dc[0][j], um[2][j],
                                          u1[1][j], dc[1][j], dc[2][j], u1[2][j]};
                        const uint32_t links = solid ? 0u : info[j];
                        if ((lid_rows >> (s - 1)) & 1u) {  // uniform
#pragma unroll
                            for (int i = 1; i < 9; ++i) {
                                const T v = own[OPP[i]];
                                C[j][i] = lane_select(lane_mask(links, i), lane_select(lane_mask(links, 9 + i), v + a.k.lid(i), v), C[j][i]);
                            }
                        } else {
#pragma unroll
                            for (int i = 1; i < 9; ++i) C[j][i] = lane_select(lane_mask(links, i), own[OPP[i]], C[j][i]);
                        }
                        if ((io_rows >> (s - 1)) & 1u) {  // uniform
                        if constexpr (St::DEV) {
                            if (type == CS_INLET) zou_he_inlet_dev<T>(C[j], a.k.rho0, a.k.in_ux, a.k.in_uy);
                            else if (type == CS_OUTLET) zou_he_outlet_dev<T>(C[j], a.k.rho0, a.k.out_rho);
                        } else {
                            if (type == CS_INLET) zou_he_inlet<T>(C[j], a.k.in_ux, a.k.in_uy);
                            else if (type == CS_OUTLET) zou_he_outlet<T>(C[j], a.k.out_rho);
                        }
                        }
                    }
                }
            }
            if (EDGE == CS_EDGE_ZERO && edge_strip) {
                // cells outside keep the outside value (below); a rho of 1 keeps them off the reciprocal's branch
#pragma unroll
                for (int j = 0; j < V; ++j) C[j][0] = lane_select(inside[j], C[j][0], T(1));
            }
            if constexpr (V == 1) {
                collide_cell<St, COLL>(a.k, C[0]);
            } else {
                Cells<T, V> X[9];
#pragma unroll
                for (int i = 0; i < 9; ++i)
#pragma unroll
                    for (int j = 0; j < V; ++j) X[i].v[j] = C[j][i];
                collide_cell<St, COLL>(a.k, X);
#pragma unroll
                for (int i = 0; i < 9; ++i)
#pragma unroll
                    for (int j = 0; j < V; ++j) C[j][i] = X[i].v[j];
            }
            if constexpr (is_16bit<St>()) {
                // every step's result is rounded to the storage type, as a store would
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    bool in;
                    const uint32_t g = (uint32_t)wrap_row(r, in);
                    ts_round<St, SR>(C[j], SR ? (a.cell_base + g * (uint32_t)a.w + col[j]) ^ A.keys[s - 1] : 0u);
                }
            }
            if constexpr (HALF) {
                if (spec) {
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        const int type = (int)(info[j] >> NODE_TYPE_SHIFT);
                        const uint32_t solid = lane_mask(type == CS_WALL || type == CS_LID, 0);  // carried unchanged
                        const T own[9] = {um[0][j], u1[0][j], um[1][j], dc[0][j], um[2][j],
                                          u1[1][j], dc[1][j], dc[2][j], u1[2][j]};
#pragma unroll
                        for (int i = 0; i < 9; ++i) C[j][i] = lane_select(solid, own[i], C[j][i]);
                    }
                }
            }
            if constexpr (EDGE == CS_EDGE_ZERO) {
                const bool rin = r >= 0 && r < a.h;
                if (edge_strip || !rin) {  // uniform over the wave
#pragma unroll
                    for (int j = 0; j < V; ++j)
#pragma unroll
                        for (int i = 0; i < 9; ++i) C[j][i] = lane_select(rin ? inside[j] : 0u, C[j][i], outside(i));
                }
            }
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int i = 0; i < 9; ++i) {
                    N[i][j] = C[j][i];
                }
            if (s < K) {
                e5 = ts_lane<false>(lprev, N[5][V - 1]);
                e8 = ts_lane<true>(lnext, N[8][0]);
            }
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int i = 0; i < 9; ++i) asm volatile("" : "+v"(N[i][j]));
            if (s == K && !FILL) {
                S* orow = fout + (int64_t)r * a.pitch;
                const int l0 = lane * V, oc = c0 + l0;
                if (l0 >= K && l0 < 64 * V - K && oc < a.w && (UNROLL == 1 || r < rb)) {  // V divides K
                    if (vec_out) {                              // uniform over the wave
#pragma unroll
                        for (int i = 0; i < 9; ++i) {
                            VecN<S, V * (int)sizeof(S)> v;
#pragma unroll
                            for (int j = 0; j < V; ++j) v.e[j] = St::nar(N[i][j]);
                            __builtin_nontemporal_store(v.raw, (RawVec<V * (int)sizeof(S)>*)at<uint32_t>(
                                                                   orow + i * a.plane, (uint32_t)oc));
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < V; ++j)
                            if (oc + j < a.w) {
#pragma unroll
                                for (int i = 0; i < 9; ++i)
                                    *at<uint32_t>(orow + i * a.plane, (uint32_t)(oc + j)) = St::nar(N[i][j]);
                            }
                    }
                }
            }
        }
    };
    int t = 0;
#pragma unroll 1
    for (; t < 2 * (K - 1); ++t, ++r1) iteration(std::true_type{}, t);
#pragma unroll 1
    while (t < iters) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u, ++t, ++r1) iteration(std::false_type{}, t);
    }
}

template <class St, int EDGE, int MODE, int K, int COLL, int V, bool SR>
__global__ __launch_bounds__(TS_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_step_ts(
    TsArgs<typename St::T, K> A)
{
    static_assert(K % V == 0 && K + 1 <= TS_RING, "strip halo and node ring");
    using Lds = TsLds<typename St::T, MODE, K, V>;
    __shared__ Lds lds[MODE == MODE_FLUID ? 1 : TS_WAVES];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int id = xcd_tile(blockIdx.x, gridDim.x) * TS_WAVES + wave;
    // the first and the last strip's chunks come first
    const int edges = A.strips > 1 ? 2 : 1, outer = edges * A.edge_chunks;
    int strip, chunk, chunks;
    if (id < outer) {
        strip = id < A.edge_chunks ? 0 : A.strips - 1;
        chunk = id < A.edge_chunks ? id : id - A.edge_chunks;
        chunks = A.edge_chunks;
    } else {
        const int inner = A.strips - edges, k = id - outer;
        if (inner <= 0 || k >= inner * A.chunks) return;
        chunk = k / inner;
        strip = 1 + k - chunk * inner;
        chunks = A.chunks;
    }
    const int ra = (int)((int64_t)A.a.h * chunk / chunks), rb = (int)((int64_t)A.a.h * (chunk + 1) / chunks);
    ts_strip<St, EDGE, MODE, K, COLL, V, SR>(A, strip * (64 * V - 2 * K) - K, ra, rb,
                                             &lds[MODE == MODE_FLUID ? 0 : wave]);
}

}  // namespace cs
