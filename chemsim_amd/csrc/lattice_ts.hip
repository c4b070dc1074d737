// Launches of the streaming temporally blocked step kernel (lbm_ts.hpp) for
// single lattices: which lattices take it, how the rows are split over waves,
// and the template dispatch.
//
// A strip of rows costs a fill of K - 1 rows whatever its length, so the
// streaming kernel needs a lattice that keeps every SIMD busy with long runs;
// the region kernels (lbm_tb.hpp) recompute a fixed share instead.  Both
// shares are known before the launch, so the choice (strip_rule.hpp) compares
// them: computed cells per kept cell, the streaming kernel's times what a cell
// costs it more.  Without half-way walls 1.12 (the ratio of measured times to
// computed cells at 1536^2 .. 8192^2 is 1.07 .. 1.14).  The half-way mode's
// region kernel keeps its cells in LDS: 1 for a periodic edge (2% of random
// cells solid, 1800 x 1700 242 -> 192 us per 8 steps); where the lattice's edge
// is a wall 1 too (cavities, us per 8 steps in strips / regions: 1700 x 2100 170 /
// 198, 1721 x 1542 148 / 153), 1.1 for three to five strips (250 x 15000 243 /
// 245, with TRT 316 / 300), 0.95 where every strip is an edge strip (150 x 20000
// 243 / 268), and 1.2 more where the last strip keeps so few columns that an
// inner one holds edge cells (1800 x 1700 192 / 175, 1459 x 2302 217 / 177, 1793 x
// 2600 264 / 255, 2360 x 3000 338 / 365); 1.19 with inlet or outlet cells, whose
// Zou-He divisions run in every row of an edge strip (channels 2048^2 231 / 220,
// 2003 x 2300 240 / 237, 1260 x 3561 247 / 237, 3051 x 1713 262 / 286, 3000^2 406 /
// 463), and 1.3 more with such a last strip (1800 x 1700 235 / 175, 3361 x 3100
// 563 / 540).  More waves than the device holds take a second, nearly empty round:
// 229500 x 48 is 2050 strips on 2048 slots, 455 / 366.
// us per 8 steps (calls of 8 steps in a row), strips / regions: Taylor-Green 2003 x
// 2300 148 / 161, 3000^2 250 / 309, 4096^2 417 / 546; half-way cavity 2048^2 183 /
// 227, 3000^2 308 / 464, 4096^2 517 / 836.  Smaller Taylor-Green lattices in forced
// strips, GLUPS: 1024^2 110 / 174, 1536^2 187 / 218.
//
// FP64 has no region kernels (a region would not fit), and its one-step kernel
// is bound by HBM at 144 bytes per cell update: GLUPS, streaming / one-step,
// 512^2 50 / 35, 1024^2 92 / 39, 2048^2 126 / 40, 4096^2 162 / 43, half-way
// cavity 2048^2 101 / 38.  Lattices of 2^20 cells on take it, of any shape: us per
// 8 steps 1 x 2^20 1948 / 5320, 4 x 300001 586 / 2731, 49 x 30000 161 / 374 (cavity
// 286 / 453), 65601 x 17 102 / 291, 98400 x 16 (one wave over the device's) 143 /
// 376: the one-step kernels compute 64 columns of a narrow lattice too.  The times
// cross lower (512^2 above); the line stays at the size up to which lattices
// are replayed from graphs and cs_lattice_temporal_steps reports one step.  KBC
// keeps the one-step kernel: its 19 divisions per cell already take as long as the
// memory, and the strips' recomputation would add to them.
//
// 16-bit storage rounds every level to 16 bits.  Against the one-step kernel
// (computed cells per kept cell 1.94 at 1536^2, 1.62 at 2048^2, 1.36 at 3072^2,
// 1.27 at 4096^2), GLUPS streaming / one-step:
//   f16 to nearest 165 / 118, 186 / 131, 243 / 144, 268 / 153
//   bf16 to nearest 131 / 110, 150 / 118, 194 / 140, 219 / 150
//   bf16 stochastic 114 / 111, 130 / 121, 170 / 140, 191 / 150
//   f16 stochastic 97 / 111, 117 / 118, 150 / 140, 161 / 150
// so f16 with stochastic rounding takes it only where the fill is small.
// Half-way cavity 2048^2 and 4096^2: f16 148 / 99, 224 / 121 to nearest, 101 /
// 95, 141 / 116 stochastic; bf16 111 / 94, 164 / 115 and 98 / 95, 138 / 118.
// What else moves the line (us per 8 steps, streaming / one-step):
//   wave slots left idle, since the one-step kernels fill the device whatever the
//   shape: 57400 x 288 (513 strips, 3 runs each) f16 stochastic 1032 / 907, 229500
//   x 96 bf16 to nearest 1350 / 1274; f16 to nearest is faster all the same, 975 /
//   1262;
//   inlets and outlets with stochastic rounding (f16 / bf16 2048^2 364 / 331, 379 /
//   331; 3000^2 634 / 628, 659 / 627; 4096^2 1073 / 1131, 1121 / 1126; bf16 3710 x
//   3135 819 / 780);
//   a solid mask: bf16 stochastic 2048^2 with a few obstacles 294 / 271, with 2%
//   of random cells 306 / 272, 3000^2 520 / 536; bf16 to nearest 1500^2 182 / 170,
//   1800 x 1700 220 / 223; f16 stochastic 4100 x 1517 396 / 382, 9100 x 817 466 / 468;
//   a wall in an inner strip (FP32 above): bf16 stochastic cavity 2353 x 3000 577 /
//   539, 3361 x 3100 779 / 737;
// against the one-step kernels' tiles of 256 columns in these modes, which a
// narrow lattice leaves half empty: 101 x 30011 channel bf16 stochastic 375 / 417.
//
// A 4-step remainder launch recomputes less in strips and in regions alike (a
// 64 x 64 region keeps 56 x 56), so its line is its own: us per 4 steps, strips /
// regions, 4096^2 309 / 337, 1794 x 3541 126 / 130, 2893 x 1432 95 / 91, 1100 x 4003
// 92 / 91; with a solid mask 3000^2 190 / 202, 1780 x 2635 108 / 102, 1100 x 4003
// 103 / 96; cavity 2048^2 101 / 140, 49 x 60000 (one region wide) 164 / 148,
// channel 201 / 143; 101 x 30011 (one strip) 79 / 83.  FP64, which has no
// regions: 0.35 to 0.55 of four single steps.
#include "lattice_ts.hpp"
#include "lbm_tb.hpp"

using namespace cs;

namespace {

template <class St, int EDGE, int MODE>
void ts_coll(cs_lattice* l, int k)
{
    if (k == 4) {  // the remainder launch, BGK only
        ts_launch<St, EDGE, MODE, 4, CS_COLL_BGK>(l);
        return;
    }
    if constexpr (std::is_same_v<St, StF32>) {
        if (l->params.collision == CS_COLL_TRT) {
            ts_launch<St, EDGE, MODE, 8, CS_COLL_TRT>(l);
            return;
        }
        if (l->params.collision == CS_COLL_REGULARIZED) {
            ts_launch<St, EDGE, MODE, 8, CS_COLL_REGULARIZED>(l);
            return;
        }
    }
    ts_launch<St, EDGE, MODE, 8, CS_COLL_BGK>(l);
}

template <class St, int EDGE>
void ts_mode(cs_lattice* l, int k)
{
    if (l->has_flags && l->params.boundary == CS_BB_HALFWAY) ts_coll<St, EDGE, MODE_HALF>(l, k);
    else if (l->has_flags) ts_coll<St, EDGE, MODE_REF>(l, k);
    else ts_coll<St, EDGE, MODE_FLUID>(l, k);
}

template <class St>
void ts_edge(cs_lattice* l, int k)
{
    if (l->params.edge == CS_EDGE_PERIODIC) ts_mode<St, CS_EDGE_PERIODIC>(l, k);
    else ts_mode<St, CS_EDGE_ZERO>(l, k);
}

}  // namespace

namespace cs {

static_assert(TS_REGION_EDGE == TB_EDGE && ts_cells<float>() == 2, "what strip_rule.hpp counts");
bool ts_takes(const cs_lattice* l) { return ts_takes(strip_case(l)); }
bool ts_takes_remainder(const cs_lattice* l) { return ts_takes_remainder(strip_case(l)); }

void launch_ts(cs_lattice* l, int k)
{
    if (l->storage == CS_F64) launch_ts_f64(l, k);
    else if (storage_bytes(l->storage) == 2) launch_ts_16(l);
    else if (l->storage == CS_F32) ts_edge<StF32>(l, k);
    else ts_edge<StF32Dev>(l, k);
}

}  // namespace cs
