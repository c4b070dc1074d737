// FP64 instantiations of the streaming temporally blocked step (lbm_ts.hpp):
// BGK, TRT and Regularized in every boundary mode.
#include "lattice_ts.hpp"

namespace cs {
namespace {

template <int EDGE, int MODE>
void f64_coll(cs_lattice* l, int k)
{
    if (k == 4) ts_launch<StF64, EDGE, MODE, 4, CS_COLL_BGK>(l);
    else if (l->params.collision == CS_COLL_TRT) ts_launch<StF64, EDGE, MODE, 8, CS_COLL_TRT>(l);
    else if (l->params.collision == CS_COLL_REGULARIZED) ts_launch<StF64, EDGE, MODE, 8, CS_COLL_REGULARIZED>(l);
    else ts_launch<StF64, EDGE, MODE, 8, CS_COLL_BGK>(l);
}

template <int EDGE>
void f64_mode(cs_lattice* l, int k)
{
    if (!l->has_flags) f64_coll<EDGE, MODE_FLUID>(l, k);
    else if (l->params.boundary == CS_BB_HALFWAY) f64_coll<EDGE, MODE_HALF>(l, k);
    else f64_coll<EDGE, MODE_REF>(l, k);
}

}  // namespace

void launch_ts_f64(cs_lattice* l, int k)
{
    if (l->params.edge == CS_EDGE_PERIODIC) f64_mode<CS_EDGE_PERIODIC>(l, k);
    else f64_mode<CS_EDGE_ZERO>(l, k);
}

}  // namespace cs
