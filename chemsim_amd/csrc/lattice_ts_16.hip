// 16-bit instantiations of the streaming temporally blocked step (lbm_ts.hpp):
// every boundary mode, round to nearest and stochastic rounding.
#include "lattice_ts.hpp"

namespace cs {
namespace {

template <class St, int EDGE, int MODE>
void dev16_round(cs_lattice* l)
{
    if (l->params.rounding == CS_ROUND_STOCHASTIC) ts_launch<St, EDGE, MODE, 8, CS_COLL_BGK, true>(l);
    else ts_launch<St, EDGE, MODE, 8, CS_COLL_BGK>(l);
}

template <class St, int EDGE>
void dev16_mode(cs_lattice* l)
{
    if (!l->has_flags) dev16_round<St, EDGE, MODE_FLUID>(l);
    else if (l->params.boundary == CS_BB_HALFWAY) dev16_round<St, EDGE, MODE_HALF>(l);
    else dev16_round<St, EDGE, MODE_REF>(l);
}

template <class St>
void dev16_edge(cs_lattice* l)
{
    if (l->params.edge == CS_EDGE_PERIODIC) dev16_mode<St, CS_EDGE_PERIODIC>(l);
    else dev16_mode<St, CS_EDGE_ZERO>(l);
}

}  // namespace

void launch_ts_16(cs_lattice* l)
{
    if (l->storage == CS_BF16DEV) dev16_edge<StBF16>(l);
    else dev16_edge<StF16>(l);
}

}  // namespace cs
