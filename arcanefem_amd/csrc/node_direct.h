// node_direct.h -- right-hand sides of plane meshes in one launch: L lanes per
// node, each forming the term of one (node, cell) pair.
#pragma once

#include "common.h"
#include "device_utils.h"

namespace afem {

// rhs[i * nb_dof + dof_index] = (add: +=) the sum of term(item) over the
// node->cell items of node i.  A plane node has few cells (6 triangles, 4
// quads), so forming a term once per node of the cell costs less than a
// second launch: on 400 x 400 quads of triangles 9.8 us with four lanes, 12
// with terms per cell and a sum per node; numbered at random 29 us, 38 with
// one thread per node.  In space (24 tetrahedra or 8 hexas a node) the terms
// per cell win by far.
template <int L, class TERM>
__global__ void __launch_bounds__(256)
k_node_direct(int32_t nb_node, const int32_t* __restrict__ nc_off, const int32_t* __restrict__ nc_items, TERM term,
              int add, int nb_dof, int dof_index, double* __restrict__ rhs)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = (int)(t & (L - 1));
  const int32_t i = (int32_t)(t / L);
  double s = 0.0;
  if (i < nb_node) {
    const int32_t e1 = nc_off[i + 1];
    for (int32_t e = nc_off[i] + lane; e < e1; e += L)
      s += term(nc_items[e]);
  }
  s = group_reduce_sum<L>(s);
  if (i < nb_node && lane == 0) {
    double* r = rhs + (int64_t)i * nb_dof + dof_index;
    *r = add ? *r + s : s;
  }
}

template <int L, class TERM>
inline void node_direct(const afem_mesh& m, const TERM& term, bool add, int nb_dof, int dof_index, double* rhs)
{
  hipLaunchKernelGGL((k_node_direct<L, TERM>), dim3(grid_for((int64_t)m.nb_node * L, 256)), dim3(256), 0, stream(),
                     m.nb_node, m.nc_offsets.p, m.nc_items.p, term, add ? 1 : 0, nb_dof, dof_index, rhs);
  check_launch("node_direct");
}

} // namespace afem
