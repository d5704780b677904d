// resident_f32.hip -- the resident conjugate-gradient kernels of the mixed solver.
#include "resident_kernel.h"

namespace afem {
namespace resident {

void launch_f32(const Args& a, int rows, bool idx16, int grid, size_t lds)
{
  if (idx16)
    launch_kernel<float, 0, true>(a, rows, grid, lds);
  else
    launch_kernel<float, 0, false>(a, rows, grid, lds);
}

} // namespace resident
} // namespace afem
