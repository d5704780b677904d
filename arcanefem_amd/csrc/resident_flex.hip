// resident_flex.hip -- the resident flexible conjugate-gradient kernels with a
// sparse preconditioner.
#include "resident_kernel.h"

namespace afem {
namespace resident {

void launch_flex(const Args& a, int rows, bool idx16, bool bf16, int grid, size_t lds)
{
  if (bf16) // comes with 16-bit offsets
    launch_kernel<float, 16, true>(a, rows, grid, lds);
  else if (idx16)
    launch_kernel<float, 32, true>(a, rows, grid, lds);
  else
    launch_kernel<float, 32, false>(a, rows, grid, lds);
}

} // namespace resident
} // namespace afem
