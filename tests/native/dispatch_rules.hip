// The compile-time rules that choose between kernels, at the sizes where they
// must hold.  Compiled for the host only; every check is a static_assert.
#include <hip/hip_runtime.h>

#include "../../dgsem_amd/csrc/adjoint_impl.hpp"

using namespace dgsem;
using namespace dgsem::detail;

// The shock-capturing adjoint forms its subcell cotangents in all directions at
// once in 3D up to N = 3.
static_assert(par_subcell_adjoint<3, 2>() && par_subcell_adjoint<3, 3>());
static_assert(!par_subcell_adjoint<3, 4>() && !par_subcell_adjoint<2, 3>());
