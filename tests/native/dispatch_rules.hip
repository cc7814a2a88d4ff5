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

// Every line end of an element has a thread and a round of the node kernel, whatever
// degree it is built from; at N = 7 one round.
template <int DIM, int N>
constexpr bool faces_covered() {
  using F = NodeFaces<DIM, N>;
  int covered = 0;
  for (int k = 0; k < F::ROUNDS; ++k)
    for (int a = 0; a < F::NN; ++a) covered += a + k * F::NN < F::COUNT ? 1 : 0;
  return covered == 2 * DIM * Shape<DIM, N>::FN;
}
static_assert(faces_covered<2, 1>() && faces_covered<2, 2>() && faces_covered<2, 3>() &&
              faces_covered<2, 4>() && faces_covered<2, 5>() && faces_covered<2, 7>());
static_assert(faces_covered<3, 2>() && faces_covered<3, 3>() && faces_covered<3, 4>() &&
              faces_covered<3, 5>() && faces_covered<3, 7>());
static_assert(NodeFaces<2, 7>::ROUNDS == 1 && NodeFaces<3, 7>::ROUNDS == 1);
