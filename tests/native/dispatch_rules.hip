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

// The pair kernel takes the grids whose blocks fit the device's CUs at once and the
// line kernel's metric table the grids above 100 000 line threads per 256 CUs,
// whatever number of CUs the device has.
template <int N, int F>
constexpr bool pair_line(int64_t E, bool viscous, int cus) {
  return pair_kernel_for<N, F, F>(E, viscous, cus) && !pair_kernel_for<N, F, F>(E + 1, viscous, cus);
}
static_assert(pair_line<3, kFluxLLF>(4096, false, 256) && pair_line<3, kFluxLLF>(512, false, 32));
static_assert(pair_line<5, kFluxLLF>(1024, false, 256) && pair_line<5, kFluxLLF>(128, false, 32));
static_assert(pair_line<7, kFluxLLF>(1024, false, 256) && pair_line<7, kFluxLLF>(512, false, 128));
static_assert(pair_line<3, kFluxHLLC>(3072, false, 256) && pair_line<5, kFluxLLF>(96, true, 32));
static_assert(box_table_for<2, 3>(12500, 256) && !box_table_for<2, 3>(12499, 256));
static_assert(box_table_for<2, 3>(1563, 32) && !box_table_for<2, 3>(1562, 32));
static_assert(box_table_for<3, 3>(1, 256) && box_table_for<3, 3>(1, 32));

// A batch with a workgroup per tile stays within the work-items of a launch.
static_assert(batch_grid(INT32_MAX, 1000, 128) == 1000 && batch_grid(512, 1000, 128) == 512);
static_assert(batch_grid(INT32_MAX, 0, 128) == 1 && batch_grid(0, 1000, 256) == 1);
static_assert((int64_t)batch_grid(INT32_MAX, INT32_MAX, 128) * 128 <= 0xffffffffll &&
              batch_grid(INT32_MAX, INT32_MAX, 128) == 33554431 &&
              batch_grid(INT32_MAX, INT32_MAX, 256) == 16777215);
