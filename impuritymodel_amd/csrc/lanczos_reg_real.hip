// Real instances of the register-resident Lanczos (krylov_reg.h).
#include "lanczos_reg.h"

namespace imped {

void launch_lanczos_reg_real(const LanczosArgs& a, unsigned nb, int n_cu, int groups, hipStream_t s) {
  launch_reg_type<double>(a, nb, n_cu, groups, s);
}

}  // namespace imped
