// Real instances of the register-resident eigensolver (krylov_reg.h).
#include "eigen_reg.h"

namespace imped {

bool launch_eigen_reg_real(const EigenArgs& a, unsigned nb, int n_cu, int groups, bool test, hipStream_t s) {
  return launch_eigen_type<double>(a, nb, n_cu, groups, test, s);
}

}  // namespace imped
