// Complex instances of the register-resident Lanczos (krylov_reg.h).
#include "lanczos_reg.h"

namespace imped {

void launch_lanczos_reg_cplx(const LanczosArgs& a, unsigned nb, int n_cu, int groups, hipStream_t s) {
  launch_reg_type<double2>(a, nb, n_cu, groups, s);
}

bool lanczos_reg_fits(int64_t n, int K) {
  if (n > kRegMaxN) return false;
  const int k = (int)std::min<int64_t>(K, n);
  switch (lanczos_reg_class(n)) {
    case 0:
    case 1:
    case 2:
    case 3:
      return true;  // at most 256 rows and steps
    case 4:
      return lanczos_reg_fixed<4, 2, 2, double2>(n, k) * 8 <= (size_t)kRegLds;
    case 5:
      return lanczos_reg_fixed<4, 2, 3, double2>(n, k) * 8 <= (size_t)kRegLds;
    default:
      return lanczos_reg_fixed<4, 2, 4, double2>(n, k) * 8 <= (size_t)kRegLds;
  }
}

}  // namespace imped
