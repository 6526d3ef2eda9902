// Loss of orthogonality of a Lanczos basis, estimated on the host from the
// recurrence coefficients alone.
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

namespace imped {

// Estimates of the inner products <v_j, v_k>, k < j, of the Lanczos vectors of
// one chain (H. D. Simon, "The Lanczos algorithm with partial
// reorthogonalization", Math. Comp. 42, 1984):
//   b_j w_{j+1,k} = b_k w_{j,k+1} + (a_k - a_j) w_{j,k} + b_{k-1} w_{j,k-1}
//                   - b_{j-1} w_{j-1,k} + rounding of order eps (b_k + b_j + |a_k| + |a_j|),
// the last two terms being the rounding of H v and of w - a v.  The basis then
// needs a Gram-Schmidt pass only in the steps where an estimate passes
// kOrthLevel (and in the step after, since two vectors feed the next one).
//
// The recurrence has to run on H - sigma, sigma = a_0: a sector's energies lie
// hundreds of hopping widths from zero, and rounding of order eps |a| / b then
// passes the level in every step (|a|/b > 450), or, left out of the estimate, lets
// the basis go ten to a hundred times past it.
//
// The level: a basis orthogonal to w gives Ritz residuals of up to w |H - sigma|, and
// full passes on H leave eps |H|, so w = 8 eps |H| / |H - sigma| (norms from the
// recurrence so far) loses nothing, at most 1e-13.  Below 1e-14 most steps would pass
// anyway, and all do.  Measured in 64-bit numpy, 200 steps, two start vectors each,
// residual of the worst of three pairs with full passes on H -> here (passes):
//   ground sector, 780 states, energies near -900   3.0e-13 -> 2.9e-14 (45)
//   random, 3000 states, width 20, at -900          3.0e-13 -> 3.1e-14 (42)
//   random, 800 states, width 150, at -900          2.2e-13 -> 6.5e-14 (70)
// the errors of the eigenvalues falling from 2e-13 to 1e-14.  A level of 1e-13 throughout
// took 44 to 48 passes, with residuals of 1.8e-12 for 2.0e-13 on a spectrum of width 700
// at -700; 16 eps in place of 8 eps left 4.1e-13 there.
constexpr double kOrthLevel = 1e-13;

struct OrthEstimate {
  std::vector<double> w, w_old, next;  // w[k] of the latest vector, of the one before, and work
  std::vector<double> a, b;
  bool again = false;                  // the step after a pass
  double sigma, norm = 0.0;            // |H - sigma| so far

  explicit OrthEstimate(double shift) : w{1.0}, sigma(std::fabs(shift)) {}
  // After step j's three-term update (alpha_j = al, |w| = bt): whether
  // v_{j+1} needs a pass against v_0..v_j.
  bool step(double al, double bt) {
    constexpr double eps = 2.2e-16;
    const int j = (int)a.size();
    a.push_back(al);
    norm = std::max(norm, std::fabs(al) + bt + (j > 0 ? b[j - 1] : 0.0));
    const double level = std::min(kOrthLevel, 8.0 * eps * (sigma + norm) / norm);
    const bool every = !(level >= 1e-14);
    next.assign(j + 2, 0.0);
    next[j + 1] = 1.0;
    double worst = 0.0;
    for (int k = 0; k < j; ++k) {
      double t = b[k] * w[k + 1] + (a[k] - al) * w[k] - b[j - 1] * w_old[k];
      if (k > 0) t += b[k - 1] * w[k - 1];
      t += std::copysign(eps * (2.0 * (b[k] + bt) + std::fabs(a[k]) + std::fabs(al)), t);
      next[k] = t / bt;
      worst = std::max(worst, std::fabs(next[k]));
    }
    next[j] = eps * (std::fabs(al) + bt + (j > 0 ? b[j - 1] : 0.0)) / bt;  // rounding of alpha_j
    worst = std::max(worst, std::fabs(next[j]));
    const bool pass = every || again || !(worst <= level) || !(bt > 0.0);
    again = pass && !again;
    return pass;
  }
  // beta_j as it came out; the estimates move on to v_{j+1}
  void done(double bt, bool passed) {
    if (passed) std::fill(next.begin(), next.end() - 1, 2.2e-16);
    b.push_back(bt);
    w_old.swap(w);
    w.swap(next);
  }
};

}  // namespace imped
