// Register-resident Krylov basis of one chain per workgroup: the pieces the
// fully reorthogonalized Lanczos kernels share.
//
// A Gram-Schmidt step reads the whole basis twice (dots, update), so where
// the basis sits decides the step's time.  The register file is the largest
// memory of a CU (512 KB, against 160 KB of LDS), so the basis goes there
// first: a chain runs on G groups of NQ waves; wave (g, q) owns rows
// (r NQ + q) 64 + lane, r < R, of every vector, and of the basis vectors
// those with l % G == g.  Its vector g + G li sits in registers for li < S
// (reg_slots, at two waves per SIMD), in LDS for the
// next kl of them, in memory beyond.  Every element of the basis is read only
// by the thread that wrote it, so no barrier guards the basis itself.
//
// Dots: a thread's products are reduced over the wave by a halving network
// (v_permlane32_swap, v_permlane16_swap, then DPP): eight values at once take
// 34 instructions, where eight wave sums take 144.  Partial sums of the NQ
// row waves meet in LDS (one barrier); each wave adds the coefficients of its
// own vectors and the update reads them as LDS broadcasts.  With G > 1 the
// groups' updates meet in LDS (one more barrier).
//
// The order of every sum is a function of the chain alone: a sum over the basis
// vectors is formed in kRegParts parts (index mod kRegParts, each in order), of which a
// group holds kRegParts / G, and added as (p0 + p2) + (p1 + p3); a row of H in
// kRegRowParts likewise; sums over the rows go by lane, row block and wave, and blocks
// past the chain's end add zeros.  So NQ, G, R, the element type (for a real or
// imaginary start vector), the place of a vector, and with them the other chains of a
// launch, change no bit of a chain's result: its eigenvectors seed plain recurrences
// whose unconverged part amplifies last bits, and a model must not depend on its batch.
#pragma once

#include "common.h"

namespace imped {

struct EigenArgs;

struct LanczosArgs {
  const int64_t* row_base;
  const int64_t* chain_n;
  const int64_t* rowptr;
  const int32_t* col;
  const double2* val;
  const double2* v0;
  int K;
  int reorth;
  double2* ws;      // 3 vectors per chain at 3*row_base
  double2* vstore;  // reorth: K vectors per chain at K*row_base (coefficients in LDS)
  double* alpha;
  double* beta;
  int32_t* kout;
  int32_t* status;
  const int32_t* chain_list;  // chains handled by this launch, one per workgroup
  int nmax;                   // register kernels: rows of the launch's largest chain,
  int kl;                     // LDS-held vectors per group of waves,
  const int32_t* pure;        // and, with a real H, per chain 1 when its start vector is real or imaginary
};

// Chains of up to this many rows run on the register kernels.
constexpr int64_t kRegMaxN = 1024;
constexpr int kRegLds = 160 * 1024;  // LDS of a CU
constexpr int kRegParts = 4;         // parts of a sum over the basis: the largest number of groups
constexpr int kRegRowParts = 2;      // parts of a row's sum

// Whether an n-row chain of K steps runs there (its coefficients fit the LDS).
bool lanczos_reg_fits(int64_t n, int K);
// Launch class of an n-row chain: chains of one class share a launch.
inline int lanczos_reg_class(int64_t n) {
  const int64_t rows = (n + 63) / 64;
  return (int)(rows <= 4 ? std::max<int64_t>(rows, 1) - 1 : 4 + (rows - 5) / 4);
}
constexpr int kRegClasses = 7;

// nb chains (a.chain_list, at most a.nmax <= kRegMaxN rows each), reorth = 1,
// on the register kernels; groups: cap on the groups of waves per chain (1, 2
// or 4).  a.pure (null: all 0): chains with 1 (real) or 2 (imaginary start
// vector; H real) run in the real launch, the others in the complex one.
void launch_lanczos_reg_real(const LanczosArgs& a, unsigned nb, int n_cu, int groups, hipStream_t s);
void launch_lanczos_reg_cplx(const LanczosArgs& a, unsigned nb, int n_cu, int groups, hipStream_t s);

// The eigensolver on the same basis: nb chains of at most a.nmax <= kRegMaxN
// rows; with test nothing is launched and the result says whether the launch's
// arrays fit the LDS (for every number of groups when for 4).
bool launch_eigen_reg_real(const EigenArgs& a, unsigned nb, int n_cu, int groups, bool test, hipStream_t s);
bool launch_eigen_reg_cplx(const EigenArgs& a, unsigned nb, int n_cu, int groups, bool test, hipStream_t s);

}  // namespace imped
