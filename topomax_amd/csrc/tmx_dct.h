// Exact fast solver of a spectrally equivalent operator of the filter, used as its PCG
// preconditioner (FP32 in the mixed scheme, FP64 in the FP64 scheme).
//
// With natural boundary conditions on the structured 'right' mesh the filter stiffness is a
// sum of Kronecker products of 1D Neumann Laplacians T (tridiag(-1, 2, -1), boundary diagonal
// 1) with the boundary half-weights W = diag(1/2, 1, ..., 1, 1/2):
//   eps^2 K = eps^2 (hy/hx) W_y (x) T_x + eps^2 (hx/hy) T_y (x) W_x   (y outer, x inner).
// The consistent mass is not such a sum: each of its triangles couples the ends of its cell's
// diagonal.  Its average over the two ways to draw the diagonals is one, with C = W - T / 2:
//   M' = (hx hy / 12) [6 W_y (x) W_x + 2 W_y (x) C_x + 2 C_y (x) W_x + 2 C_y (x) C_x],
// and A' = eps^2 K + M' is diagonalised by the DCT-I in y: T_y v_m = lambda_m W_y v_m with
// v_m[j] = cos(pi j m / n), lambda_m = 2 - 2 cos(pi m / n), v_m' W_y v_k = D_m delta_mk
// (D_m = n / 2, or n for m = 0, n).  So A'^-1 r = sum_m v_m (x) X_m^-1 (v_m' r) / D_m with
//   X_m = (eps^2 hy/hx - hx hy (2 - lambda_m / 2) / 12) T_x
//         + (eps^2 (hx/hy) lambda_m + hx hy (1 - lambda_m / 6)) W_x,
// diagonally dominant for any eps: a DCT-I along y, one tridiagonal solve along x per mode
// (partition method: block eliminations, cyclic reduction of the blocks' interface system in
// LDS), and the same DCT-I again (the matrix C[j, m] = cos(pi j m / n) is symmetric).  A - A' is
// the diagonals' antisymmetric part, (hx hy / 6) sin sin in the symbols: with eps/h = 1 the
// spectrum of A'^-1 A is 1 -+ 0.046, against [0.86, 1] for the lumped mass hx hy W_y (x) W_x
// (TMX_OPT_FILTER_DCT 1), and both come close to 1 as eps/h grows.  PCG iterations of a filter
// solve to 1e-11, two solves a step, lumped / averaged:
// 60 x 20 cells (eps/h = 1) 8 + 8 / 7 + 8, 40 x 40 (0.8) 9 + 9 / 8 + 8, 320 x 160 6 + 6 / 5 + 6,
// 640 x 320 and above the same.
//
// The DCT-I of the n + 1 values of a y-column is computed from a complex FFT of length 2n in
// LDS (k_dct1_cols): two columns a, b are packed as a + i b and extended evenly
// (z[2n - j] = z[j]); the DFT of a real even sequence is real, so the real and imaginary parts
// of the FFT are the two columns' transforms, up to the end-point terms
//   T[m] = (Y[m] + r_0 + (-1)^m r_n) / 2,   Y = DFT_2n of the even extension.
// The FFT is a mixed-radix Stockham transform (radices 2, 3, 4, 5, 7, and direct sums for the
// primes from 11 to kMaxPrime); other grids keep the multigrid V-cycle.
#pragma once

#include "tmx_kernels.h"
#include "tmx_solver.h"

namespace tmx {

// radix plan of one FFT length (stages applied in order)
struct FftPlan {
  static constexpr int kMaxStages = 16;
  int L = 0;
  int nstages = 0;
  int radix[kMaxStages] = {};
  bool direct = false;  // some radix has no butterfly of its own
};

// the radix plan of length L: the prime factors above 7 first (none above max_prime; false when
// there is one), then radices 4, 2, 3, 5, 7
bool fft_plan(int L, int max_prime, FftPlan& plan);

template <typename T>
class DctPrecond {
 public:
  // nx, ny: cells; 2 ny has no prime factor above max_prime (7 or kMaxPrime; above 7 on grids
  // of more than kMinNodesDirect nodes only), nx + 1 <= kMaxRow, and the FFT of 2 ny points fits
  // the LDS budget
  static bool supported(int nx, int ny, int max_prime);
  // eps: the filter's length scale
  int init(int nx, int ny, double hx, double hy, double eps, hipStream_t s);
  // z = A'^-1 r (vectors of (nx + 1)(ny + 1) values; lumped: with the lumped mass in A'),
  // partials of r.z into rz if given
  int apply(const T* r, T* z, bool lumped, RedSlot* rz, hipStream_t s);

  // Whether a filter solve with it is faster than with the V-cycle: always without direct stages;
  // with them, by the estimated time of an iteration, in us, times the iterations.
  //  - DCT: a direct stage of radix p takes p products a point (fft_stage_direct), in each
  //    thread one after the other: 0.077 us for each of the p ceil(2 ny / 256) products, while a
  //    CU has no more than one workgroup (two columns); several share the LDS.  The rest of an
  //    iteration takes 43 + ny / 50.
  //  - V-cycle: about 49 for 4000 nodes and 6 more for each doubling; 77 when the finest level
  //    is coarsened to a nested one.
  //  - iterations for eps/h = 1, 2, 5, 16, 50: DCT 7, 6, 5, 4, 3 (12 at 1/4), V-cycle 6 to 8.
  // Solves of 9430 combinations of nx = 2 .. 2999, ny = 11 .. 2000 with a largest prime of 11 to
  // 443, and eps/h = 1/4 .. 50 (seeded random rho, to 1e-11) take 0.6% more on average than with
  // the faster of the two for each; 38% more with the V-cycle throughout, 25% with the DCT.
  // V-cycle / DCT in us, FP64: 333 x 111 cells with eps/h = 8 (p = 37) 550 / 252, 512 x 257 with
  // 16 702 / 542 and with 1.5 629 / 889, 16 x 257 with 16 426 / 558, 4 x 347 369 / 645,
  // 512 x 1041 (p = 347) 1078 / 2000.
  static bool pays(int nx, int ny, double hx, double hy, double eps);

  // largest prime factor of 2 ny that has a direct stage
  static constexpr int kMaxPrime = sizeof(T) == 4 ? 450 : 350;
  // fewest nodes of a grid that such a prime's transform is used on: the V-cycle of a smaller
  // one is a few launches (33 x 11 cells 296 / 413, 66 x 22 490 / 352)
  static constexpr size_t kMinNodesDirect = 1024;
  // longest x row: one workgroup of 256 threads solves it, 12 rows per thread, with the row
  // and two coefficient arrays in LDS (40 KB in FP32, 80 KB in FP64 at this length)
  static constexpr int kMaxRow = 3072;
  // fewest y-columns per FFT workgroup (two per complex sequence of 2 ny points; ny <= 2048);
  // four when their sequences and the twiddle table fit 64 KB of LDS
  static constexpr int kCols = 2;

 private:
  int nx_ = 0, ny_ = 0, mx_ = 0;
  double hx_ = 0, hy_ = 0, eps_ = 0;
  FftPlan plan_;
  DevBuf<T> tw_;  // twiddles exp(-2 pi i k / 2n), k < 2n, as (re, im) pairs
  DevBuf<T> t_;   // transformed modes: row m = mode m (n + 1 rows of nx + 1 values)
};

}  // namespace tmx
