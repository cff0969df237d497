// Fused legs of a 2-D V(2,2) cycle (see vcycle_2d.hip).
#pragma once
#include "common.hpp"

namespace et {

// Convergence test of a PCG iteration: r.r from its n_rr partials, status and stop flag into sc
// (SC_* slots) and {R, status, stop} to pinned host memory (pcg_check.hpp).
struct PcgCheck {
  double* sc = nullptr;
  const double* rr_part = nullptr;
  int n_rr = 0;
  double tol = 0, wmin = 0, dw = 0;
  double* ring = nullptr;
};

// workgroups of either leg (partial sums written by vcycle2_up when part is given)
int vcycle2_tiles(const Grid& g);

// x1 = two Jacobi sweeps from the zero guess, r = b - A x1, bc = R r (g.coarse()).
// op: K0 (8 x 8, with E and cons) on level 0, else the half-stored block stencil.  With ck (level 0),
// the test of the iteration runs first and omega is the one it sets.
template <typename T>
int vcycle2_down(const Grid& g, bool level0, const T* op, const T* E, const uint8_t* cons, const T* b, const T* Dinv,
                 const double* omega, double wscale, T* x1, T* r, T* bc, const PcgCheck* ck, hipStream_t s);

// e = two Jacobi sweeps on A e = r from e0 = P xc, x = x1 + e; part (level 0 only, may be null): sums of bdot.x
template <typename T>
int vcycle2_up(const Grid& g, bool level0, const T* op, const T* E, const uint8_t* cons, const T* xc, const T* r,
               const T* x1, const T* Dinv, const double* omega, double wscale, T* x, const double* bdot, double* part,
               hipStream_t s);

}  // namespace et
