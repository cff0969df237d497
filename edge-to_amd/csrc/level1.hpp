// Matrix-free operator of the first coarse multigrid level (3-D, even element
// counts): A_1 = R A_hat R^T applied element by element from the fine element
// densities, with stored rows at the coarse nodes that constrained fine DOFs
// reach.  See level1.hip.
#pragma once
#include "common.hpp"

namespace et {

// Tiling of the level-1 operator (level1.hip).
struct L1Plan {
  int cx, cy;    // element columns per tile
  int ntx, nty;  // tiles along x, y
  int zl, ntz;   // nodes per tile along z, tiles along z
  int lpc, cpw;  // lanes per element column, columns per wavefront
  bool split;    // one output component per wavefront
};

struct Level1MF {
  Grid g0{}, g1{};
  bool mixed = false;         // FP32 apply (else FP64)
  void* cf = nullptr;         // element coefficients (kL1Terms, working precision)
  void* Eh = nullptr;         // per coarse element: transform of its 8 children's E [n_elem1][8]
  uint8_t* special = nullptr; // per coarse element: a child touches a constrained DOF
  int* aidx = nullptr;        // per coarse node: row in the correction list, or -1
  int* alist = nullptr;       // corrected coarse nodes
  int* acount = nullptr;      // device counter
  int* acount_h = nullptr;    // pinned copy
  int n_aff = 0;
  void* rows = nullptr;       // operator rows of the corrected nodes [n_aff][27][3][3], working precision
  int rows_cap = 0;
  L1Plan plan{};

  int init(const Grid& fine, const double* K0_host, bool mixed_, hipStream_t s);
  // After the level-1 Galerkin stencil S1 (true operator, FP64) has been built
  // from E, cons and the element flags: refresh E transforms and rows.
  int setup(const double* E, const uint8_t* eflag, const double* S1, hipStream_t s);
  // Level-1 operator in the smoother modes (0 y = Ax, 1 b - Ax, 2 Jacobi, 3 Jacobi + add).
  template <typename T>
  int apply(int mode, const T* x, const T* b, const T* Dinv, const double* omega, double wscale,
            const T* xadd, T* y, hipStream_t s) const;
  void release();
};

bool level1_supported(const Grid& fine, int n_level);
// whether the fixed term list of the element product holds every entry of
// H M_0 H / 64 above rtol * max for this element matrix (host)
bool level1_terms_cover(const double* K0_host, double rtol);
void set_level1_mf(int on);
int get_level1_mf();

}  // namespace et
