// Convergence test of a PCG iteration (device code).
#pragma once
#include "solver.hpp"

namespace et {

// omega of the next V-cycle: min + d/2 exp((-clip(R, tol, 0.1) + tol) * 500)
__device__ __forceinline__ double pcg_omega(double R, double tol, double wmin, double dw) {
  const double Rc = fmin(fmax(R, tol), 1e-1);
  return wmin + dw / 2.0 * exp((-Rc + tol) * 500.0);
}

// What the test reads, loaded ahead of the sum of r.r.
struct PcgState {
  double stop, pq, bb, R, status;
};
__device__ __forceinline__ PcgState pcg_state(const double* sc) {
  return {sc[SC_STOP], sc[SC_PQ], sc[SC_BB], sc[SC_R], sc[SC_STATUS]};
}

// Convergence / breakdown test of one iteration, evaluated on the device so the
// host never waits on the current iteration: R = |r| / |b|; non-finite p.q or r.r,
// p.q <= 0 and R < tol stop the loop (first reason wins, as in a plain sequential
// loop).  While running, omega is set for the next V-cycle.  {R, status, stop} is
// published to pinned host memory (the caller fences).  One thread.
__device__ inline void pcg_check(const PcgCheck& ck, PcgState st, double rr) {
  double* sc = ck.sc;
  if (st.stop == 0.0) {
    const double R = sqrt(rr) / sqrt(st.bb);
    st.R = R;
    st.status = (double)ET_OK;
    if (!isfinite(st.pq) || !isfinite(rr)) {
      st.status = (double)ET_ENONFINITE;
      st.stop = 1.0;
    } else if (!(st.pq > 0.0)) {
      st.status = (double)ET_EBREAKDOWN;
      st.stop = 1.0;
    } else if (R < ck.tol) {
      st.stop = 1.0;
    }
    sc[SC_RR] = rr;
    sc[SC_R] = st.R;
    sc[SC_STATUS] = st.status;
    sc[SC_STOP] = st.stop;
    if (st.stop == 0.0) sc[SC_OMEGA] = pcg_omega(R, ck.tol, ck.wmin, ck.dw);
  }
  ck.ring[0] = st.R;
  ck.ring[1] = st.status;
  ck.ring[2] = st.stop;
}

}  // namespace et
