// Unpreconditioned Krylov solvers on a matrix-free operator (the structured
// grid operator or the general-mesh operator, KrylovOp): conjugate gradients
// and restarted GMRES, the iterations of CuCG / CuGMRES (solvers/_gpu.py:11-107),
// which hand the stiffness operator to cupyx.scipy.sparse.linalg.cg / gmres.
//
// CG (cupyx cg semantics): atol = tol |b|; rho = r.r, beta = rho / rho_old,
// p = r + beta p, q = A p, alpha = rho / p.q, x += alpha p, r -= alpha q,
// stop when |r| <= atol.  A small system is bound by the chain of launches, so an iteration is as
// few as possible: on an assembled operator two, the row pass (the test of the previous step,
// p = r + beta p formed while it is gathered, q = A p, p.q) and the x / r update; on any other
// operator four (p update with the test, operator, p.q, x / r update).  28 611 unknowns, 1.2 M
// entries: 25 us per iteration in five launches, 12 us in two.  The state lives on the device
// and every kernel here returns at once after the stop, so the host enqueues chunks of iterations and
// reads the state once per chunk.
//
// GMRES(m) (cupyx gmres semantics): each cycle forms r = b - A x, stops if
// |r| <= atol, runs m Arnoldi steps with one classical Gram-Schmidt pass per
// step (h = V^T u, u -= V h, H[j+1, j] = |u|) and then solves the (m+1) x m
// least-squares problem on the host (Givens rotations) and updates x += V y.
// The convergence test is once per cycle, as in the reference.
//
// All reductions are two-stage with a fixed block count, so results are
// reproducible run to run.  The caller provides the workspace (krylov_work_size).
#include <algorithm>
#include <cmath>
#include <vector>

#include "blas.hpp"
#include "common.hpp"
#include "stiffness.hpp"

namespace et {

// State of the iterations.  Iteration k reads slot (k - 1) & 1 and writes slot k & 1 (the first reads
// slot 1), so no kernel reads a slot that one of its own blocks writes.
struct CgSlot {
  double rho;
  int stop, iters;
};
struct CgState {
  CgSlot slot[2];
  double atol2, bb, rr0;  // rr0: r.r before the first step
  // what the host reads: written by cg_report_kernel
  double rr;
  int stop, iters;
};

// iterations enqueued between two reads of the state, at least and at most
constexpr int kCgChunk = 8, kCgChunkMax = 64;

// Iterations to enqueue next, done of them behind |r|^2 = rr0 -> rr.  Each read drains the queue (about
// 20 us, two steps of an assembled operator), and the steps enqueued past the stop are wasted.  On an
// assembled operator these are empty launches: half of the steps that the mean rate so far leaves.
// On any other the product runs all the same, at a step's full price: the shortest chunk.  Tetrahedra
// matrix-free, 16 iterations: 2.4 ms; with a longer chunk after the first read 8.8 ms.
static int cg_chunk(bool assembled, int done, double rr0, double rr, double atol2) {
  if (!assembled) return kCgChunk;
  const double rate = std::log(rr0 / rr), left = std::log(rr / atol2);
  const double est = rate > 0.0 ? left / rate * done / 2 : kCgChunkMax;
  return (int)std::fmin(std::fmax(est, (double)kCgChunk), (double)kCgChunkMax);
}

// r (interleaved with the search direction, so that one gather fetches both)
struct alignas(8) CgPair {
  double r, p;
};

// partial sums of b.b and r.r; with rp also rp = {r, 0}
__global__ __launch_bounds__(256) void cg_start_kernel(int64_t n, const double* __restrict__ b,
                                                       const double* __restrict__ r, CgPair* __restrict__ rp,
                                                       double* __restrict__ part_bb, double* __restrict__ part_rr) {
  double sb = 0.0, sr = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
    const double bv = b[t], rv = r[t];
    sb += bv * bv;
    sr += rv * rv;
    if (rp != nullptr) rp[t] = CgPair{rv, 0.0};
  }
  sb = block_sum256(sb);
  sr = block_sum256(sr);
  if (threadIdx.x == 0) {
    part_bb[blockIdx.x] = sb;
    part_rr[blockIdx.x] = sr;
  }
}

__global__ void cg_init_kernel(const double* __restrict__ part_bb, const double* __restrict__ part_rr, int nb,
                               double tol, CgState* st) {
  double bb = 0.0, rr = 0.0;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) {
    bb += part_bb[t];
    rr += part_rr[t];
  }
  bb = block_sum256(bb);
  rr = block_sum256(rr);
  if (threadIdx.x == 0) {
    const double atol = tol * sqrt(bb);
    st->bb = bb;
    st->atol2 = atol * atol;
    // |r| <= atol before any step stops at once (|b| = 0 is handled by the host)
    st->slot[1] = CgSlot{rr, bb == 0.0 || rr <= st->atol2 ? 1 : 0, 0};
    st->rr = st->rr0 = rr;
    st->stop = st->slot[1].stop;
    st->iters = 0;
  }
}

// The convergence test of step k - 1 and the start of step k, evaluated by every block from the same
// partials in the same order; block 0 records it.  Returns whether step k runs; beta = rho / rho_old
// (0 on the first step).
__device__ __forceinline__ bool cg_begin(CgState* st, int k, const double* __restrict__ part_rr, int nb,
                                         double& beta) {
  const CgSlot prev = st->slot[(k + 1) & 1];
  CgSlot cur = prev;
  beta = 0.0;
  if (k > 0 && !prev.stop) {
    double rr = 0.0;
    for (int t = threadIdx.x; t < nb; t += blockDim.x) rr += part_rr[t];
    rr = block_sum256_all(rr);
    cur.rho = rr;
    cur.iters = k;
    cur.stop = rr <= st->atol2 || !(rr == rr) ? 1 : 0;
    beta = rr / prev.rho;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) st->slot[k & 1] = cur;
  return !cur.stop;
}

// p = r (first step) or p = r + beta p
__global__ __launch_bounds__(256) void cg_p_kernel(int64_t n, CgState* __restrict__ st, int k,
                                                   const double* __restrict__ part_rr, int nb,
                                                   const double* __restrict__ r, double* __restrict__ p) {
  double beta;
  if (!cg_begin(st, k, part_rr, nb, beta)) return;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x)
    p[t] = k == 0 ? r[t] : r[t] + beta * p[t];
}

__global__ __launch_bounds__(256) void cg_pq_kernel(int64_t n, const CgState* __restrict__ st, int k,
                                                    const double* __restrict__ p, const double* __restrict__ q,
                                                    double* __restrict__ partial) {
  if (st->slot[k & 1].stop) return;
  double s = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x)
    s += p[t] * q[t];
  s = block_sum256(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// Step k of an assembled operator up to p.q: p = r + beta p formed for every gathered entry and
// stored for the own row, q = A p, per-block sums of p.q.  8 lanes per row as in the plain product
// (lane j sums entries j, j + 8, ..., then a fixed tree), blocks striding over the rows.
__global__ __launch_bounds__(256) void cg_csr_kernel(int64_t n, CgState* __restrict__ st, int k,
                                                     const double* __restrict__ part_rr, int nb,
                                                     const int* __restrict__ row_ptr, const int* __restrict__ cols,
                                                     const double* __restrict__ vals,
                                                     const CgPair* __restrict__ rp, double* __restrict__ p,
                                                     double* __restrict__ q, double* __restrict__ part_pq) {
  constexpr int NP = 6;
  const int lane = threadIdx.x & 7;
  // the first row's entries are on their way while the partials are summed; entries count from the
  // row's first (a matrix of nearly 2^31 entries leaves no room above them in an int)
  int64_t row = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
  int a = 0, len = 0;
  double pv[NP];
  CgPair pg[NP], own{0.0, 0.0};
  auto fetch = [&]() {
    const int64_t rc = row < n ? row : n - 1;
    a = row_ptr[rc];
    len = row < n ? row_ptr[rc + 1] - a : 0;
    own = rp[rc];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int t = lane + 8 * u;
      const bool in = t < len;
      pv[u] = in ? vals[a + t] : 0.0;
      pg[u] = in ? rp[cols[a + t]] : CgPair{0.0, 0.0};
    }
  };
  fetch();
  double beta;
  if (!cg_begin(st, k, part_rr, nb, beta)) return;
  double dot = 0.0;
  for (int64_t row0 = (int64_t)blockIdx.x * 32;;) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < NP; ++u)
      if (lane + 8 * u < len) s += pv[u] * (k == 0 ? pg[u].r : pg[u].r + beta * pg[u].p);
    for (int t = lane + 8 * NP; t < len; t += 8) {
      const CgPair v = rp[cols[a + t]];
      s += vals[a + t] * (k == 0 ? v.r : v.r + beta * v.p);
    }
    s += __shfl_xor(s, 4, 8);
    s += __shfl_xor(s, 2, 8);
    s += __shfl_xor(s, 1, 8);
    if (row < n && lane == 0) {
      const double pn = k == 0 ? own.r : own.r + beta * own.p;
      p[row] = pn;
      q[row] = s;
      dot += pn * s;
    }
    row0 += (int64_t)gridDim.x * 32;
    if (row0 >= n) break;
    row = row0 + (threadIdx.x >> 3);
    fetch();
  }
  dot = block_sum256(dot);
  if (threadIdx.x == 0) part_pq[blockIdx.x] = dot;
}

// alpha = rho / p.q (every block sums the same partials in the same order);
// x += alpha p, r -= alpha q, partial sums of r.r.  PAIR: r lives in rp, which also takes p.
template <bool PAIR>
__global__ __launch_bounds__(256) void cg_xr_kernel(int64_t n, const CgState* __restrict__ st, int k,
                                                    const double* __restrict__ part_pq, int nb,
                                                    const double* __restrict__ p, const double* __restrict__ q,
                                                    double* __restrict__ x, double* __restrict__ r,
                                                    CgPair* __restrict__ rp, double* __restrict__ part_rr) {
  // the first values are on their way while the partials are summed
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t step = (int64_t)gridDim.x * blockDim.x, t0 = t < n ? t : n - 1;
  double pv = p[t0], qv = q[t0], xv = x[t0], rv = PAIR ? rp[t0].r : r[t0];
  if (st->slot[k & 1].stop) return;
  double pq = 0.0;
  for (int u = threadIdx.x; u < nb; u += blockDim.x) pq += part_pq[u];
  const double alpha = st->slot[k & 1].rho / block_sum256_all(pq);
  double s = 0.0;
  while (t < n) {
    x[t] = xv + alpha * pv;
    rv -= alpha * qv;
    if (PAIR)
      rp[t] = CgPair{rv, pv};
    else
      r[t] = rv;
    s += rv * rv;
    t += step;
    if (t >= n) break;
    pv = p[t];
    qv = q[t];
    xv = x[t];
    rv = PAIR ? rp[t].r : r[t];
  }
  s = block_sum256(s);
  if (threadIdx.x == 0) part_rr[blockIdx.x] = s;
}

// the test of the last enqueued step, k - 1, for the host (step k repeats it)
__global__ void cg_report_kernel(const double* __restrict__ part_rr, int nb, int k, CgState* st) {
  const CgSlot prev = st->slot[(k + 1) & 1];
  double rr = 0.0;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) rr += part_rr[t];
  rr = block_sum256(rr);
  if (threadIdx.x != 0) return;
  st->rr = prev.stop ? prev.rho : rr;
  st->iters = prev.stop ? prev.iters : k;
  st->stop = prev.stop || rr <= st->atol2 || !(rr == rr) ? 1 : 0;
}

namespace {
inline int64_t up256(int64_t bytes) { return (bytes + 255) / 256 * 256; }
}  // namespace

// without the interleaved copy of p: assembled operators then take separate passes
static int64_t cg_work_min(int64_t n) {
  const int64_t vec = up256(n * (int64_t)sizeof(double));
  const int64_t red = up256(kRedBlocks * (int64_t)sizeof(double));
  return 3 * vec + 2 * red + up256(sizeof(CgState)) + up256(4 * sizeof(double));
}

int64_t krylov_work_size(int64_t n, int restart) {
  const int64_t vec = up256(n * (int64_t)sizeof(double));
  const int64_t red = up256(kRedBlocks * (int64_t)sizeof(double));
  if (restart <= 0)  // CG: r, p, q, two reduction buffers, state + scalars; p interleaved with r
    return cg_work_min(n) + vec;
  // GMRES: V (restart columns), u, r, reductions, H and scalars
  return up256((int64_t)restart * n * (int64_t)sizeof(double)) + 2 * vec +
         up256((int64_t)(restart + 2) * kRedBlocks * (int64_t)sizeof(double)) +
         up256((int64_t)(restart + 2) * (restart + 1) * (int64_t)sizeof(double));
}

namespace {

// carve the caller's workspace
struct Carve {
  char* p;
  template <typename T>
  T* take(int64_t count) {
    T* out = reinterpret_cast<T*>(p);
    p += up256(count * (int64_t)sizeof(T));
    return out;
  }
};

int residual_norm(const KrylovOp& op, const double* b, const double* x, double* r, double* partial, double* out,
                  hipStream_t s) {
  ET_TRY(op.apply(1, x, b, r, s));
  return dot(op.n, r, r, partial, out, s);
}

// the structured operator (fine-grid kernels when `fine`, a copy of which the
// operator keeps) as a Krylov operator
KrylovOp structured_op(const Grid& g, const double* K0, const double* E, const uint8_t* cons, const WhtTable* fine) {
  KrylovOp op;
  op.n = g.n_nodes() * g.dim;
  const bool has = fine != nullptr;
  WhtTable tab{};
  if (has) tab = *fine;
  op.apply = [=](int mode, const double* x, const double* b, double* y, hipStream_t s) {
    return level0_op<double>(mode, g, K0, E, cons, x, b, nullptr, nullptr, 1.0, nullptr, y, s, has ? &tab : nullptr);
  };
  return op;
}

}  // namespace

int cg_solve(const Grid& g, const double* K0, const double* E, const uint8_t* cons, const WhtTable* fine, const double* b,
             double* x, double tol, int maxiter, void* work, int64_t work_bytes, int* iters, double* residual,
             hipStream_t s) {
  return cg_solve_op(structured_op(g, K0, E, cons, fine), b, x, tol, maxiter, work, work_bytes, iters, residual,
                     s);
}

int cg_solve_op(const KrylovOp& op, const double* b, double* x, double tol, int maxiter, void* work,
                int64_t work_bytes, int* iters, double* residual, hipStream_t s) {
  const int64_t n = op.n;
  ET_REQUIRE(maxiter >= 1, "cg: maxiter must be >= 1");
  ET_REQUIRE(work_bytes >= cg_work_min(n), "cg: work buffer too small");
  const bool pair = op.row_ptr != nullptr && work_bytes >= krylov_work_size(n, 0);
  Carve c{static_cast<char*>(work)};
  double* p = c.take<double>(n);
  double* q = c.take<double>(n);
  double* part_a = c.take<double>(kRedBlocks);
  double* part_b = c.take<double>(kRedBlocks);
  CgState* st = c.take<CgState>(1);
  double* scal = c.take<double>(4);  // [1] |b - A x|^2 after the loop
  double* r = c.take<double>(pair ? 2 * n : n);
  CgPair* rp = pair ? reinterpret_cast<CgPair*>(r) : nullptr;
  // one value per thread up to kRedBlocks blocks of the vector passes; each block of the next pass
  // sums one partial per block of this one
  const int nb = (int)std::min<int64_t>(kRedBlocks, (n + 255) / 256);
  const int nbr = (int)std::min<int64_t>(kRedBlocks, (n + 31) / 32);  // blocks of the row pass
  const int nb_pq = pair ? nbr : nb;
  // r = b - A x, |b|^2, |r|^2
  ET_TRY(op.apply(1, x, b, pair ? p : r, s));
  cg_start_kernel<<<nb, 256, 0, s>>>(n, b, pair ? p : r, rp, part_a, part_b);
  cg_init_kernel<<<1, 256, 0, s>>>(part_a, part_b, nb, tol, st);
  ET_CHECK_LAUNCH();
  CgState h{};
  int chunk = kCgChunk;
  for (int done = 0;;) {
    const int end = done + std::min(chunk, maxiter - done);
    for (int k = done; k < end; ++k) {
      if (pair) {
        cg_csr_kernel<<<nbr, 256, 0, s>>>(n, st, k, part_b, nb, op.row_ptr, op.cols, op.vals, rp, p, q, part_a);
        cg_xr_kernel<true><<<nb, 256, 0, s>>>(n, st, k, part_a, nb_pq, p, q, x, nullptr, rp, part_b);
      } else {
        cg_p_kernel<<<nb, 256, 0, s>>>(n, st, k, part_b, nb, r, p);
        ET_TRY(op.apply(0, p, nullptr, q, s));
        cg_pq_kernel<<<nb, 256, 0, s>>>(n, st, k, p, q, part_a);
        cg_xr_kernel<false><<<nb, 256, 0, s>>>(n, st, k, part_a, nb_pq, p, q, x, r, nullptr, part_b);
      }
    }
    done = end;
    cg_report_kernel<<<1, 256, 0, s>>>(part_b, nb, done, st);
    ET_CHECK_LAUNCH();
    ET_CHECK_HIP(hipMemcpyAsync(&h, st, sizeof(CgState), hipMemcpyDeviceToHost, s));
    ET_CHECK_HIP(hipStreamSynchronize(s));
    if (h.stop || done >= maxiter) break;
    chunk = cg_chunk(pair, done, h.rr0, h.rr, h.atol2);
  }
  if (h.bb == 0.0) {
    // |b| = 0: x = b = 0 at once, as cupyx returns
    ET_CHECK_HIP(hipMemsetAsync(x, 0, n * sizeof(double), s));
    if (iters) *iters = 0;
    if (residual) *residual = 0.0;
    return ET_OK;
  }
  // the reported residual is the true one, |b - A x| / |b| (solvers/_gpu.py:43)
  ET_TRY(residual_norm(op, b, x, q, part_b, scal + 1, s));
  double rr = 0.0;
  ET_CHECK_HIP(hipMemcpyAsync(&rr, scal + 1, sizeof(double), hipMemcpyDeviceToHost, s));
  ET_CHECK_HIP(hipStreamSynchronize(s));
  const double bb = h.bb;
  if (iters) *iters = h.iters;
  if (residual) *residual = bb > 0.0 ? std::sqrt(rr / bb) : 0.0;
  if (!(rr == rr)) {
    set_error("cg: non-finite residual");
    return ET_ENONFINITE;
  }
  if (!(h.rr <= h.atol2) && bb > 0.0) {
    set_error("cg: maxiter reached without meeting the tolerance");
    return ET_ENOCONV;
  }
  return ET_OK;
}

// ------------------------------------------------------------------ GMRES ---

// partial[k * nb + block] = sum over the block's slice of V[k] . u, k = blockIdx.y
__global__ __launch_bounds__(256) void gm_multidot_kernel(int64_t n, const double* __restrict__ V,
                                                          const double* __restrict__ u,
                                                          double* __restrict__ partial, int nb) {
  const double* v = V + (int64_t)blockIdx.y * n;
  double s = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x)
    s += v[t] * u[t];
  s = block_sum256(s);
  if (threadIdx.x == 0) partial[(int64_t)blockIdx.y * nb + blockIdx.x] = s;
}

// one block per k: out[k * stride] = sum of partial[k * nb ...]
__global__ void gm_finalize_kernel(const double* __restrict__ partial, int nb, double* __restrict__ out,
                                   int stride, int sqrt_it) {
  double s = 0.0;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) s += partial[(int64_t)blockIdx.x * nb + t];
  s = block_sum256(s);
  if (threadIdx.x == 0) out[blockIdx.x * stride] = sqrt_it ? sqrt(s) : s;
}

// u -= sum_k V[k] h[k], k < kk
__global__ __launch_bounds__(256) void gm_orth_kernel(int64_t n, const double* __restrict__ V,
                                                      const double* __restrict__ h, int kk,
                                                      double* __restrict__ u) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int k = 0; k < kk; ++k) s += V[(int64_t)k * n + t] * h[k];
    u[t] -= s;
  }
}

// v = u / *nrm (a zero norm, an exact breakdown, leaves v = 0)
__global__ __launch_bounds__(256) void gm_scale_kernel(int64_t n, const double* __restrict__ u,
                                                       const double* __restrict__ nrm, double* __restrict__ v) {
  const double d = *nrm;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x)
    v[t] = d != 0.0 ? u[t] / d : 0.0;
}

// x += sum_k V[k] y[k]
__global__ __launch_bounds__(256) void gm_update_kernel(int64_t n, const double* __restrict__ V,
                                                        const double* __restrict__ y, int m,
                                                        double* __restrict__ x) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int k = 0; k < m; ++k) s += V[(int64_t)k * n + t] * y[k];
    x[t] += s;
  }
}

// least squares min |beta e1 - H y| for the (m+1) x m upper Hessenberg H
// (column-major, leading dimension m+1) by Givens rotations
static void hessenberg_lstsq(int m, std::vector<double> H, double beta, double* y) {
  const int ld = m + 1;
  std::vector<double> g(m + 1, 0.0);
  g[0] = beta;
  for (int j = 0; j < m; ++j) {
    const double a = H[j + j * ld], b = H[j + 1 + j * ld];
    const double r = std::hypot(a, b);
    const double c = r != 0.0 ? a / r : 1.0, sn = r != 0.0 ? b / r : 0.0;
    for (int k = j; k < m; ++k) {
      const double h1 = H[j + k * ld], h2 = H[j + 1 + k * ld];
      H[j + k * ld] = c * h1 + sn * h2;
      H[j + 1 + k * ld] = -sn * h1 + c * h2;
    }
    const double g1 = g[j], g2 = g[j + 1];
    g[j] = c * g1 + sn * g2;
    g[j + 1] = -sn * g1 + c * g2;
  }
  for (int j = m - 1; j >= 0; --j) {
    double s = g[j];
    for (int k = j + 1; k < m; ++k) s -= H[j + k * ld] * y[k];
    const double d = H[j + j * ld];
    y[j] = d != 0.0 ? s / d : 0.0;
  }
}

int gmres_solve(const Grid& g, const double* K0, const double* E, const uint8_t* cons, const WhtTable* fine,
                const double* b, double* x, double tol, int restart, int maxiter, void* work, int64_t work_bytes,
                int* iters, double* residual, hipStream_t s) {
  return gmres_solve_op(structured_op(g, K0, E, cons, fine), b, x, tol, restart, maxiter, work, work_bytes, iters,
                        residual, s);
}

int gmres_solve_op(const KrylovOp& op, const double* b, double* x, double tol, int restart, int maxiter,
                   void* work, int64_t work_bytes, int* iters, double* residual, hipStream_t s) {
  const int64_t n = op.n;
  ET_REQUIRE(restart >= 1 && restart <= 256, "gmres: restart must be in [1, 256]");
  ET_REQUIRE(maxiter >= 1, "gmres: maxiter must be >= 1");
  ET_REQUIRE(work_bytes >= krylov_work_size(n, restart), "gmres: work buffer too small");
  const int m = (int)std::min<int64_t>(restart, n);
  Carve c{static_cast<char*>(work)};
  double* V = c.take<double>((int64_t)restart * n);
  double* u = c.take<double>(n);
  double* r = c.take<double>(n);
  double* partial = c.take<double>((int64_t)(restart + 2) * kRedBlocks);
  double* Hd = c.take<double>((int64_t)(restart + 2) * (restart + 1));  // H (m+1 x m), then scalars
  double* sc = Hd + (int64_t)(m + 1) * m;                            // [0] |b|, [1] |r|, [2..] y
  const int nb = kRedBlocks;
  ET_TRY(dot(n, b, b, partial, sc, s));
  double bnorm2 = 0.0;
  ET_CHECK_HIP(hipMemcpyAsync(&bnorm2, sc, sizeof(double), hipMemcpyDeviceToHost, s));
  ET_CHECK_HIP(hipStreamSynchronize(s));
  if (bnorm2 == 0.0) {
    // |b| = 0: x = b = 0 at once, as cupyx returns
    ET_CHECK_HIP(hipMemsetAsync(x, 0, n * sizeof(double), s));
    if (iters) *iters = 0;
    if (residual) *residual = 0.0;
    return ET_OK;
  }
  const double bnorm = std::sqrt(bnorm2);
  const double atol = tol * bnorm;
  std::vector<double> H((size_t)(m + 1) * m), y(m);
  int it = 0;
  double rnorm = 0.0;
  const unsigned grid = (unsigned)std::min<int64_t>(kRedBlocks, (n + 255) / 256);
  while (true) {
    ET_TRY(op.apply(1, x, b, r, s));
    gm_multidot_kernel<<<dim3(nb, 1), 256, 0, s>>>(n, r, r, partial, nb);
    gm_finalize_kernel<<<1, 256, 0, s>>>(partial, nb, sc + 1, 1, 1);
    ET_CHECK_LAUNCH();
    ET_CHECK_HIP(hipMemcpyAsync(&rnorm, sc + 1, sizeof(double), hipMemcpyDeviceToHost, s));
    ET_CHECK_HIP(hipStreamSynchronize(s));
    if (!(rnorm == rnorm)) {
      set_error("gmres: non-finite residual");
      return ET_ENONFINITE;
    }
    if (bnorm == 0.0 || rnorm <= atol || it >= maxiter) break;
    gm_scale_kernel<<<grid, 256, 0, s>>>(n, r, sc + 1, V);
    for (int j = 0; j < m; ++j) {
      ET_TRY(op.apply(0, V + (int64_t)j * n, nullptr, u, s));
      // h = V[:, :j+1]^T u into column j of H, then u -= V h
      gm_multidot_kernel<<<dim3(nb, j + 1), 256, 0, s>>>(n, V, u, partial, nb);
      gm_finalize_kernel<<<j + 1, 256, 0, s>>>(partial, nb, Hd + (int64_t)j * (m + 1), 1, 0);
      gm_orth_kernel<<<grid, 256, 0, s>>>(n, V, Hd + (int64_t)j * (m + 1), j + 1, u);
      gm_multidot_kernel<<<dim3(nb, 1), 256, 0, s>>>(n, u, u, partial, nb);
      gm_finalize_kernel<<<1, 256, 0, s>>>(partial, nb, Hd + (int64_t)j * (m + 1) + j + 1, 1, 1);
      if (j + 1 < m) gm_scale_kernel<<<grid, 256, 0, s>>>(n, u, Hd + (int64_t)j * (m + 1) + j + 1, V + (int64_t)(j + 1) * n);
      ET_CHECK_LAUNCH();
    }
    ET_CHECK_HIP(hipMemcpyAsync(H.data(), Hd, H.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    ET_CHECK_HIP(hipStreamSynchronize(s));
    hessenberg_lstsq(m, H, rnorm, y.data());
    ET_CHECK_HIP(hipMemcpyAsync(sc + 2, y.data(), m * sizeof(double), hipMemcpyHostToDevice, s));
    gm_update_kernel<<<grid, 256, 0, s>>>(n, V, sc + 2, m, x);
    ET_CHECK_LAUNCH();
    // the host copy of y must stay valid until the transfer has run
    ET_CHECK_HIP(hipStreamSynchronize(s));
    it += m;
  }
  if (iters) *iters = it;
  if (residual) *residual = bnorm > 0.0 ? rnorm / bnorm : 0.0;
  if (!(rnorm <= atol) && bnorm > 0.0) {
    set_error("gmres: maxiter reached without meeting the tolerance");
    return ET_ENOCONV;
  }
  return ET_OK;
}

}  // namespace et
