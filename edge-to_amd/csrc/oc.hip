// Optimality-criteria design update on the device, with no host round trip.
//
// The reference bisects lambda in [1e-9, 1e9] (TopOpt/_cuda.py:242-280) with a
// host synchronisation per step.  Two forms, both stream-ordered (the whole
// update can be captured in a graph), with the reference's decisions and
// stopping rule:
//
// Up to kOcSmall elements one workgroup holds the design in registers and does
// the whole bisection, a step per barrier (4 800 elements, 42 steps: 202 us in
// 55 launches, 48 us in one).  Above, one pass evaluates the volume at every
// midpoint of the next kOcDepth bisection levels at once (the 2^kOcDepth - 1
// nodes of the subtree below the current bracket, formed exactly as the
// sequential 0.5 * (l1 + l2) would form them); the next pass begins by walking
// the subtree with those volumes, every workgroup for itself (4.19 M elements,
// 42 steps: 592 us with a launch for the walk and a division per volume term,
// 334 us so; 65 536 elements 207 -> 139 us).  A fixed
// number of passes is enqueued, enough for the longest bisection the bracket
// and the 1e-4 stopping rule allow (73 steps); passes after the stop return at
// once.  The new design is evaluated once, at the last midpoint tried.
#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "blas.hpp"

namespace et {

// Bisection state at the start of the work buffer (callers may read `steps`
// there once the stream has reached the update).
struct OcState {
  double l1, l2, lmid, sabs;
  int done, steps;
};
static_assert(sizeof(OcState) == 40, "OcState layout is part of the C ABI");

constexpr int kOcDepth = 3;                       // bisection levels per pass
constexpr int kOcCand = (1 << kOcDepth) - 1;      // midpoints evaluated per pass
constexpr int kOcPasses = 26;                     // 75 >= 73 steps: every bisection ends
constexpr int64_t kOcStateBytes = 256;            // state slot (keeps ocp 256-byte aligned)

__host__ __device__ inline bool oc_continue(double l1, double l2) { return (l2 - l1) / (l2 + l1) > 1e-4; }

// midpoints of the subtree below [l1, l2] in heap order (node i: left child
// 2i+1 = [lo, m_i], right child 2i+2 = [m_i, hi])
__device__ inline void oc_midpoints(double l1, double l2, double (&m)[kOcCand]) {
  double lo[kOcCand], hi[kOcCand];
  lo[0] = l1;
  hi[0] = l2;
#pragma unroll
  for (int i = 0; i < kOcCand; ++i) {
    m[i] = 0.5 * (lo[i] + hi[i]);
    if (2 * i + 2 < kOcCand) {
      lo[2 * i + 1] = lo[i];
      hi[2 * i + 1] = m[i];
      lo[2 * i + 2] = m[i];
      hi[2 * i + 2] = hi[i];
    }
  }
}

// ocP clipped from below, as the update uses it
__device__ __forceinline__ double oc_clip(double ocp_raw, bool all_zero) {
  return all_zero ? 1e-3 : fmax(1e-12, ocp_raw);
}

// p / l from inv = 1 / l correctly rounded: one residual step gives the correctly rounded quotient
// where the first, p * inv, is within a unit of the last place (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990).  Its error is bounded by one and a half
// units only; of 1.5e9 random pairs, half of them with l just below a power of two, none exceeded
// one, and every result was the correctly rounded one.  A quotient that overflows comes out NaN,
// which the clipping below takes as the upper bound, as it does infinity.
__device__ __forceinline__ double oc_div(double p, double l, double inv) {
  const double q = p * inv;
  return fma(fma(-q, l, p), inv, q);
}

// the move limits, both within [0, 1]: clipping to [0, 1] as well changes nothing
__device__ __forceinline__ double oc_upper(double x, double move) { return fmin(fmax(x + move, 0.0), 1.0); }
__device__ __forceinline__ double oc_lower(double x, double move) { return fmin(fmax(x - move, 0.0), 1.0); }

__device__ __forceinline__ double oc_value(double xl, double xu, double p, double l, double inv) {
  return fmax(xl, fmin(xu, oc_div(p, l, inv)));
}

// x * sqrt(max(-dc/A, 0)) with NaN -> 0
__device__ __forceinline__ double oc_raw(double x, double dc, double A) {
  double q = -dc / A;
  q = q > 0.0 ? q : 0.0;
  const double v = x * sqrt(q);
  return v != v ? 0.0 : v;  // nan_to_num(nan=0)
}

// ocp = x * sqrt(max(-dc/A, 0)) with NaN -> 0 (SingleMaterial.__ocP__,
// MaterialModels.py:83-90), and per-block sums of |ocp|.  A: the element measure,
// Ae[t] per element where Ae is given (general meshes, mesh.As of shape (n, 1)).
__global__ __launch_bounds__(256) void oc_prep_kernel(int64_t n, const double* __restrict__ x,
                                                      const double* __restrict__ dc, double A,
                                                      const double* __restrict__ Ae,
                                                      double* __restrict__ ocp,
                                                      double* __restrict__ partial) {
  double s = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x) {
    const double v = oc_raw(x[t], dc[t], Ae != nullptr ? Ae[t] : A);
    ocp[t] = v;
    s += fabs(v);
  }
  s = block_sum256(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void oc_init_kernel(int nb, const double* __restrict__ partial, OcState* st) {
  double s = 0.0;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) s += partial[t];
  s = block_sum256(s);
  if (threadIdx.x == 0) {
    st->sabs = s;
    st->l1 = 1e-9;
    st->l2 = 1e9;
    st->lmid = 0.5 * (st->l1 + st->l2);
    st->done = !oc_continue(st->l1, st->l2);
    st->steps = 0;
  }
}

// v of the lane that the DPP control selects, 0 where it selects none
template <int CTRL, int ROWS>
__device__ __forceinline__ double oc_dpp(double v) {
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, int2{__builtin_amdgcn_update_dpp(0, b.x, CTRL, ROWS, 0xf, false),
                                         __builtin_amdgcn_update_dpp(0, b.y, CTRL, ROWS, 0xf, false)});
}

// Sum over the workgroup, returned to every thread, behind one barrier (s_part must not be in use).
// The wavefront's part goes through lane moves of the vector unit (shifts by 1, 2, 4, 8 within rows of
// 16, then the row totals upwards; lane 63 ends with the sum), not through LDS permutes: the sum is
// on the critical path of every bisection step.
__device__ __forceinline__ double oc_block_sum(double v, double* s_part, int nw) {
  v += oc_dpp<0x111, 0xf>(v);
  v += oc_dpp<0x112, 0xf>(v);
  v += oc_dpp<0x114, 0xf>(v);
  v += oc_dpp<0x118, 0xf>(v);
  v += oc_dpp<0x142, 0xa>(v);
  v += oc_dpp<0x143, 0xc>(v);
  if ((threadIdx.x & 63) == 63) s_part[threadIdx.x >> 6] = v;
  __syncthreads();
  double a = 0.0, b = 0.0;
  for (int w = 0; w < nw; w += 2) {
    a += s_part[w];
    b += s_part[w + 1];
  }
  return a + b;
}

constexpr int kOcThreads = 1024;      // one-workgroup form
constexpr int kOcPassThreads = 512;   // a pass keeps 7 midpoints, their inverses and sums: 1024 threads spill

// Takes up to kOcDepth of the reference's steps with the volumes of the pass that wrote `partial`
// (nb sums per midpoint, summed in a fixed order): l2 = lmid if the volume fraction is within vf,
// else l1 = lmid.  Every thread of the workgroup returns the new state.
__device__ __forceinline__ OcState oc_walk(const OcState& prev, const double* __restrict__ partial, int nb,
                                           double vol, double vf, double (*s_part)[kOcPassThreads / 64]) {
  OcState c = prev;
  double tot[kOcCand];
#pragma unroll
  for (int k = 0; k < kOcCand; ++k) {
    double s = 0.0;
    for (int t = threadIdx.x; t < nb; t += kOcPassThreads) s += partial[k * nb + t];
    tot[k] = oc_block_sum(s, s_part[k], kOcPassThreads / 64);
  }
  double m[kOcCand];
  oc_midpoints(c.l1, c.l2, m);
  int node = 0;
#pragma unroll
  for (int d = 0; d < kOcDepth; ++d) {
    double total = 0.0;
#pragma unroll
    for (int k = 0; k < kOcCand; ++k) {
      if (k == node) {
        c.lmid = m[k];
        total = tot[k];
      }
    }
    const bool feasible = total / vol <= vf;
    if (feasible)
      c.l2 = c.lmid;
    else
      c.l1 = c.lmid;
    ++c.steps;
    if (!oc_continue(c.l1, c.l2)) {
      c.done = 1;
      break;
    }
    node = feasible ? 2 * node + 1 : 2 * node + 2;
  }
  return c;
}

// Pass k: the walk with pass k - 1's volumes, then the per-block volume sums at every midpoint of the
// next subtree.  Reads state slot k & 1 and partial half (k - 1) & 1, writes the other of each.
__global__ __launch_bounds__(kOcPassThreads) void oc_pass_kernel(int64_t n, const double* __restrict__ x,
                                                             const double* __restrict__ ocp, double A,
                                                             const double* __restrict__ Ae, double move, double vol,
                                                             double vf, OcState* st, double* part, int k, int nb) {
  __shared__ double s_part[kOcCand][kOcPassThreads / 64];
  const OcState prev = st[k & 1];
  OcState c = prev;
  if (k > 0 && !prev.done) c = oc_walk(prev, part + ((k - 1) & 1) * kOcCand * nb, nb, vol, vf, s_part);
  if (blockIdx.x == 0 && threadIdx.x == 0) st[(k + 1) & 1] = c;
  if (c.done) return;
  double m[kOcCand], inv[kOcCand], s[kOcCand];
  oc_midpoints(c.l1, c.l2, m);
#pragma unroll
  for (int i = 0; i < kOcCand; ++i) {
    inv[i] = 1.0 / m[i];
    s[i] = 0.0;
  }
  const bool all_zero = c.sabs == 0.0;
  for (int64_t t = (int64_t)blockIdx.x * kOcPassThreads + threadIdx.x; t < n; t += (int64_t)gridDim.x * kOcPassThreads) {
    const double xl = oc_lower(x[t], move), xu = oc_upper(x[t], move);
    const double pv = oc_clip(ocp[t], all_zero), av = Ae != nullptr ? Ae[t] : A;
#pragma unroll
    for (int i = 0; i < kOcCand; ++i) s[i] += oc_value(xl, xu, pv, m[i], inv[i]) * av;
  }
  __syncthreads();  // the walk's sums have been read
  double* out = part + (k & 1) * kOcCand * nb;
#pragma unroll
  for (int i = 0; i < kOcCand; ++i) {
    const double v = oc_block_sum(s[i], s_part[i], kOcPassThreads / 64);
    if (threadIdx.x == 0) out[i * nb + blockIdx.x] = v;
  }
}

__global__ __launch_bounds__(256) void oc_final_kernel(int64_t n, const double* __restrict__ x,
                                                       const double* __restrict__ ocp, double move,
                                                       const OcState* __restrict__ st,
                                                       double* __restrict__ xn) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double l = st->lmid;
  xn[t] = oc_value(oc_lower(x[t], move), oc_upper(x[t], move), oc_clip(ocp[t], st->sabs == 0.0), l, 1.0 / l);
}

// The whole update by one workgroup, E elements per thread in registers.
template <int E, bool MEASURES>
__global__ __launch_bounds__(kOcThreads) void oc_small_kernel(int n, const double* __restrict__ x,
                                                              const double* __restrict__ dc, double A,
                                                              const double* __restrict__ Ae, double move, double vol,
                                                              double vf, OcState* st, double* __restrict__ xn) {
  __shared__ double s_part[2][kOcThreads / 64];
  // past the end both limits are 0, so the element counts for nothing
  double xl[E], xu[E], pv[E], av[MEASURES ? E : 1];
  double sabs = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int t = threadIdx.x + e * kOcThreads;
    const bool in = t < n;
    const int tc = in ? t : n - 1;
    const double xv = x[tc], a = MEASURES ? Ae[tc] : A;
    xl[e] = in ? oc_lower(xv, move) : 0.0;
    xu[e] = in ? oc_upper(xv, move) : 0.0;
    pv[e] = oc_raw(xv, dc[tc], a);
    if (MEASURES) av[e] = a;
    sabs += in ? fabs(pv[e]) : 0.0;
  }
  sabs = oc_block_sum(sabs, s_part[0], kOcThreads / 64);
#pragma unroll
  for (int e = 0; e < E; ++e) pv[e] = oc_clip(pv[e], sabs == 0.0);
  OcState c;
  c.l1 = 1e-9;
  c.l2 = 1e9;
  c.lmid = 0.5 * (c.l1 + c.l2);
  c.sabs = sabs;
  c.steps = 0;
  // at most 73 steps by the bracket and the stopping rule
  while (oc_continue(c.l1, c.l2) && c.steps < kOcDepth * kOcPasses) {
    c.lmid = 0.5 * (c.l1 + c.l2);
    const double inv = 1.0 / c.lmid;
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) s += oc_value(xl[e], xu[e], pv[e], c.lmid, inv) * (MEASURES ? av[e] : A);
    ++c.steps;
    const double tot = oc_block_sum(s, s_part[c.steps & 1], kOcThreads / 64);
    if (tot / vol <= vf)
      c.l2 = c.lmid;
    else
      c.l1 = c.lmid;
  }
  c.done = !oc_continue(c.l1, c.l2);
  const double inv = 1.0 / c.lmid;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int t = threadIdx.x + e * kOcThreads;
    if (t < n) xn[t] = oc_value(xl[e], xu[e], pv[e], c.lmid, inv);
  }
  if (threadIdx.x == 0) *st = c;
}

// Largest design of the one-workgroup form: 10 elements per thread in 60 of its 128 registers (12
// spill).  A bisection of 42 steps takes 63 us there against 137 us in passes.
constexpr int64_t kOcSmall = 10 * kOcThreads;
// with a measure per element a third array is held
constexpr int64_t kOcSmallMeasures = 8 * kOcThreads;
// Blocks of a pass: two per compute unit.  More would keep more loads in flight, but every block of
// the next pass reads all their sums.
constexpr int kOcBlocks = 512;
static_assert(2 * kOcBlocks * kOcCand <= kOcCand * kRedBlocks, "two halves of partial sums fit the work buffer");
static_assert(2 * sizeof(OcState) <= kOcStateBytes, "two states fit the state slot");

template <bool MEASURES>
static void oc_small(int64_t n, const double* x, const double* dc, double A, const double* Ae, double move, double vol,
                     double vf, OcState* st, double* xn, hipStream_t s) {
#define ET_OC_SMALL(E) \
  oc_small_kernel<E, MEASURES><<<1, kOcThreads, 0, s>>>((int)n, x, dc, A, Ae, move, vol, vf, st, xn)
  if (n <= kOcThreads)
    ET_OC_SMALL(1);
  else if (n <= 2 * kOcThreads)
    ET_OC_SMALL(2);
  else if (n <= 3 * kOcThreads)
    ET_OC_SMALL(3);
  else if (n <= 4 * kOcThreads)
    ET_OC_SMALL(4);
  else if (n <= 5 * kOcThreads)
    ET_OC_SMALL(5);
  else if (n <= 6 * kOcThreads)
    ET_OC_SMALL(6);
  else if (n <= 8 * kOcThreads)
    ET_OC_SMALL(8);
  else if constexpr (!MEASURES)
    ET_OC_SMALL(10);
#undef ET_OC_SMALL
}

int64_t oc_work_size(int64_t n) {
  return kOcStateBytes + n * (int64_t)sizeof(double) + kOcCand * kRedBlocks * (int64_t)sizeof(double);
}

int oc_update(int64_t n, const double* x, const double* dc, double A, double vol, double vf,
              double move, double* xn, void* work, int* steps, hipStream_t s, const double* Ae) {
  ET_REQUIRE(n > 0 && x && dc && xn && work, "oc_update: bad arguments");
  ET_REQUIRE((Ae != nullptr || A > 0) && vol > 0, "oc_update: element measure and volume must be positive");
  ET_REQUIRE(xn != x && xn != dc, "oc_update: x_new must not alias x or dc");
  ET_REQUIRE((reinterpret_cast<uintptr_t>(work) & 7) == 0, "oc_update: work must be 8-byte aligned");
  OcState* st = static_cast<OcState*>(work);
  double* ocp = reinterpret_cast<double*>(static_cast<char*>(work) + kOcStateBytes);
  double* partial = ocp + n;
  if (Ae == nullptr && n <= kOcSmall) {
    oc_small<false>(n, x, dc, A, nullptr, move, vol, vf, st, xn, s);
  } else if (Ae != nullptr && n <= kOcSmallMeasures) {
    oc_small<true>(n, x, dc, A, Ae, move, vol, vf, st, xn, s);
  } else {
    const int np = (int)std::min<int64_t>(kRedBlocks, (n + 255) / 256);
    const int nb = (int)std::min<int64_t>(kOcBlocks, (n + kOcPassThreads - 1) / kOcPassThreads);
    oc_prep_kernel<<<np, 256, 0, s>>>(n, x, dc, A, Ae, ocp, partial);
    oc_init_kernel<<<1, 256, 0, s>>>(np, partial, st);
    // a pass walks with the volumes of the one before it
    static_assert(kOcDepth * (kOcPasses - 1) >= 73 && kOcPasses % 2 == 0, "ends, with the final state in slot 0");
    for (int pass = 0; pass < kOcPasses; ++pass)
      oc_pass_kernel<<<nb, kOcPassThreads, 0, s>>>(n, x, ocp, A, Ae, move, vol, vf, st, partial, pass, nb);
    oc_final_kernel<<<grid_for(n), kBlock, 0, s>>>(n, x, ocp, move, st, xn);
  }
  ET_CHECK_LAUNCH();
  if (steps != nullptr) {
    OcState h{};
    ET_CHECK_HIP(hipMemcpyAsync(&h, st, sizeof(OcState), hipMemcpyDeviceToHost, s));
    ET_CHECK_HIP(hipStreamSynchronize(s));
    *steps = h.steps;
    if (!h.done) {
      set_error("oc_update: bisection did not terminate");
      return ET_ENOCONV;
    }
  }
  return ET_OK;
}

// ------------------------------------------------ allocation-free variant ---
//
// For callers that cannot allocate device memory (code under graph capture,
// tight serving loops): the same kernels on a work buffer in a file-scope
// device array.  Each GPU holds its own copy of the array for the life of the
// process; its device address is looked up once per device (the host-side
// name of a __device__ array is only a stand-in).  Every call on one GPU
// shares that array: calls that overlap on one GPU (different streams, or
// host threads) race.  Nothing in it needs clearing between calls: the state
// is initialised by the first kernel of every update, ocp and the partial
// sums are written before they are read.

constexpr int64_t kOcNoAllocMaxN = int64_t(1) << 20;  // elements
constexpr int64_t kOcScratchBytes =
    kOcStateBytes + kOcNoAllocMaxN * (int64_t)sizeof(double) + kOcCand * kRedBlocks * (int64_t)sizeof(double);

static __device__ __align__(256) unsigned char scratch[kOcScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int64_t oc_noalloc_max_n() { return kOcNoAllocMaxN; }

int oc_update_noalloc(int64_t n, const double* x, const double* dc, double A, double vol, double vf,
                      double move, double* xn, int* steps, hipStream_t s) {
  ET_REQUIRE(n > 0 && n <= kOcNoAllocMaxN,
             "oc_update_noalloc: n must be in [1, 1048576] (size of the static work array)");
  int dev = -1;
  ET_CHECK_HIP(hipGetDevice(&dev));
  ET_REQUIRE(dev >= 0 && dev < kMaxDevices, "oc_update_noalloc: device index out of range");
  void* work = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
      void* p = nullptr;
      ET_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      ET_REQUIRE(p != nullptr, "oc_update_noalloc: no device address for the work array");
      g_scratch_ptr[dev] = p;
    }
    work = g_scratch_ptr[dev];
  }
  return oc_update(n, x, dc, A, vol, vf, move, xn, work, steps, s, nullptr);
}

// sum (a - b)^2, used for the RMS design change of the SIMP loop
__global__ __launch_bounds__(256) void sqdist_partial_kernel(int64_t n, const double* __restrict__ a,
                                                             const double* __restrict__ b,
                                                             double* __restrict__ partial) {
  double s = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x) {
    const double d = a[t] - b[t];
    s += d * d;
  }
  s = block_sum256(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

int sqdist(int64_t n, const double* a, const double* b, double* partial, double* out,
           hipStream_t s) {
  sqdist_partial_kernel<<<kRedBlocks, 256, 0, s>>>(n, a, b, partial);
  ET_CHECK_LAUNCH();
  return reduce_finalize(partial, out, s);
}

}  // namespace et
