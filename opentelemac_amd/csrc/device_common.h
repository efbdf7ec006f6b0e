// What the kernel files share: error check, the solver state, deterministic
// reductions.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

#include "../../include/bief_hip.h"
#include "layout.h"

namespace bhip {

constexpr int kThreads = 256;
static_assert(kThreads == kPhaseSlots, "colour phases are balanced for this workgroup size");
constexpr int kWaves = kThreads / 64;

#define HIP_OK(expr)                                              \
  do {                                                            \
    hipError_t e_ = (expr);                                       \
    if (e_ != hipSuccess) {                                       \
      fprintf(stderr, "libbiefhip: %s failed: %s (%s:%d)\n", #expr, \
              hipGetErrorString(e_), __FILE__, __LINE__);         \
      return BHIP_EDEVICE;                                        \
    }                                                             \
  } while (0)

// ---------------------------------------------------------------------------
// solver state (device resident)
// ---------------------------------------------------------------------------
enum : int { ST_RUNNING = 0, ST_CONVERGED = 1, ST_FINAL = 2, ST_MAXITER = 3 };

// Iteration m of a CG solve runs U_m (vector update, parity p = m & 1) then
// E_m (direction + EBE mat-vec). Slot [p] is written by iteration m and read
// by iteration m + 1.
struct SolveState {
  double xl;        // max(||b'||^2, 1) (gracjg.F:189-209)
  double eps2xl;    // stop threshold on ||r||^2 (inner solves: relative)
  double rr0;       // ||r_0||^2 of the solve (inner solves scale eps2xl by it)
  double dot;       // result of k_reduce_into
  double rr[2];     // RMRM of iteration m, by parity
  double rho[2];    // RO of iteration m (informational)
  int m[2];         // iteration number M, by parity
  int status[2];    // ST_RUNNING or ST_FINAL (NITMAX reached), by parity
  int done;         // sticky: 0, ST_CONVERGED or ST_MAXITER
  int nitmax;
  int final_m;      // M at exit
  int use_rr0;      // threshold = eps2xl * rr0
  double final_rr;  // RMRM at exit
  int final_flag;   // set by the update kernel that applied the last X update
  int zero_rhs;     // ||b'|| < 1e-15 (gracjg.F:194-202)
  double xl_raw;    // ||b'||^2
  // mixed precision outer loop (device-side control)
  double eps2_outer;   // outer stop threshold on the FP64 ||r'||^2
  double rr_outer;     // last FP64 ||r'||^2
  double inner_eps2;   // inner relative threshold
  int inner_nitmax;    // iteration cap of one inner solve
  int nitmax_total;    // NITMAX of the whole mixed solve (inner iterations)
  int outer_done;      // the outer loop has stopped (outer_status says why)
  int outer_status;    // ST_CONVERGED or ST_MAXITER once outer_done
  int outer_count;     // inner solves started
  int inner_total;     // inner iterations of finished inner solves
  int done1;           // inner solve finished: (M << 2) | status, set by a kernel
                       // after the one that applied the last update
  int fresh;           // an outer test started an inner solve whose first
                       // kernel has not run yet (set by k_outer_check,
                       // cleared by the first update kernel of that solve)
  int xpar;            // which of the two FP64 solution buffers holds x
  int dpar;            // reliable updates: parity of the direction the next inner
                       // start continues from, -1 for a fresh start
  int reliable;        // mixed path: inner CG continued across outer steps
  int inner_pairs[8];  // CG iterations (update + direction launches) of the
                       // first inner solves, the next solve's launch plan
  int stop;            // CG kernels of this solve return at once. Set by the
                       // kernel after the one that set done, so that no
                       // workgroup of a direction kernel skips its work on a
                       // flag another workgroup of the same launch has set
  int gave_up;         // the persistent CG gave up waiting for its workgroups
  int unused;
  long long t_start;   // device clock at the set-up of the solve
  long long t_done;    // device clock when this system stopped
};

// ---------------------------------------------------------------------------
// deterministic reductions
// ---------------------------------------------------------------------------
__device__ inline double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// fixed-order block sum; result valid in thread 0
__device__ inline double block_sum(double v, double* sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += sh[i];
  }
  __syncthreads();
  return s;
}

// Fixed-order sum of n partials computed by every workgroup that calls it
// (identical result in all of them); valid in all threads.
__device__ inline double reduce_partials(const double* __restrict__ partial, int n,
                                         double* sh, double* bcast) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += partial[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) *bcast = s;
  __syncthreads();
  s = *bcast;
  __syncthreads();
  return s;
}

// reduce_partials in two steps, for kernels that want other loads in
// flight meanwhile: load_partials issues this thread's share of the partial
// sums first (indices clamped, no branches around the loads); sum_partials
// adds them in reduce_partials' order, so the result is the same to the bit.
template <int P>
__device__ inline void load_partials(double (&pv)[P], const double* __restrict__ partial,
                                     int n) {
#pragma unroll
  for (int k = 0; k < P; ++k) pv[k] = partial[min((int)threadIdx.x + k * kThreads, n - 1)];
}
template <int P>
__device__ inline double sum_partials(const double (&pv)[P], const double* __restrict__ partial,
                                      int n, double* sh, double* bcast) {
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < P; ++k)
    if ((int)threadIdx.x + k * kThreads < n) s += pv[k];
  for (int i = threadIdx.x + P * kThreads; i < n; i += blockDim.x) s += partial[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) *bcast = s;
  __syncthreads();
  s = *bcast;
  __syncthreads();
  return s;
}

// XCD-aware block order: workgroup g is dispatched to XCD g % 8; each XCD
// gets a contiguous range of node blocks so that blocks sharing halo nodes
// share an L2. Bijective for any block count.
__device__ inline int xcd_block(int g, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int xcd = g & 7, k = g >> 3;
  return xcd * q + (xcd < r ? xcd : r) + k;
}

__device__ inline int load_relaxed(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void store_relaxed(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace bhip
