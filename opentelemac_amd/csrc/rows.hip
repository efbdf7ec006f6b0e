// Persistent Krylov kernels on assembled rows (rows.h), MI355X. What follows is
// CG's; GMRES is built alike and described at its kernel.
//
// One launch runs a whole CG solve, from X and B to X in the caller's order.
// Mixed precision: FP64 residuals on FP64 rows with X in LDS, and between them
// inner solves on FP32 rows. Each workgroup (one per CU, 1024 threads) keeps the
// residual and the (inner) solution of its rows in registers, `group` rows per
// thread, and D and A D in LDS; the first coefficients of each row stay in
// registers too where they fit (RowProduct). Larger groups read the matrix again
// each iteration, out of the last-level cache (143 MB for 2M rows in FP64).
//
// Workgroups meet once per iteration: D.AD, AD.AD, R.AD and R.R together, with
// the exchange of A D of the halo rows. RO is R.R / D.AD; the next ||R||^2 is
// R.R - 2 RO R.AD + RO^2 AD.AD, which is what a second meeting would add up
// to the last digits (see kTrust); R and D of the halo follow locally. There
// are no fences: every word that crosses workgroups is written and read with
// 64-bit relaxed atomics at agent scope and carries the number of the meeting
// in its low half (a double travels as two such words), so reading the right
// number is the synchronisation. Each workgroup writes its sums to kReplicas
// places and reads all sums of its system from one of them, which spreads the
// readers over the memory channels. Measured for one sum: 1.35 us for 16
// workgroups, 1.6 for 64, 2.0 for 128, 2.8 for 256 (one place instead of 8:
// 4.0 for 256; two levels of 16: 3.5).
//
// us per iteration, FP64 / mixed: 1.4 / 1.6 (1,000 nodes, one workgroup), 3.2 /
// 3.1 (20k), 3.9 / 3.7 (100k), 4.9 / 4.5 (260k), 5.8 / 5.4 (500k), 11.2 / 7.9 (1M),
// 24.4 / 17.7 (2M). The two-kernel CG takes 15 at 20k, 50 (FP64) at 2M and 22 (FP32)
// at 1M. Beside the iterations a solve takes 75 to 130 us up to 500k nodes (PRECD1,
// the rows, this launch's start, the state back on the host) and 310 / 380 at 2M.
// What bounds it: below 500k the meeting (two trips through memory, 1.7 us for 20
// workgroups, 3.5 for 245), then the matrix. At 2M rows in FP64 the counters see
// 143 MB per iteration (the entries are 120) at 5.9 TB/s, from the last-level
// cache: a copy of as much reaches 6.9, one of 1 GiB 5.2. Each wave has one slice's
// loads in flight; more of them spill. In FP32 at 2M also registers (33 spilled:
// with one launch per inner solve 16.7, but the launches take what that gains).
//
// Sums are binary trees over the rows' leaf numbers (rows.h) and do not depend
// on how many rows a workgroup holds: a system gives the same bits alone and
// in an ensemble.
//
// Every wait ends: on the number it waits for, or after kWaitTicks of the
// device clock, when the launch gives up (abort in the sync words), leaves the
// initial solution as it was and the host solves element by element, this time
// and the next ones (BHIP_ROWS_WAIT=<ticks> changes the limit; 0 gives up at the
// first word that is not there yet, which the tests use).
// All workgroups of a system must be resident at once: threads and processes
// take turns on a GPU. A process that sees none of the others' files, or a
// mask on the CUs, can keep some from starting: the limit is for them. When a
// launch has more workgroups than fit the GPU, they take their numbers in the
// order in which they start, so the system with the lowest numbers always has
// all of its own running (RowLayout::launch).
#include "rows_dev.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <memory>
#include <new>
#include <vector>

namespace bhip {

typedef unsigned long long u64;

constexpr int kReplicas = 8;
constexpr int kSums = 4;  // sums of one meeting of CG
constexpr int kGmMaxK = 20, kGmSums = 2 * kGmMaxK + 4;  // of GMRES
// ||R||^2 of the next iteration is taken from this one's sums while it is at
// least this part of ||R||^2: its relative error is then below 4e-16 / kTrust
constexpr double kTrust = 1e-3;
constexpr int kRowWaves = kSlab / 64;
constexpr u64 kWaitTicks = 400000000ull;  // 4 s of the 100 MHz clock, unless the
                                          // environment says otherwise (rows_create)

__device__ inline u64 ld_word(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_word(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double ld_f64(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a value in numbered words: two for a double, one for a float
// (the words of a double are `stride` apart)
__device__ inline void post(u64* p, size_t stride, unsigned e, double v) {
  const u64 b = __double_as_longlong(v);
  st_word(p, (b & 0xffffffff00000000ull) | e);
  st_word(p + stride, (b << 32) | e);
}
__device__ inline void post(u64* p, size_t, unsigned e, float v) {
  st_word(p, ((u64)__float_as_uint(v) << 32) | e);
}
// one look: the value, if it is the one numbered e
__device__ inline bool look(const u64* p, size_t stride, unsigned e, double& v) {
  const u64 a = ld_word(p), b = ld_word(p + stride);
  v = __longlong_as_double((a & 0xffffffff00000000ull) | (b >> 32));
  return (unsigned)a == e && (unsigned)b == e;
}
__device__ inline bool look(const u64* p, size_t, unsigned e, float& v) {
  const u64 a = ld_word(p);
  v = __uint_as_float((unsigned)(a >> 32));
  return (unsigned)a == e;
}
// one wait's limit: from its 256th look on
struct Deadline {
  u64 ticks;
  const int* abort;
  u64 t0 = 0;
  int n = 0;
  __device__ bool past() {
    if ((++n & 255) != 0 && ticks != 0) return false;
    const u64 now = wall_clock64();
    if (!t0) t0 = now;
    return now - t0 >= ticks || load_relaxed(abort);
  }
};

// the sync words of one precision
struct SyncWords {
  u64* slots;       // [2][kReplicas][kSums][nwg][2] sums, by parity of the meeting
  u64* xch;         // [2][2][exported rows], by parity of the meeting (a float has one
                    // word only)
  unsigned* epoch;  // [2][nsys] number of the last meeting, by parity of the solve
  int* abort;       // the launch has given up
  unsigned* ticket; // workgroups started (launches larger than the GPU)
  u64* start;       // the clock before the first of several rounds or launches
  u64 ticks;        // longest wait
};

struct RowArgs {
  const int32_t* slice_off;
  const int32_t* pair_off;
  const unsigned* ids;
  const uint16_t* rowpos;
  const int32_t* wg_row0;
  const int32_t* wg_sys;
  const int32_t* sys_wg;
  const int32_t* halo_off;
  const int32_t* halo_row;
  const int32_t* halo_src;
  const int32_t* exp_off;
  const uint16_t* exp_loc;
  int nwg, nsys, nexp, nhalo;
  SyncWords sy;
  int ep;        // parity of the solve
  int first;     // first workgroup of the launch
  int ticketed;  // workgroup numbers by order of start
  int rounds;    // not all workgroups run from the start
};

// ---------------------------------------------------------------------------
// sums
// ---------------------------------------------------------------------------
// Lane exchanges by DPP within rows of 16 lanes and the permlane swaps across
// them. fold<M>(x, y): x + x of lane ^ M where bit M of the lane is 0, y + y of
// lane ^ M where it is 1; one step of sums over lanes that halves the values
// a lane carries. (fold<M>(x, x): x + x of lane ^ M.)
template <int CTRL>
__device__ inline double dpp(double v) {
  const u64 b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((u64)hi << 32) | lo);
}
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kHalfMirror = 0x141, kMirror = 0x140, kRor8 = 0x128;
__device__ inline double xor4(double v) {
  const u64 b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_ds_swizzle((int)(unsigned)b, 0x101f);
  const unsigned hi = __builtin_amdgcn_ds_swizzle((int)(unsigned)(b >> 32), 0x101f);
  return __longlong_as_double(((u64)hi << 32) | lo);
}
template <int M>
__device__ inline double fold(double x, double y) {
  if constexpr (M >= 16) {
    const u64 a = __double_as_longlong(x), b = __double_as_longlong(y);
    auto swap = [](unsigned p, unsigned q) {
      if constexpr (M == 16)
        return __builtin_amdgcn_permlane16_swap(p, q, false, false);
      else
        return __builtin_amdgcn_permlane32_swap(p, q, false, false);
    };
    const auto lo = swap((unsigned)a, (unsigned)b);
    const auto hi = swap((unsigned)(a >> 32), (unsigned)(b >> 32));
    return __longlong_as_double(((u64)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((u64)hi[1] << 32) | lo[1]);
  } else {
    const bool up = threadIdx.x & M;
    const double keep = up ? y : x, give = up ? x : y;
    if constexpr (M == 8)
      return keep + dpp<kRor8>(give);
    else if constexpr (M == 2)
      return keep + dpp<kXor2>(give);
    else
      return keep + dpp<kXor1>(give);
  }
}
// sum over 16 lanes, over 64 (in all of them)
__device__ inline double sum16(double v) {
  v += dpp<kXor1>(v);
  v += dpp<kXor2>(v);
  v += dpp<kHalfMirror>(v);
  return v + dpp<kMirror>(v);
}
__device__ inline double sum64(double v) {
  v = sum16(v);
  v = fold<16>(v, v);
  return fold<32>(v, v);
}

template <int V>
struct Sums {
  double v[V];
};

// The workgroup's V (1 or 4) sums of val(k) over threads and their rows k, as
// aligned binary trees over leaves (thread t's k-th row is leaf t * R + k).
// Sum i is valid in wave i. sh: [V * kRowWaves]. One barrier between two calls
// is enough for sh. Four sums over the lanes of a wave: the first two steps
// halve the sums a lane carries, 7 additions in all.
template <int R, int V, typename F>
__device__ inline double tree_sum(F&& val, double* sh) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  static_assert(V == 1 || V == 4, "sums");
  Sums<V> a[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    a[k] = val(k);
    // pairs, pairs of pairs, ... as soon as they are complete
#pragma unroll
    for (int h = 1; h < R && ((k + 1) & (2 * h - 1)) == 0; h *= 2) {
#pragma unroll
      for (int i = 0; i < V; ++i) a[k + 1 - 2 * h].v[i] = a[k + 1 - 2 * h].v[i] + a[k + 1 - h].v[i];
    }
    if constexpr (R >= 4)
      if (k & 1) __builtin_amdgcn_sched_barrier(0);
  }
  double s;
  int which = 0;
  if constexpr (V == 4) {
    const double p = fold<1>(a[0].v[0], a[0].v[2]), q = fold<1>(a[0].v[1], a[0].v[3]);
    s = fold<2>(p, q);
    which = (lane & 1 ? 2 : 0) + (lane & 2 ? 1 : 0);
    s += xor4(s);
  } else {
    s = a[0].v[0];
    s += dpp<kXor1>(s);
    s += dpp<kXor2>(s);
    s += dpp<kHalfMirror>(s);
  }
  s += dpp<kRor8>(s);
  s = fold<16>(s, s);
  s = fold<32>(s, s);
  if (lane < V) sh[which * kRowWaves + w] = s;
  __syncthreads();
  double t = 0.0;
  if (w < V) t = sum16(sh[w * kRowWaves + (lane & 15)]);
  return t;
}

// ---------------------------------------------------------------------------
// row products
// ---------------------------------------------------------------------------
// sum of W entries of this lane's row of a slice (v, id: the slice's
// coefficients and id words, the same in the whole wave), W / 2 more loads
// for the ids, all in flight at once
template <typename T, int W>
__device__ inline T row_dot(const T* __restrict__ v, const unsigned* __restrict__ id,
                            unsigned lane, const T* ys, T s = (T)0) {
  T c[W];
  unsigned i[(W + 1) / 2];
#pragma unroll
  for (int j = 0; j < (W + 1) / 2; ++j) i[j] = id[j * 64 + lane];
#pragma unroll
  for (int j = 0; j < W; ++j) c[j] = v[j * 64 + lane];
#pragma unroll
  for (int j = 0; j < W; ++j) s += c[j] * ys[j & 1 ? i[j / 2] >> 16 : i[j / 2] & 0xffffu];
  return s;
}
// sum over the w entries of the slice's rows from entry `from` (even) on, C
// (4 or 8) at a time
template <int C, typename T>
__device__ inline T slice_dot(const T* __restrict__ v, const unsigned* __restrict__ id,
                              unsigned lane, int from, int w, const T* ys) {
  v += from * 64;
  id += from * 32;
  w -= from;
  T s = (T)0;
#pragma nounroll
  while (w >= C) {
    s += row_dot<T, C>(v, id, lane, ys);
    v += C * 64;
    id += C * 32;
    w -= C;
  }
  if constexpr (C > 4) {
    switch (w) {
      case 7: return s + row_dot<T, 7>(v, id, lane, ys);
      case 6: return s + row_dot<T, 6>(v, id, lane, ys);
      case 5: return s + row_dot<T, 5>(v, id, lane, ys);
      case 4: return s + row_dot<T, 4>(v, id, lane, ys);
      default: break;
    }
  }
  switch (w) {
    case 3: return s + row_dot<T, 3>(v, id, lane, ys);
    case 2: return s + row_dot<T, 2>(v, id, lane, ys);
    case 1: return s + row_dot<T, 1>(v, id, lane, ys);
    default: return s;
  }
}

// The first F entries of one row, kept in registers for a whole solve.
// Slices with fewer read their last one again and multiply it by zero; empty
// ones read an id word of their own and the coefficients behind them.
template <typename T, int F>
struct RowFront {
  T c[F];
  unsigned i[F / 2];  // two ids each
};
template <typename T, int F>
__device__ inline void load_front(RowFront<T, F>& f, const T* __restrict__ v,
                                  const unsigned* __restrict__ id, unsigned lane, int w) {
  const int last = max(w - 1, 0);
#pragma unroll
  for (int j = 0; j < F / 2; ++j) f.i[j] = (id + min(j, last / 2) * 64)[lane];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const T c = (v + min(j, last) * 64)[lane];
    f.c[j] = j < w ? c : (T)0;
  }
}
template <typename T, int F>
__device__ inline T front_dot(const RowFront<T, F>& f, const T* ys) {
  T s = (T)0;
#pragma unroll
  for (int j = 0; j < F; ++j)
    s += f.c[j] * ys[j & 1 ? f.i[j / 2] >> 16 : f.i[j / 2] & 0xffffu];
  return s;
}

// as = A ds of the workgroup's rows, without the diagonal: thread t's k-th row
// at k * kSlab + t. The coefficients of small partitions stay in registers
// for the whole solve. Whatever the registers hold, a row's terms are added in
// one order, so its sum is the same to the bit in every partition: a chain of
// 8, and to it the sum of the others' chains of 4. (Up to 12 that is what
// slice_dot<8> does, with more loads in flight.)
template <typename T, int R>
struct RowProduct {
  static constexpr bool kKeep = R * sizeof(T) <= 16 || R == 4;
  // 4 rows per thread: 4 entries each. 8 would be 48 of the 128 registers in
  // FP32 and spill (1M nodes 10.8 us per iteration instead of 7.6); FP64 without
  // any takes 11.3 instead of 9.4 at 700k nodes, 14.0 instead of 11.2 at 1M
  static constexpr int kFront = R == 4 ? 4 : 8;
  RowFront<T, kFront> front[kKeep ? R : 1];
  int wid[kKeep ? R : 1];
  // the slice of this wave's k-th rows: its coefficients, id words and width
  static __device__ __forceinline__ int slice(const RowArgs& ra, const T* val, int wg, int k, const T*& v,
                                     const unsigned*& id) {
    const int q = __builtin_amdgcn_readfirstlane((wg * R + k) * kSlices + (int)(threadIdx.x >> 6));
    const int o = ra.slice_off[q];
    v = val + (size_t)o * 64;
    id = ra.ids + (size_t)ra.pair_off[q] * 64;
    return ra.slice_off[q + 1] - o;
  }
  __device__ __forceinline__ void load(const RowArgs& ra, const T* val, int wg, int k) {
    if constexpr (kKeep) {
      const T* v;
      const unsigned* id;
      wid[k] = slice(ra, val, wg, k, v, id);
      load_front(front[k], v, id, threadIdx.x & 63, wid[k]);
    }
  }
  __device__ __forceinline__ void apply(const RowArgs& ra, const T* val, int wg, const T* ds, T* as) const {
    const int t = threadIdx.x, lane = t & 63;
    if constexpr (kKeep) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        T s = front_dot(front[k], ds);
        if (wid[k] > kFront) {
          const T* v;
          const unsigned* id;
          const int w = slice(ra, val, wg, k, v, id);
          if constexpr (kFront == 4) {
            const T* v4 = v + 4 * 64;
            const unsigned* id4 = id + 2 * 64;
            switch (w) {
              case 5: s = row_dot<T, 1>(v4, id4, lane, ds, s); break;
              case 6: s = row_dot<T, 2>(v4, id4, lane, ds, s); break;
              case 7: s = row_dot<T, 3>(v4, id4, lane, ds, s); break;
              default: s = row_dot<T, 4>(v4, id4, lane, ds, s);
            }
          }
          if (kFront == 8 || w > 8) s += slice_dot<4>(v, id, lane, 8, w, ds);
        }
        as[k * kSlab + t] = s;
        // (one slab's gathers at a time)
        if constexpr (R >= 2) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma nounroll
      for (int k = 0; k < R; ++k) {
        const T* v;
        const unsigned* id;
        const int w = slice(ra, val, wg, k, v, id);
        as[k * kSlab + t] = w <= 12 ? slice_dot<8>(v, id, lane, 0, w, ds)
                                    : row_dot<T, 8>(v, id, lane, ds) +
                                          slice_dot<4>(v, id, lane, 8, w, ds);
      }
    }
  }
};

// ---------------------------------------------------------------------------
// CG
// ---------------------------------------------------------------------------
template <typename T, int R, bool DQ>
__global__ void __launch_bounds__(kSlab)
k_cg_rows(RowArgs ra, const T* __restrict__ val, const double* __restrict__ val64, RowsCg a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double sh_sum[kSums * kRowWaves];
  __shared__ double sh_in[kRowWaves];
  __shared__ int sh_bad, sh_wg;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t == 0) {
    sh_bad = 0;
    sh_wg = ra.ticketed ? (int)(atomicAdd(ra.sy.ticket, 1u) % (unsigned)ra.nwg) : ra.first + blockIdx.x;
  }
  __syncthreads();
  const int wg = __builtin_amdgcn_readfirstlane(sh_wg);
  const int sys = ra.wg_sys[wg];
  const int g0 = ra.sys_wg[sys], gang = ra.sys_wg[sys + 1] - g0;
  const bool lead = wg == g0 && t == 0;
  SolveState* st = a.st + sys;
  unsigned e = __hip_atomic_load(ra.sy.epoch + ra.ep * ra.nsys + sys, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
  constexpr bool kMixed = sizeof(T) == 4;
  const u64 t_start = ra.rounds ? ld_word(ra.sy.start) : wall_clock64();
  if (load_relaxed(ra.sy.abort)) {
    store_relaxed(&st->gave_up, 1);
    if (lead)
      __hip_atomic_store(ra.sy.epoch + (1 - ra.ep) * ra.nsys + sys, e, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const int r0 = ra.wg_row0[wg];
  const uint16_t* rowpos = ra.rowpos + (size_t)wg * R * kSlab;
  const int h0 = ra.halo_off[wg], nh = ra.halo_off[wg + 1] - h0;
  const int x0 = ra.exp_off[wg], nx = ra.exp_off[wg + 1] - x0;
  // (D first: its gathers' addresses then have a constant base)
  T* ds = reinterpret_cast<T*>(smem_raw);  // D: own rows, then halo
  T* dh = ds + R * kSlab;
  T* ah = dh + nh;                         // A D of the halo as it arrives
  T* rh = ah + nh;                         // R of the halo
  T* as = rh + nh;                         // A D of own rows
  // mixed: X, own rows, then halo
  double* xs = reinterpret_cast<double*>(smem_raw) + (2 * R * kSlab + 3 * nh + 1) / 2;

  double rr = 0.0, rr_prev = 1.0, thr = 0.0, xl_raw = 0.0;
  int m = 0, nitmax = a.nitmax;
  // mixed: inner solves started, their iterations so far, whether the last
  // one's direction can be continued
  int outer = 0, itot = 0;
  bool cont = false;

  RowProduct<T, R> prod;
  unsigned have = 0;  // bit k: this thread has a k-th row
  T rv[R], xv[R], dq[DQ ? R : 1];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    // (a few rows' addresses at a time)
    if constexpr (R >= 4) __builtin_amdgcn_sched_barrier(0);
    rv[k] = xv[k] = (T)0;
    if constexpr (DQ) dq[k] = (T)0;
    double x = 0.0;
    const int p = rowpos[k * kSlab + t];
    if (p != 0xffff) {
      const int row = r0 + p;
      have |= 1u << k;
      x = a.x0[row];
      if constexpr (!kMixed) rv[k] = a.b[row];
      if constexpr (DQ) dq[k] = (T)a.diag[row];
    }
    if constexpr (kMixed) {
      xs[k * kSlab + t] = x;
      ds[k * kSlab + t] = (T)0;
    } else {
      ds[k * kSlab + t] = xv[k] = x;
    }
    prod.load(ra, val, wg, k);
  }
  for (int h = t; h < nh; h += kSlab) {
    const int row = ra.halo_row[h0 + h];
    const double x = a.x0[row];
    if constexpr (kMixed) {
      xs[R * kSlab + h] = x;
      dh[h] = (T)0;
    } else {
      dh[h] = x;
    }
  }
  __syncthreads();

  // the thread's first exported row and first halo value
  const int my_exp = t < nx ? ra.exp_loc[x0 + t] : 0;
  const int my_src = t < nh ? ra.halo_src[h0 + t] : 0;

  // a meeting: the system's V sums of val(k) and, with `halo`, the exchange
  // of A D (into ah); false when it gave up
  auto meet = [&](auto val, auto sums, auto halo, double* sum) -> bool {
    constexpr int V = sums.value;
    ++e;
    const double s = tree_sum<R, V>(val, sh_sum);
    if (gang == 1) {
      if (lane == 0 && wave < V) sh_in[wave] = s;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < V; ++i) sum[i] = sh_in[i];
      return true;
    }
    // (opaque: the addresses below are made anew instead of kept over the loop)
    int tt = t;
    asm volatile("" : "+v"(tt));
    u64* slots = ra.sy.slots + (size_t)(e & 1) * kReplicas * kSums * ra.nwg * 2;
    u64* xch = ra.sy.xch + (size_t)(e & 1) * 2 * ra.nexp;
    if (wave < V && lane < kReplicas)
      post(slots + ((size_t)(lane * kSums + wave) * ra.nwg + wg) * 2, 1, e, s);
    if constexpr (halo.value) {
      // (A D is complete: tree_sum's barrier)
      if (tt < nx) post(xch + x0 + tt, ra.nexp, e, as[my_exp]);
      for (int i = tt + kSlab; i < nx; i += kSlab)
        post(xch + x0 + i, ra.nexp, e, as[ra.exp_loc[x0 + i]]);
    }
    // 256 threads per sum, one workgroup each; every thread looks for its sum
    // and its first halo value together
    const int sw = tt & 255, sv = tt >> 8;
    const u64* sp =
        slots + ((size_t)((wg & (kReplicas - 1)) * kSums + sv) * ra.nwg + g0 + sw) * 2;
    bool need_s = sv < V && sw < gang, need_h = halo.value && tt < nh;
    const u64* hp = xch + my_src;
    double p = 0.0;
    T hv = (T)0;
    Deadline dl = {ra.sy.ticks, ra.sy.abort};
    while (need_s || need_h) {
      if (need_s) need_s = !look(sp, 1, e, p);
      if constexpr (halo.value)
        if (need_h) need_h = !look(hp, ra.nexp, e, hv);
      if ((need_s || need_h) && dl.past()) break;
    }
    bool ok = !(need_s || need_h);
    if constexpr (halo.value) {
      if (tt < nh) ah[tt] = hv;
      for (int h = tt + kSlab; h < nh && ok; h += kSlab) {
        T v2;
        while (!look(xch + ra.halo_src[h0 + h], ra.nexp, e, v2))
          if (dl.past()) {
            ok = false;
            break;
          }
        ah[h] = v2;
      }
    }
    p = sum64(sv < V && sw < gang ? p : 0.0);
    if (lane == 0) sh_in[wave] = p;
    if (!ok) sh_bad = 1;
    __syncthreads();
    if (sh_bad) {
      if (t == 0) {
        store_relaxed(ra.sy.abort, 1);
        store_relaxed(&st->gave_up, 1);
      }
      return false;
    }
#pragma unroll
    for (int i = 0; i < V; ++i)
      sum[i] = (sh_in[4 * i] + sh_in[4 * i + 1]) + (sh_in[4 * i + 2] + sh_in[4 * i + 3]);
    return true;
  };

  auto product = [&]() {
    prod.apply(ra, val, wg, ds, as);
    if constexpr (DQ) {
#pragma unroll
      for (int k = 0; k < R; ++k) as[k * kSlab + t] += dq[k] * ds[k * kSlab + t];
    } else {
#pragma unroll
      for (int k = 0; k < R; ++k) as[k * kSlab + t] += ds[k * kSlab + t];
    }
  };
  bool zero = false;  // ||B|| is 0, so X = 0 (gracjg.F:194-202)
  bool stop;
  int status = ST_CONVERGED;
  double rr_out = 0.0;  // mixed: ||R||^2 in FP64
  if constexpr (!kMixed) {
    // R = A X - B, with ||B||^2 (gracjg.F:189-219); D = R
    product();
    auto start = [&](int k) -> Sums<kSums> {
      const double b = (double)rv[k], r = as[k * kSlab + t] - b;
      rv[k] = as[k * kSlab + t] = r;
      return {{b * b, r * r, 0.0, 0.0}};
    };
    double sum[kSums];
    if (!meet(start, std::integral_constant<int, kSums>(), std::true_type(), sum)) return;
    xl_raw = sum[0];
    rr = sum[1];
    thr = a.eps * a.eps * (xl_raw < 1.0 ? 1.0 : xl_raw);
#pragma unroll
    for (int k = 0; k < R; ++k) ds[k * kSlab + t] = rv[k];
    if (gang > 1)
      for (int h = t; h < nh; h += kSlab) rh[h] = dh[h] = ah[h];
    __syncthreads();
    zero = sqrt(xl_raw) < 1e-15;
    // stop test (gracjg.F:306-324; strict for the initial residual, :219)
    stop = zero || rr < thr;
  }
  for (;;) {
  if constexpr (kMixed) {
    // R = B - A X in FP64 with its norm, and ||B||^2; FP32 from here on
    // (through memory, so that the product can be a rolled loop)
    // (opaque: addresses made here, not kept over the inner solves)
    int tt = t;
    asm volatile("" : "+v"(tt));
    double* res = a.res + (size_t)wg * R * kSlab;
#pragma nounroll
    for (int k = 0; k < R; ++k) {
      const double* v;
      const unsigned* id;
      const int w = RowProduct<double, R>::slice(ra, val64, wg, k, v, id);
      double s = slice_dot<8>(v, id, lane, 0, w, xs);
      const int p = rowpos[k * kSlab + tt];
      double q = 0.0;
      if (p != 0xffff) {
        const double x = xs[k * kSlab + tt];
        if constexpr (DQ) s += a.diag[r0 + p] * x; else s += x;
        q = a.b[r0 + p] - s;
      }
      res[k * kSlab + tt] = q;
    }
    auto start = [&](int k) -> Sums<kSums> {
      const int p = rowpos[k * kSlab + tt];
      const double q = res[k * kSlab + tt], b = p != 0xffff ? a.b[r0 + p] : 0.0;
      as[k * kSlab + t] = rv[k] = (T)q;
      return {{b * b, q * q, 0.0, 0.0}};
    };
    double sum[kSums];
    if (!meet(start, std::integral_constant<int, kSums>(), std::true_type(), sum)) return;
    xl_raw = sum[0];
    rr_out = sum[1];
    const double eps2 = a.eps * a.eps * (xl_raw < 1.0 ? 1.0 : xl_raw);
    zero = sqrt(xl_raw) < 1e-15;
    const int left = a.nitmax - itot;
    if (zero || rr_out <= eps2 || left <= 0 || outer >= kMaxOuter) {
      status = zero || rr_out <= eps2 ? ST_CONVERGED : ST_MAXITER;
      break;
    }
    ++outer;
    // the inner solve: D = R, or continued R + BETA D
    rr = rr_out;
    thr = a.inner_eps * a.inner_eps * rr;
    nitmax = min(a.inner_nitmax, left) + (cont ? 1 : 0);
    m = cont ? 1 : 0;
    const T beta = (T)(cont ? rr / rr_prev : 0.0);
    if (!cont) rr_prev = 1.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      xv[k] = (T)0;
      ds[k * kSlab + t] = cont ? rv[k] + beta * ds[k * kSlab + t] : rv[k];
    }
    if (gang > 1)
      for (int h = tt; h < nh; h += kSlab) {
        rh[h] = ah[h];
        dh[h] = cont ? ah[h] + beta * dh[h] : ah[h];
      }
    __syncthreads();
    status = ST_CONVERGED;
    stop = m == 0 ? rr < thr : rr <= thr;
  }
  while (!stop) {
    product();  // AD
    // D.AD, AD.AD, R.AD, R.R
    auto dots = [&](int k) -> Sums<kSums> {
      if (!(have >> k & 1)) return {};
      const double d = (double)ds[k * kSlab + t], s = (double)as[k * kSlab + t];
      const double r = (double)rv[k];
      return {{d * s, s * s, r * s, r * r}};
    };
    double sum[kSums];
    if (!meet(dots, std::integral_constant<int, kSums>(), std::true_type(), sum)) return;
    rr = sum[3];
    // RO, X -= RO D (gracjg.F:380-388); after iteration NITMAX no more
    const double rho = rr / sum[0];
    const T rhot = (T)rho;
#pragma unroll
    for (int k = 0; k < R; ++k) xv[k] -= rhot * ds[k * kSlab + t];
    if (m >= nitmax) {
      status = ST_MAXITER;
      break;
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (have >> k & 1) rv[k] -= rhot * as[k * kSlab + t];
    // ||R||^2 after this update, from the sums before it (no second meeting).
    // It loses digits where it falls far in one step, and the stop test wants
    // the sum itself: both are summed anew
    rr_prev = rr;
    rr = rr - 2.0 * rho * sum[2] + rho * rho * sum[1];
    if (!(rr > kTrust * rr_prev && rr > 1.001 * thr)) {
      auto own = [&](int k) -> Sums<1> {
        return {{(have >> k & 1) ? (double)rv[k] * (double)rv[k] : 0.0}};
      };
      if (!meet(own, std::integral_constant<int, 1>(), std::false_type(), &rr)) return;
    }
    ++m;
    stop = rr <= thr;
    if (stop) break;
    // D = R + BETA D, halo included
    const T beta = (T)(rr / rr_prev);
#pragma unroll
    for (int k = 0; k < R; ++k) ds[k * kSlab + t] = rv[k] + beta * ds[k * kSlab + t];
    if (gang > 1) {
      int h = t;
      asm volatile("" : "+v"(h));
      for (; h < nh; h += kSlab) {
        const T r = rh[h] - rhot * ah[h];
        rh[h] = r;
        dh[h] = r + beta * dh[h];
      }
    }
    __syncthreads();
  }
  if constexpr (!kMixed) break;
  const int used = m - (cont ? 1 : 0);
  itot += used;
  cont = a.reliable && used >= 1 && status == ST_CONVERGED;
  int tx = t;
  asm volatile("" : "+v"(tx));
  // X -= what the inner solve has found, halo included. (One sum, although
  // nobody wants it: no workgroup may be two meetings ahead of another.)
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if constexpr (kMixed) xs[k * kSlab + tx] -= (double)xv[k];
    as[k * kSlab + tx] = xv[k];
  }
  auto none = [&](int) -> Sums<1> { return {{0.0}}; };
  double sum0;
  if (!meet(none, std::integral_constant<int, 1>(), std::true_type(), &sum0)) return;
  if (gang > 1)
    for (int h = tx; h < nh; h += kSlab) xs[R * kSlab + h] -= (double)ah[h];
  __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (have >> k & 1) {
      const int row = r0 + rowpos[k * kSlab + t];
      double x = (double)xv[k];
      if constexpr (kMixed) x = xs[k * kSlab + t];
      if (a.scale) x *= a.scale[row];
      a.x[a.idx ? a.idx[row] : row] = zero ? 0.0 : x;
    }
  if (lead) {
    st->xl_raw = xl_raw;
    st->xl = xl_raw < 1.0 ? 1.0 : xl_raw;
    st->zero_rhs = zero;
    st->t_start = t_start;
    if constexpr (kMixed) {
      st->rr_outer = zero ? 0.0 : rr_out;
      st->outer_count = outer;
      st->inner_total = itot;
      st->outer_status = status;
      st->outer_done = 1;
    } else {
      st->final_m = zero ? 0 : m;
      st->final_rr = zero ? 0.0 : rr;
    }
    st->t_done = zero ? t_start : wall_clock64();
    st->done = status;
    __hip_atomic_store(ra.sy.epoch + (1 - ra.ep) * ra.nsys + sys, e, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------------------
// GMRES(K), a whole solve; mixed: FP32 cycles, each from the FP64 residual
// ---------------------------------------------------------------------------
// One meeting per Arnoldi step: w = A V_j with w.V_i and V_j.V_i (i <= j), w.w
// and the exchange of w of the halo rows. From these every workgroup has the
// coefficients of modified Gram-Schmidt, h_i = w.V_i - sum over l < i of h_l
// V_l.V_i (the dot of V_i with what the earlier steps leave of w), and ||w -
// sum h_i V_i||^2, summed anew where it falls below kTrust w.w. The halo's V
// follow from the exchanged w. The basis lies in memory, each thread's rows
// together, and mostly in L2; V_j and w are in LDS, R0 in registers.
//
// us per solve at K = 5, FP64 / mixed (in brackets: from the host, one kernel per
// orthogonalisation step, 11 launches for a cycle of K = 3, 9 of them with a sum
// over all workgroups): 90k nodes 522 / 531 (2310 / 2661), 500k 854 / 838 (2896 /
// 3120), 2M 3238 / 2088 (5275 / 4711); 11 cycles each. A step takes 7 us at 90k,
// most of it the meeting, 55 at 2M, where the basis (170 MB in FP64) and the
// matrix come from the last-level cache.
struct GmLds {
  double part[kGmSums * kRowWaves];
  double tot[kGmSums * 4];
  double h[kGmMaxK + 1][kGmMaxK];
  double g[kGmMaxK][kGmMaxK];  // V_i.V_l
  double coef[kGmMaxK + 1];
  double cs[kGmMaxK], sn[kGmMaxK], y[kGmMaxK + 1];
  int bad, exit_now;
};

// v: 8 sums over the 64 lanes; the lane's sum is that of v[sum8_index()]
__device__ inline int sum8_index() {
  const int l = threadIdx.x;
  return (l & 32 ? 4 : 0) + (l & 16 ? 2 : 0) + (l & 8 ? 1 : 0);
}
__device__ inline double sum8(const double (&v)[8]) {
  const double a0 = fold<32>(v[0], v[4]), a1 = fold<32>(v[1], v[5]);
  const double a2 = fold<32>(v[2], v[6]), a3 = fold<32>(v[3], v[7]);
  double s = fold<8>(fold<16>(a0, a2), fold<16>(a1, a3));
  s += dpp<kXor1>(s);
  s += dpp<kXor2>(s);
  return s + dpp<kHalfMirror>(s);
}
__device__ inline double lane_value(double v, int lane) {
  const u64 b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double(((u64)hi << 32) | lo);
}

template <typename T, int R>
__global__ void __launch_bounds__(kSlab)
k_gmres_rows(RowArgs ra, const T* __restrict__ val, const double* __restrict__ val64,
             RowsGmres a, T* basis, T* hbasis) {
  constexpr bool kMixed = sizeof(T) == 4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ GmLds sh;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wg = blockIdx.x, gang = ra.nwg;
  const bool lead = wg == 0 && t == 0;
  unsigned e = __hip_atomic_load(ra.sy.epoch + ra.ep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (load_relaxed(ra.sy.abort)) {
    store_relaxed(&a.st->gave_up, 1);
    return;
  }
  const int r0 = ra.wg_row0[wg];
  const uint16_t* rowpos = ra.rowpos + (size_t)wg * R * kSlab;
  const int h0 = ra.halo_off[wg], nh = ra.halo_off[wg + 1] - h0;
  const int x0 = ra.exp_off[wg], nx = ra.exp_off[wg + 1] - x0;
  T* ds = reinterpret_cast<T*>(smem_raw);  // V_j: own rows, then halo
  T* dh = ds + R * kSlab;
  T* ah = dh + nh;                         // A V_j of the halo
  T* as = ah + nh;                         // A V_j of own rows
  // mixed: X, own rows, then halo
  double* xs = reinterpret_cast<double*>(smem_raw) + (2 * R * kSlab + 2 * nh + 1) / 2;
  // this thread's part of the scratch: V, A V (FP64) and the diagonal
  const size_t vstride = (size_t)ra.nwg * R * kSlab, hstride = ra.nhalo;
  T* vb = basis + (size_t)wg * R * kSlab + t;
  T* avb = vb + (size_t)a.krylov * vstride;
  T* dq = vb + (size_t)(kMixed ? 1 : 2) * a.krylov * vstride;
  T* vh = hbasis + h0;
  if (t == 0) sh.bad = 0;
  __syncthreads();

  auto total = [&](int s) {
    return (sh.tot[4 * s] + sh.tot[4 * s + 1]) + (sh.tot[4 * s + 2] + sh.tot[4 * s + 3]);
  };
  // a meeting: n sums from the waves' sh.part[sum][wave], and with `halo` the
  // exchange of `as` (into ah); false when it gave up
  auto meet = [&](int n, bool halo) -> bool {
    ++e;
    __syncthreads();
    u64* slots = ra.sy.slots + (size_t)(e & 1) * kReplicas * kGmSums * ra.nwg * 2;
    u64* xch = ra.sy.xch + (size_t)(e & 1) * 2 * ra.nexp;
    for (int s = wave; s < n; s += kRowWaves) {
      const double v = sum16(sh.part[s * kRowWaves + (lane & 15)]);
      if (gang == 1) {
        if (lane < 4) sh.tot[4 * s + lane] = lane ? 0.0 : v;
      } else if (lane < kReplicas) {
        post(slots + ((size_t)(lane * kGmSums + s) * ra.nwg + wg) * 2, 1, e, v);
      }
    }
    if (gang == 1) {
      __syncthreads();
      return true;
    }
    if (halo)
      for (int i = t; i < nx; i += kSlab) post(xch + x0 + i, ra.nexp, e, as[ra.exp_loc[x0 + i]]);
    // 256 threads per sum, one workgroup each, up to 16 sums at a time
    const int sw = t & 255, sv = t >> 8;
    bool ok = true;
    for (int s0 = 0; s0 < n; s0 += 16) {
      const u64* sp =
          slots + ((size_t)((wg & (kReplicas - 1)) * kGmSums + s0 + sv) * ra.nwg + sw) * 2;
      unsigned need = 0;
      double p[4] = {};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + sv + 4 * i < n && sw < gang) need |= 1u << i;
      Deadline dl = {ra.sy.ticks, ra.sy.abort};
      while (need) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (need >> i & 1)
            if (look(sp + (size_t)8 * i * ra.nwg, 1, e, p[i])) need &= ~(1u << i);
        if (need && dl.past()) break;
      }
      ok = ok && !need;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + 4 * i < n) {
          const double q = sum64(p[i]);
          // (sum s0 + sv + 4 i; its waves are 4 sv .. 4 sv + 3)
          if (lane == 0 && s0 + sv + 4 * i < n) sh.tot[(s0 + sv + 4 * i) * 4 + (wave & 3)] = q;
        }
    }
    if (halo)
      for (int h = t; h < nh && ok; h += kSlab) {
        T v = (T)0;
        Deadline dl = {ra.sy.ticks, ra.sy.abort};
        while (!look(xch + ra.halo_src[h0 + h], ra.nexp, e, v))
          if (dl.past()) {
            ok = false;
            break;
          }
        ah[h] = v;
      }
    if (!ok) sh.bad = 1;
    __syncthreads();
    if (sh.bad) {
      if (t == 0) {
        store_relaxed(ra.sy.abort, 1);
        store_relaxed(&a.st->gave_up, 1);
      }
      return false;
    }
    return true;
  };
  // one sum of val(k) over rows, as sum `s` of the next meeting
  auto sum_rows = [&](int s, auto val1) {
    double p = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) p += val1(k);
    p = sum64(p);
    if (lane == 0) sh.part[s * kRowWaves + wave] = p;
  };

  RowProduct<T, R> prod;
  auto product = [&]() {
    prod.apply(ra, val, wg, ds, as);
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const T d = ds[k * kSlab + t];
      as[k * kSlab + t] += a.diag ? dq[(size_t)k * kSlab] * d : d;
    }
  };
  T rv[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if constexpr (R >= 4) __builtin_amdgcn_sched_barrier(0);
    const int p = rowpos[k * kSlab + t];
    double x = 0.0;
    T d = (T)0;
    rv[k] = (T)0;
    if (p != 0xffff) {
      x = a.x0[r0 + p];
      if constexpr (!kMixed) rv[k] = a.b[r0 + p];
      if (a.diag) d = (T)a.diag[r0 + p];
    }
    if constexpr (kMixed)
      xs[k * kSlab + t] = x;
    else
      ds[k * kSlab + t] = x;
    if (a.diag) dq[(size_t)k * kSlab] = d;
    prod.load(ra, val, wg, k);
  }
  for (int h = t; h < nh; h += kSlab) {
    const double x = a.x0[ra.halo_row[h0 + h]];
    if constexpr (kMixed)
      xs[R * kSlab + h] = x;
    else
      dh[h] = x;
  }
  __syncthreads();
  // R0 = A X - B with its norm, and ||B||^2 (gmres.f:188-207), as the sums 0 and
  // 1 of a meeting that brings the halo of R0; mixed: in FP64, times `sc` in FP32
  double sc = 1.0;
  auto residual = [&]() -> bool {
    if constexpr (kMixed) {
      int tt = t;
      asm volatile("" : "+v"(tt));
      double bb = 0.0, rr = 0.0;
#pragma nounroll
      for (int k = 0; k < R; ++k) {
        const double* v;
        const unsigned* id;
        const int w = RowProduct<double, R>::slice(ra, val64, wg, k, v, id);
        double s = slice_dot<8>(v, id, lane, 0, w, xs);
        const int p = rowpos[k * kSlab + tt];
        double q = 0.0, b = 0.0;
        if (p != 0xffff) {
          const double x = xs[k * kSlab + tt];
          b = a.b[r0 + p];
          s += a.diag ? a.diag[r0 + p] * x : x;
          q = s - b;
        }
        bb += b * b;
        rr += q * q;
        as[k * kSlab + tt] = (T)(q * sc);
      }
      bb = sum64(bb);
      rr = sum64(rr);
      if (lane == 0) {
        sh.part[wave] = bb;
        sh.part[kRowWaves + wave] = rr;
      }
    } else {
      product();
      sum_rows(0, [&](int k) { return (double)rv[k] * (double)rv[k]; });
#pragma unroll
      for (int k = 0; k < R; ++k) {
        rv[k] = as[k * kSlab + t] - rv[k];
        as[k * kSlab + t] = rv[k];
      }
      sum_rows(1, [&](int k) { return (double)rv[k] * (double)rv[k]; });
    }
    return meet(2, true);
  };
  if (!residual()) return;
  double nb = sqrt(total(0)), nr0 = sqrt(total(1));
  int m = 0;
  const int relat = nb < 1.0 ? 0 : 1;
  if (nb < 1.0) nb = 1.0;
  double prec = nr0 / nb;
  int products = 0;
  bool updated = false;
  bool stop = prec <= a.eps;  // (gmres.f:207)
  while (!stop) {
    ++m;
    if constexpr (kMixed)
      if (!(nr0 > 1e-25 && nr0 < 1e25) && nr0 > 0.0 && nr0 < 1e300) {
        // R0 again, scaled into FP32's range
        sc = 1.0 / nr0;
        if (!residual()) return;
      }
    // V_0 = -R0 / ||R0|| (gmres.f:243), halo included
    const double r1 = -1.0 / (nr0 * sc);
    sc = 1.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const T r = kMixed ? as[k * kSlab + t] : rv[k];
      ds[k * kSlab + t] = vb[(size_t)k * kSlab] = (T)(r1 * (double)r);
    }
    for (int h = t; h < nh; h += kSlab) dh[h] = vh[h] = (T)(r1 * (double)ah[h]);
    __syncthreads();
    int kk = a.krylov;
    for (int j = 0; j < kk; ++j) {
      product();
      if constexpr (!kMixed) {
#pragma unroll
        for (int k = 0; k < R; ++k)
          avb[j * vstride + (size_t)k * kSlab] = as[k * kSlab + t];
      }
      // sums 2 q and 2 q + 1: w.V_q and V_j.V_q; w.w follows
      for (int q0 = 0; q0 < j + 2; q0 += 4) {
        double v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int q = q0 + i;
          double pw = 0.0, pd = 0.0;
          if (q < j) {
            T b[R];
#pragma unroll
            for (int k = 0; k < R; ++k) b[k] = vb[q * vstride + (size_t)k * kSlab];
#pragma unroll
            for (int k = 0; k < R; ++k) {
              pw += (double)as[k * kSlab + t] * (double)b[k];
              pd += (double)ds[k * kSlab + t] * (double)b[k];
            }
          } else if (q == j) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
              const double d = (double)ds[k * kSlab + t];
              pw += (double)as[k * kSlab + t] * d;
              pd += d * d;
            }
          } else if (q == j + 1) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
              const double w = (double)as[k * kSlab + t];
              pw += w * w;
            }
          }
          v[2 * i] = pw;
          v[2 * i + 1] = pd;
        }
        const double s = sum8(v);
        const int i = 2 * q0 + sum8_index();
        if ((lane & 7) == 0 && i < 2 * j + 3) sh.part[i * kRowWaves + wave] = s;
      }
      const bool last = j == a.krylov - 1;
      if (!meet(2 * j + 3, !last)) return;
      // every wave for itself: lane q <= j has w.V_q and row q of V.V
      const double c = lane <= j ? total(2 * lane) : 0.0;
      const double ww = total(2 * j + 2);
      double hq = c;
      if (lane <= j) sh.g[j][lane] = sh.g[lane][j] = total(2 * lane + 1);
      const double* grow = sh.g[min(lane, j)];
      // K-th column (gmres.f:285-296): H(I,K) = w.V_I, H(K+1,K) by Pythagoras
      bool reduced = last;
      if (!last) {
        for (int l = 0; l < j; ++l) {
          const double hl = lane_value(hq, l);
          if (lane > l && lane <= j) hq -= hl * grow[l];
        }
        double gh = 0.0;
        for (int l = 0; l <= j; ++l) gh += lane_value(hq, l) * grow[l];
        double n2 = ww + sum64(lane <= j ? hq * (gh - 2.0 * c) : 0.0);
        if (lane <= j) sh.coef[lane] = hq;
        T w[R];
#pragma unroll
        for (int k = 0; k < R; ++k) w[k] = as[k * kSlab + t] - (T)sh.coef[j] * ds[k * kSlab + t];
        for (int q = 0; q < j; ++q) {
          const T hc = (T)sh.coef[q];
#pragma unroll
          for (int k = 0; k < R; ++k) w[k] -= hc * vb[q * vstride + (size_t)k * kSlab];
        }
        if (!(n2 > kTrust * ww)) {
          sum_rows(0, [&](int k) { return (double)w[k] * (double)w[k]; });
          if (!meet(1, false)) return;
          n2 = total(0);
        }
        const double r = sqrt(n2);
        if (r < 1e-20) {
          // reduction of the Krylov space (gmres.f:274-283)
          reduced = true;
          kk = j + 1;
          ++products;
        } else {
          if (wave == 0 && lane <= j) sh.h[lane][j] = hq;
          if (t == 0) sh.h[j + 1][j] = r;
          const double s = 1.0 / r;
#pragma unroll
          for (int k = 0; k < R; ++k) {
            const T v = (T)(s * (double)w[k]);
            ds[k * kSlab + t] = vb[(j + 1) * vstride + (size_t)k * kSlab] = v;
          }
          for (int h = t; h < nh; h += kSlab) {
            T v = ah[h] - (T)sh.coef[j] * dh[h];
            for (int q = 0; q < j; ++q) v -= (T)sh.coef[q] * vh[q * hstride + h];
            dh[h] = vh[(j + 1) * hstride + h] = (T)(s * (double)v);
          }
          __syncthreads();
        }
      }
      if (reduced) {
        if (wave == 0 && lane <= j) sh.h[lane][j] = c;
        if (t == 0) {
          double hk = ww;
          for (int q = 0; q <= j; ++q) hk -= sh.h[q][j] * sh.h[q][j];
          sh.h[j + 1][j] = sqrt(max(hk, 0.0));
        }
      }
    }
    // (steps past a reduction count: the host-driven solver runs them too)
    products += a.krylov;
    // Givens rotations and H y = e (gmres.f:304-350)
    if (t == 0) {
      auto& h = sh.h;
      double* y = sh.y;
      y[0] = nr0;
      int ex = 0;
      for (int i = 0; i < kk; ++i) {
        for (int j = 0; j < i; ++j) {
          const double zz = sh.cs[j] * h[j][i] + sh.sn[j] * h[j + 1][i];
          h[j + 1][i] = -sh.sn[j] * h[j][i] + sh.cs[j] * h[j + 1][i];
          h[j][i] = zz;
        }
        const double rr = sqrt(h[i][i] * h[i][i] + h[i + 1][i] * h[i + 1][i]);
        if (fabs(rr) < 1e-6) {
          ex = 1;
          break;
        }
        sh.cs[i] = h[i][i] / rr;
        sh.sn[i] = h[i + 1][i] / rr;
        h[i][i] = rr;
        y[i + 1] = -sh.sn[i] * y[i];
        y[i] = sh.cs[i] * y[i];
      }
      if (!ex)
        for (int j = kk - 1; j >= 0; --j) {
          double v = y[j];
          for (int l = j + 1; l < kk; ++l) v -= h[j][l] * y[l];
          y[j] = v / h[j][j];
        }
      sh.exit_now = ex;
    }
    __syncthreads();
    if (sh.exit_now) {
      stop = true;
      break;
    }
    // X += sum y_l V_l, R0 += sum y_l A V_l (gmres.f:354-359); mixed: X in FP64,
    // halo included, and R0 anew
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int p = rowpos[k * kSlab + t];
      double xv = 0.0;
      if constexpr (kMixed)
        xv = xs[k * kSlab + t];
      else if (p != 0xffff)
        xv = updated ? a.x[r0 + p] : a.x0[r0 + p];
#pragma unroll 2
      for (int l = 0; l < kk; ++l) {
        const double yl = sh.y[l];
        xv += yl * (double)vb[l * vstride + (size_t)k * kSlab];
        if constexpr (!kMixed) rv[k] += yl * avb[l * vstride + (size_t)k * kSlab];
      }
      if constexpr (kMixed)
        xs[k * kSlab + t] = xv;
      else if (p != 0xffff)
        a.x[r0 + p] = xv;
    }
    updated = true;
    if constexpr (kMixed) {
      for (int h = t; h < nh; h += kSlab) {
        double xv = xs[R * kSlab + h];
#pragma unroll 2
        for (int l = 0; l < kk; ++l) xv += sh.y[l] * (double)vh[l * hstride + h];
        xs[R * kSlab + h] = xv;
      }
      __syncthreads();
      if (!residual()) return;
      nr0 = sqrt(total(1));
      prec = nr0 / nb;
      stop = !(prec >= a.eps && m < a.nitmax);
      continue;
    }
    nr0 = fabs(sh.y[kk]);
    prec = nr0 / nb;
    stop = !(prec >= a.eps && m < a.nitmax);
    if (!stop) {
      // R0 of the halo, and ||R0|| itself: |E(K+1)| is it up to rounding that
      // grows by ||R0||^2 / |E(K+1)|^2 each cycle if V_0 is divided by it
#pragma unroll
      for (int k = 0; k < R; ++k) as[k * kSlab + t] = rv[k];
      sum_rows(0, [&](int k) { return (double)rv[k] * (double)rv[k]; });
      if (!meet(1, true)) return;
      nr0 = sqrt(total(0));
      prec = nr0 / nb;
      stop = !(prec >= a.eps);
    }
  }
  if constexpr (kMixed)
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int p = rowpos[k * kSlab + t];
      if (p != 0xffff && updated) a.x[r0 + p] = xs[k * kSlab + t];
    }
  if (lead) {
    a.st->prec = prec;
    a.st->relat = relat;
    a.st->m = m;
    a.st->products = products;
    a.st->updated = updated;
    __hip_atomic_store(ra.sy.epoch + 1 - ra.ep, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------------------
// D A D and assembly of one node block: its coefficients are scaled, written
// back and kept in LDS, where the block's 16 slices sum them. A gather from
// memory instead takes a cache line per coefficient (k_rows_assemble: 138 us
// for 2M nodes in FP64, after 49 us for the scaling alone). Bound by memory:
// 105 us for 2M nodes in FP64 (450 MB, 4.3 TB/s), 48 us for 1M in FP32. More
// blocks than CUs: 512 threads, so that one block gathers while another loads;
// else 1024 (20k nodes 11.2 -> 8.5 us, 100k 14.7 -> 11.3).
// ---------------------------------------------------------------------------
constexpr int kDmdThreads = 1024;
template <int NDP, bool Q, typename T>
__global__ void __launch_bounds__(kDmdThreads)
k_dmd_rows(RowsDmd a, T* __restrict__ val, double* __restrict__ val64, const int32_t* __restrict__ slice_off,
           const int32_t* __restrict__ ref_off, const uint8_t* __restrict__ ref_end,
           const uint16_t* __restrict__ refs, const int32_t* __restrict__ slab_slice, int group) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int npair = NDP * (NDP - 1) / 2, nc = Q ? 2 * npair : npair;
  const int b = xcd_block(blockIdx.x, a.nblocks);
  const int t = threadIdx.x, wave = t >> 6;
  const unsigned lane = t & 63;
  const int s0 = a.color_off[(size_t)b * (kMaxColors + 1)];
  const int ns = a.color_off[(size_t)b * (kMaxColors + 1) + kMaxColors] - s0;
  const size_t np = a.nslot_pad;
  double* cs = reinterpret_cast<double*>(smem_raw);  // [nc][ns]
  double* ds = cs + (size_t)nc * ns;
  if (a.d) {
    const int n0 = a.node_start[b], nown = a.node_start[b + 1] - n0;
    const int h0 = a.halo_start[b], nloc = nown + a.halo_start[b + 1] - h0;
    for (int l = t; l < nloc; l += (int)blockDim.x)
      ds[l] = a.d[l < nown ? n0 + l : a.halo[h0 + l - nown]];
    __syncthreads();
  }
  for (int i = t; i < ns; i += (int)blockDim.x) {
    const int s = s0 + i;
    double c[nc], dv[NDP];
#pragma unroll
    for (int q = 0; q < nc; ++q) c[q] = a.src[q * np + s];
    if (a.d) {
#pragma unroll
      for (int k = 0; k < NDP; ++k) dv[k] = ds[a.lid[k * np + s]];
      int q = 0;
#pragma unroll
      for (int p = 0; p < NDP; ++p)
#pragma unroll
        for (int j = p + 1; j < NDP; ++j, ++q) {
          // elements: XM * D(j) * D(i) (om1111.f:583-600); segments (NDP 2):
          // XM * D(GLOSEG1) * D(GLOSEG2) (omseg.f:524-536)
#pragma unroll
          for (int h = 0; h < nc / npair; ++h) {
            double& v = c[h * npair + q];
            v = NDP == 2 ? v * dv[p] * dv[j] : v * dv[j] * dv[p];
            a.xa[(h * npair + q) * np + s] = v;
          }
        }
    }
#pragma unroll
    for (int q = 0; q < nc; ++q) cs[q * ns + i] = c[q];
  }
  __syncthreads();
  // the block's slices: for each of its 16 / group waves, one per row of a thread
  const int q0 = slab_slice[b];
  constexpr int U = kRefChunk;
  for (int i = wave; i < kSlices; i += (int)(blockDim.x >> 6)) {
    const int q = __builtin_amdgcn_readfirstlane(q0 + i % group * kSlices + i / group);
    const int c1 = ref_off[q + 1];
    T* out = val + (size_t)slice_off[q] * 64;
    double* out64 = val64 + (size_t)slice_off[q] * 64;
    double s = 0.0;
    for (int c = ref_off[q]; c < c1; c += U) {
      const uint16_t* p = refs + (size_t)c * 64;
      int f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] = p[u * 64 + lane];
      const int ends = ref_end[c / U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = (f[u] & 0x7fff) + (Q && (f[u] & 0x8000) ? npair * ns : 0);
        s += f[u] == 0xffff ? 0.0 : cs[k];
        if (ends >> u & 1) {
          out[lane] = (T)s;
          out += 64;
          if constexpr (sizeof(T) == 4) {
            if (val64) out64[lane] = s;
            out64 += 64;
          }
          s = 0.0;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// assembly from memory: one wave per slice, two chunks of references in
// flight. Bound by the cache line each gathered coefficient takes (600k-node
// prisms: 34M references, 146 us).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
k_rows_assemble(T* __restrict__ val, double* __restrict__ val64, const double* __restrict__ xa,
                const int32_t* __restrict__ slice_off, const int32_t* __restrict__ ref_off,
                const uint8_t* __restrict__ ref_end, const int32_t* __restrict__ refs, int nslice,
                unsigned lower) {
  // each XCD takes a contiguous range of slices: a block's coefficients are
  // read by the slices of its rows
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int q = __builtin_amdgcn_readfirstlane(b * 4 + (int)(threadIdx.x >> 6));
  const unsigned lane = threadIdx.x & 63;
  if (q >= nslice) return;
  const int c0 = ref_off[q], c1 = ref_off[q + 1];
  T* out = val + (size_t)slice_off[q] * 64;
  double* out64 = val64 + (size_t)slice_off[q] * 64;
  double s = 0.0;
  constexpr int U = kRefChunk;
  auto load = [&](int c, int (&r)[U]) {
    const int32_t* p = refs + (size_t)c * 64;
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = p[u * 64 + lane];
  };
  auto gather = [&](const int (&r)[U], double (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int f = r[u];
      // (no branch around the load: reference 0 stands in for none)
      const size_t i = f == -1 ? 0 : (size_t)(f & 0x7fffffff) + (f < 0 ? lower : 0u);
      const double x = xa[i];
      v[u] = f == -1 ? 0.0 : x;
    }
  };
  auto add = [&](int c, const double (&v)[U]) {
    const int ends = ref_end[c / U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s += v[u];
      if (ends >> u & 1) {
        out[lane] = (T)s;
        out += 64;
        if constexpr (sizeof(T) == 4) {
          if (val64) out64[lane] = s;
          out64 += 64;
        }
        s = 0.0;
      }
    }
  };
  for (int c = c0; c < c1; c += 2 * U) {
    int ra[U], rb[U];
    double va[U], vb[U];
    load(c, ra);
    if (c + U < c1) {
      load(c + U, rb);
      gather(ra, va);
      gather(rb, vb);
      add(c, va);
      add(c + U, vb);
    } else {
      gather(ra, va);
      add(c, va);
    }
  }
}

// before the launches of a solve whose workgroups do not all run from the start
__global__ void k_rows_start(SyncWords sy) {
  *sy.ticket = 0;
  *sy.start = wall_clock64();
}

__global__ void k_zero_words(u64* p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    p[i] = 0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// device memory of one context's rows; BHIP_ROWS_BYTES limits it
struct RowsMem {
  size_t used = 0, limit = SIZE_MAX;
};
template <typename T>
struct Buf {
  T* p = nullptr;
  size_t bytes = 0;
  RowsMem* mem = nullptr;
  ~Buf() { (void)release(); }
  // (a failure for want of memory is not left as HIP's last error: the caller
  // has another way)
  hipError_t alloc(size_t n, RowsMem& m) {
    const size_t want = std::max<size_t>(n, 1) * sizeof(T);
    if (want > m.limit - m.used) return hipErrorOutOfMemory;
    const hipError_t e = hipMalloc((void**)&p, want);
    if (e != hipSuccess) {
      if (e == hipErrorOutOfMemory) (void)hipGetLastError();
      p = nullptr;
      return e;
    }
    m.used += want;
    bytes = want;
    mem = &m;
    return e;
  }
  hipError_t release() {
    if (!p) return hipSuccess;
    const hipError_t e = hipFree(p);
    mem->used -= bytes;
    p = nullptr;
    bytes = 0;
    return e;
  }
  hipError_t put(const std::vector<T>& v, RowsMem& m, hipStream_t s) {
    hipError_t e = alloc(v.size(), m);
    if (e == hipSuccess && !v.empty())
      e = hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s);
    return e;
  }
};

struct RowsDev {
  RowsMem mem;
  int nslice = 0, group = 1, nwg = 0, nsys = 1, max_halo = 0;
  int64_t nent = 0;
  int ncu = 0, nexp = 0, max_gang = 1;
  std::vector<int32_t> launch;
  Buf<int32_t> wg_row0, slice_off, pair_off, ref_off, refs, wg_sys, sys_wg, halo_off, halo_row, halo_src,
      exp_off;
  Buf<uint16_t> rowpos, ids, exp_loc, refs16;
  Buf<int32_t> slab_slice;  // by_block: first slice of each block's slab
  bool by_block = false;
  int max_slots = 0, lds_max = 0;
  Buf<uint8_t> ref_end;
  Buf<double> v64;
  Buf<float> v32;
  Buf<double> res;  // mixed CG: FP64 residual of each row
  Buf<u64> words;
  SyncWords sy[3];  // CG FP64, CG FP32, GMRES
  int ep[3] = {0, 0, 0};
  size_t sy_words[3] = {0, 0, 0};
  // a launch that is not known to have ended well (rows_ended) may have left
  // any meeting's number in the words: they are cleared before the next one
  bool open[3] = {false, false, false};
  // GMRES: fits (FP64, FP32), scratch for a basis of gm_k vectors
  bool gm_fits[2] = {false, false};
  int nhalo = 0;
  Buf<unsigned char> gm, gmh;
};

template <typename T, typename F>
static hipError_t with_cg_kernel(int group, bool dq, F&& f) {
#define BHIP_CG(R) (dq ? f(&k_cg_rows<T, R, true>) : f(&k_cg_rows<T, R, false>))
  switch (group) {
    case 1: return BHIP_CG(1);
    case 2: return BHIP_CG(2);
    case 4: return BHIP_CG(4);
    default: return BHIP_CG(8);
  }
#undef BHIP_CG
}

template <typename T>
static hipError_t cg_fits(const RowsDev& r, int lds_max, bool* fits) {
  const size_t lds = cg_lds(r.group, r.max_halo, sizeof(T));
  for (int dq = 0; dq < 2; ++dq) {
    const hipError_t e = with_cg_kernel<T>(r.group, dq, [&](auto kern) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
      int nb = 0;
      if (e == hipSuccess)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &nb, reinterpret_cast<const void*>(kern), kSlab, lds);
      *fits = *fits && nb >= 1;
      return e;
    });
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

static size_t gm_lds(const RowsDev& r, int bytes) {
  // V_j and A V_j of own rows and of the halo; mixed: X of both in FP64
  return (size_t)2 * (r.group * kSlab + r.max_halo) * bytes +
         (bytes == 4 ? ((size_t)r.group * kSlab + r.max_halo + 1) * sizeof(double) : 0);
}

template <typename T, typename F>
static hipError_t with_gm_kernel(int group, F&& f) {
  switch (group) {
    case 1: return f(&k_gmres_rows<T, 1>);
    case 2: return f(&k_gmres_rows<T, 2>);
    case 4: return f(&k_gmres_rows<T, 4>);
    default: return f(&k_gmres_rows<T, 8>);
  }
}

template <typename T>
static hipError_t gm_fits(const RowsDev& r, int lds_max, bool* fits) {
  const size_t lds = gm_lds(r, sizeof(T));
  lds_max -= (int)((sizeof(GmLds) + 1023) / 1024 * 1024);
  *fits = lds_max > 0 && lds <= (size_t)lds_max && r.nsys == 1 && r.nwg <= r.ncu;
  if (!*fits) return hipSuccess;
  return with_gm_kernel<T>(r.group, [&](auto kern) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    int nb = 0;
    if (e == hipSuccess)
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(kern),
                                                       kSlab, lds);
    *fits = nb >= 1;
    return e;
  });
}

static u64 wait_ticks() {
  const char* ev = getenv("BHIP_ROWS_WAIT");
  return ev ? strtoull(ev, nullptr, 10) : kWaitTicks;
}

static RowsDev* rows_build(const Layout& L, int nsys, const int64_t* node_off,
                           hipStream_t stream, hipError_t* err) {
  *err = hipSuccess;
  int dev = 0, ncu = 0, lds_max = 0;
  if ((*err = hipGetDevice(&dev)) != hipSuccess) return nullptr;
  if ((*err = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) !=
      hipSuccess)
    return nullptr;
  if ((*err = hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) !=
      hipSuccess)
    return nullptr;
  lds_max -= 2048;  // the CG kernels' static LDS: their sums
  size_t limit = SIZE_MAX;
  if (const char* ev = getenv("BHIP_ROWS_BYTES")) limit = strtoull(ev, nullptr, 10);
  RowLayout R;
  if (limit == 0 || lds_max <= 0 || !build_rows(L, nsys, node_off, ncu, lds_max, R))
    return nullptr;
  std::unique_ptr<RowsDev> r(new RowsDev());
  r->nslice = R.nslice;
  r->group = R.group;
  r->nwg = R.nwg;
  r->nsys = nsys;
  r->max_halo = R.max_halo;
  r->by_block = R.by_block;
  r->max_slots = R.max_slots;
  r->lds_max = lds_max + 2048;
  r->mem.limit = limit;
  r->nent = R.nent + 64;  // load_front reads one entry column of an empty slice too
  r->ncu = ncu;
  r->nexp = (int)R.exp_loc.size();
  r->launch = R.launch;
  r->max_gang = R.max_gang;
  bool fits = true;
  if ((*err = cg_fits<double>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if ((*err = cg_fits<float>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if (!fits) return nullptr;
  if ((*err = gm_fits<double>(*r, r->lds_max, &r->gm_fits[0])) != hipSuccess) return nullptr;
  if ((*err = gm_fits<float>(*r, r->lds_max, &r->gm_fits[1])) != hipSuccess) return nullptr;
  r->nhalo = (int)R.halo_row.size();
  // without memory for them there are no rows, and SOLVE runs element by element
  auto ok = [&](hipError_t e) {
    if (e == hipSuccess) return true;
    if (e != hipErrorOutOfMemory) *err = e;
    (void)hipStreamSynchronize(stream);  // (copies of the host arrays are under way)
    return false;
  };
  std::vector<int32_t> slab_slice;
  if (R.by_block)
    for (int b = 0; b < L.nblocks; ++b) {
      // the workgroup that holds the block's rows, and the first of its waves that do
      const int row = L.node_start[b];
      const int g = (int)(std::upper_bound(R.wg_row0.begin(), R.wg_row0.end(), row) -
                          R.wg_row0.begin()) - 1;
      slab_slice.push_back(g * R.group * kSlices + (row - R.wg_row0[g]) / kSlab * (kSlices / R.group));
    }
  if (!ok(r->wg_row0.put(R.wg_row0, r->mem, stream)) || !ok(r->refs16.put(R.refs16, r->mem, stream)) ||
      !ok(r->slab_slice.put(slab_slice, r->mem, stream)) || !ok(r->slice_off.put(R.slice_off, r->mem, stream)) ||
      !ok(r->pair_off.put(R.pair_off, r->mem, stream)) ||
      !ok(r->refs.put(R.refs, r->mem, stream)) ||
      !ok(r->wg_sys.put(R.wg_sys, r->mem, stream)) || !ok(r->sys_wg.put(R.sys_wg, r->mem, stream)) ||
      !ok(r->halo_off.put(R.halo_off, r->mem, stream)) || !ok(r->halo_row.put(R.halo_row, r->mem, stream)) ||
      !ok(r->halo_src.put(R.halo_src, r->mem, stream)) || !ok(r->exp_off.put(R.exp_off, r->mem, stream)) ||
      !ok(r->rowpos.put(R.rowpos, r->mem, stream)) || !ok(r->ids.put(R.ids, r->mem, stream)) ||
      !ok(r->exp_loc.put(R.exp_loc, r->mem, stream)) || !ok(r->ref_end.put(R.ref_end, r->mem, stream)) ||
      !ok(r->ref_off.put(R.ref_off, r->mem, stream)) || !ok(r->v64.alloc(r->nent, r->mem)))
    return nullptr;
  // sync words of CG in both precisions and of GMRES: sums, exchange, then
  // the counters
  const bool gm = r->gm_fits[0] || r->gm_fits[1];
  const size_t nexp = R.exp_loc.size();
  const size_t nepoch = (2 * (size_t)nsys + 1) / 2 + 1;  // in 64-bit words
  const size_t tail = 4 * nexp + nepoch + 3;
  const size_t nslot[3] = {(size_t)2 * kReplicas * kSums * R.nwg * 2,
                           (size_t)2 * kReplicas * kSums * R.nwg * 2,
                           gm ? (size_t)2 * kReplicas * kGmSums * R.nwg * 2 : 0};
  const size_t nwords = nslot[0] + nslot[1] + nslot[2] + 3 * tail;
  if (!ok(r->words.alloc(nwords, r->mem))) return nullptr;
  u64* p = r->words.p;
  for (int k = 0; k < 3; ++k) {
    SyncWords& s = r->sy[k];
    s.slots = p;
    s.xch = (p += nslot[k]);
    s.epoch = reinterpret_cast<unsigned*>(p += 4 * nexp);
    s.ticket = reinterpret_cast<unsigned*>(p += nepoch);
    s.start = p += 1;
    s.abort = reinterpret_cast<int*>(p += 1);
    s.ticks = wait_ticks();
    p += 1;
    r->sy_words[k] = p - s.slots;
  }
  hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, stream, r->words.p, (long)nwords);
  if (!ok(hipGetLastError()) || !ok(hipStreamSynchronize(stream))) return nullptr;
  return r.release();
}

RowsDev* rows_create(const Layout& L, int nsys, const int64_t* node_off, hipStream_t stream,
                     hipError_t* err) {
  try {
    return rows_build(L, nsys, node_off, stream, err);
  } catch (const std::bad_alloc&) {  // no host memory for them: no rows either
    return nullptr;
  }
}

void rows_destroy(RowsDev* r) { delete r; }

bool rows_meet(const RowsDev* r) { return r->max_gang > 1; }

size_t rows_bytes(const RowsDev* r) { return r->mem.used; }

hipError_t rows_reserve(RowsDev* r, int bytes) {
  if (bytes == 8 || r->v32.p) return hipSuccess;
  hipError_t e = r->res.alloc((size_t)r->nwg * r->group * kSlab, r->mem);
  if (e == hipSuccess) {
    e = r->v32.alloc(r->nent, r->mem);
    if (e != hipSuccess) (void)r->res.release();
  }
  return e;
}

hipError_t rows_assemble(RowsDev* r, int bytes, bool both, const double* xa, int nslot_pad,
                         int npair, bool nonsym, hipStream_t stream) {
  const int nslice = r->nslice;
  const unsigned lower = nonsym ? (unsigned)npair * (unsigned)nslot_pad : 0u;
  const dim3 grid((nslice + 3) / 4), block(256);
  double* none = nullptr;
  if (bytes == 8)
    hipLaunchKernelGGL(k_rows_assemble<double>, grid, block, 0, stream, r->v64.p, none, xa,
                       r->slice_off.p, r->ref_off.p, r->ref_end.p, r->refs.p, nslice, lower);
  else
    hipLaunchKernelGGL(k_rows_assemble<float>, grid, block, 0, stream, r->v32.p,
                       both ? r->v64.p : none, xa, r->slice_off.p, r->ref_off.p, r->ref_end.p,
                       r->refs.p, nslice, lower);
  return hipGetLastError();
}

bool rows_by_block(const RowsDev* r) { return r->by_block; }

hipError_t rows_dmd(RowsDev* r, int bytes, bool both, const RowsDmd& a, hipStream_t stream) {
  const int nc = a.ndp * (a.ndp - 1) / 2 * (a.nonsym ? 2 : 1);
  const size_t lds = ((size_t)nc * r->max_slots + a.max_local + 1) * sizeof(double);
  auto go = [&](auto kern, auto* val) -> hipError_t {
    if (lds > (size_t)r->lds_max) return hipErrorInvalidValue;
    if (lds > 65536) {
      const hipError_t e =
          hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, r->lds_max);
      if (e != hipSuccess) return e;
    }
    const int threads = a.nblocks <= r->ncu ? kDmdThreads : kDmdThreads / 2;
    hipLaunchKernelGGL(kern, dim3(a.nblocks), dim3(threads), lds, stream, a, val,
                       both ? r->v64.p : (double*)nullptr, r->slice_off.p, r->ref_off.p, r->ref_end.p, r->refs16.p, r->slab_slice.p,
                       r->group);
    return hipGetLastError();
  };
#define BHIP_DMD_ROWS(NDP, Q)                                        \
  (bytes == 8 ? go(&k_dmd_rows<NDP, Q, double>, r->v64.p)            \
              : go(&k_dmd_rows<NDP, Q, float>, r->v32.p))
  if (a.ndp == 2) return a.nonsym ? BHIP_DMD_ROWS(2, true) : BHIP_DMD_ROWS(2, false);
  return a.nonsym ? BHIP_DMD_ROWS(3, true) : BHIP_DMD_ROWS(3, false);
#undef BHIP_DMD_ROWS
}

// for a launch of kind k, which counts as open from here on
static RowArgs row_args(RowsDev* r, int k, hipStream_t stream) {
  if (r->open[k]) {
    hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, stream, r->sy[k].slots,
                       (long)r->sy_words[k]);
    r->ep[k] = 0;
    r->sy[k].ticks = wait_ticks();
  }
  r->open[k] = true;
  RowArgs a;
  a.slice_off = r->slice_off.p;
  a.pair_off = r->pair_off.p;
  a.ids = reinterpret_cast<const unsigned*>(r->ids.p);
  a.rowpos = r->rowpos.p;
  a.wg_row0 = r->wg_row0.p;
  a.wg_sys = r->wg_sys.p;
  a.sys_wg = r->sys_wg.p;
  a.halo_off = r->halo_off.p;
  a.halo_row = r->halo_row.p;
  a.halo_src = r->halo_src.p;
  a.exp_off = r->exp_off.p;
  a.exp_loc = r->exp_loc.p;
  a.nwg = r->nwg;
  a.nsys = r->nsys;
  a.nexp = r->nexp;
  a.nhalo = r->nhalo;
  a.sy = r->sy[k];
  a.ep = r->ep[k];
  r->ep[k] ^= 1;
  a.first = 0;
  a.rounds = r->nwg > r->ncu;
  a.ticketed = a.rounds && r->launch.size() == 2;
  return a;
}

void rows_ended(RowsDev* r, RowsKind k) { r->open[k] = false; }

hipError_t rows_cg(RowsDev* r, bool mixed, RowsCg a, hipStream_t stream) {
  a.res = r->res.p;
  RowArgs ra = row_args(r, mixed ? kRowsCgMixed : kRowsCg, stream);
  if (ra.rounds) hipLaunchKernelGGL(k_rows_start, dim3(1), dim3(1), 0, stream, ra.sy);
  const size_t lds = cg_lds(r->group, r->max_halo, mixed ? 4 : 8);
  auto go = [&](auto kern, auto* val) -> hipError_t {
    for (size_t i = 0; i + 1 < r->launch.size(); ++i) {
      ra.first = r->launch[i];
      hipLaunchKernelGGL(kern, dim3(r->launch[i + 1] - ra.first), dim3(kSlab), lds, stream, ra,
                         val, r->v64.p, a);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  };
  if (mixed)
    return with_cg_kernel<float>(r->group, a.diag != nullptr,
                                 [&](auto kern) { return go(kern, r->v32.p); });
  return with_cg_kernel<double>(r->group, a.diag != nullptr,
                                [&](auto kern) { return go(kern, r->v64.p); });
}

bool rows_gmres_fits(const RowsDev* r, int bytes) { return r->gm_fits[bytes == 4]; }

template <typename T>
hipError_t rows_gmres(RowsDev* r, const RowsGmres& a, hipStream_t stream) {
  if (a.krylov < 1 || a.krylov > kGmMaxK) return hipErrorInvalidValue;
  // V, A V (FP64 only) and the diagonal of own rows; V of the halo
  const size_t own = (size_t)r->nwg * r->group * kSlab * sizeof(T) *
                     ((sizeof(T) == 8 ? 2 : 1) * a.krylov + 1);
  const size_t halo = (size_t)std::max(r->nhalo, 1) * sizeof(T) * a.krylov;
  auto grow = [&](Buf<unsigned char>& b, size_t want) -> hipError_t {
    if (b.bytes >= want) return hipSuccess;
    const hipError_t e = b.release();
    return e == hipSuccess ? b.alloc(want, r->mem) : e;
  };
  hipError_t e = grow(r->gm, own);
  if (e == hipSuccess) e = grow(r->gmh, halo);
  if (e != hipSuccess) return e;
  const RowArgs ra = row_args(r, kRowsGmres, stream);
  const T* val;
  if constexpr (sizeof(T) == 8)
    val = r->v64.p;
  else
    val = r->v32.p;
  return with_gm_kernel<T>(r->group, [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(r->nwg), dim3(kSlab), gm_lds(*r, sizeof(T)), stream, ra, val,
                       r->v64.p, a, reinterpret_cast<T*>(r->gm.p),
                       reinterpret_cast<T*>(r->gmh.p));
    return hipGetLastError();
  });
}
template hipError_t rows_gmres<double>(RowsDev*, const RowsGmres&, hipStream_t);
template hipError_t rows_gmres<float>(RowsDev*, const RowsGmres&, hipStream_t);


}  // namespace bhip
