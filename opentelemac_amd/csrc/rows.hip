// Persistent Krylov kernels on assembled rows (rows.h), MI355X.
//
// One launch runs a whole CG solve. Each workgroup (one per CU, 1024 threads)
// keeps the residual and the solution of its rows in registers, `group` rows
// per thread, and D and A D in LDS; the first kFront coefficients of each row
// stay in registers too where they fit (FP64 groups of 1 and 2, FP32 up to 4).
// Larger groups read the matrix again each iteration, out of the last-level
// cache (120 MB for 2M rows in FP64).
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
// us per iteration, FP64 / FP32 rows: 1.4 / 1.7 (1,000 nodes, one workgroup),
// 3.2 / 3.1 (20k), 3.9 / 3.7 (100k), 4.7 / 4.7 (260k), 5.8 / 5.5 (500k), 14.0 /
// 7.9 (1M), 24.4 / 16.7 (2M). The two-kernel CG takes 15 at 20k, 50 (FP64) at
// 2M and 22 (FP32) at 1M. What bounds it: below 500k the meeting (two trips
// through memory, 1.7 us for 20 workgroups, 3.5 for 245), then the matrix
// (8.0 TB/s in FP64 and 8.7 in FP32 at 2M rows).
//
// Sums are binary trees over the rows' leaf numbers (rows.h) and do not depend
// on how many rows a workgroup holds: a system gives the same bits alone and
// in an ensemble.
//
// Every wait ends: on the number it waits for, or after kWaitTicks of the
// device clock, when the launch gives up (abort in the sync words), leaves the
// initial solution as it was and the host falls back to the two-kernel CG
// (BHIP_ROWS_WAIT=<ticks> changes the limit; 0 gives up at the first word that
// is not there yet, which the tests use).
// All workgroups of a system must be resident at once: the host launches at
// most one such kernel per GPU at a time. When a launch has more workgroups
// than fit the GPU, they take their numbers in the order in which they start,
// so the system with the lowest numbers always has all of its own running.
#include "rows_dev.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <memory>
#include <vector>

namespace bhip {

typedef unsigned long long u64;

constexpr int kReplicas = 8;
constexpr int kSums = 4;  // sums of one meeting
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
struct Deadline {
  u64 t0, ticks;
  const int* abort;
  __device__ bool past(int& n) const {
    return ((++n & 255) == 0 || ticks == 0) &&
           ((u64)wall_clock64() - t0 >= ticks || load_relaxed(abort));
  }
};

// the sync words of one precision
struct SyncWords {
  u64* slots;       // [2][kReplicas][kSums][nwg][2] sums, by parity of the meeting
  u64* xch;         // [2][2][exported rows], by parity of the meeting (a float has one
                    // word only)
  unsigned* epoch;  // [2][nsys] number of the last meeting, by parity of the launch
  int* abort;       // a launch has given up
  unsigned* ticket; // workgroups started (launches larger than the GPU)
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
  int nwg, nsys, nexp;
  SyncWords sy;
  int ep;        // parity of the launch
  int ticketed;  // workgroup numbers by order of start
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
                            unsigned lane, const T* ys) {
  T c[W];
  unsigned i[(W + 1) / 2];
#pragma unroll
  for (int j = 0; j < (W + 1) / 2; ++j) i[j] = id[j * 64 + lane];
#pragma unroll
  for (int j = 0; j < W; ++j) c[j] = v[j * 64 + lane];
  T s = (T)0;
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

// The first kFront entries of one row, kept in registers for a whole solve.
// Slices with fewer read their last one again and multiply it by zero.
constexpr int kFront = 8;
template <typename T>
struct RowFront {
  T c[kFront];
  unsigned i[kFront / 2];  // two ids each
};
template <typename T>
__device__ inline void load_front(RowFront<T>& f, const T* __restrict__ v,
                                  const unsigned* __restrict__ id, unsigned lane, int w) {
  const int last = max(w - 1, 0);
#pragma unroll
  for (int j = 0; j < kFront / 2; ++j) f.i[j] = (id + min(j, last / 2) * 64)[lane];
#pragma unroll
  for (int j = 0; j < kFront; ++j) {
    const T c = (v + min(j, last) * 64)[lane];
    f.c[j] = j < w ? c : (T)0;
  }
}
template <typename T>
__device__ inline T front_dot(const RowFront<T>& f, const T* ys) {
  T s = (T)0;
#pragma unroll
  for (int j = 0; j < kFront; ++j)
    s += f.c[j] * ys[j & 1 ? f.i[j / 2] >> 16 : f.i[j / 2] & 0xffffu];
  return s;
}

// ---------------------------------------------------------------------------
// CG
// ---------------------------------------------------------------------------
template <typename T, int R, bool DQ>
__global__ void __launch_bounds__(kSlab)
k_cg_rows(RowArgs ra, const T* __restrict__ val, RowsCg<T> a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double sh_sum[kSums * kRowWaves];
  __shared__ double sh_in[kRowWaves];
  __shared__ int sh_bad, sh_wg;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t == 0) {
    sh_bad = 0;
    sh_wg = ra.ticketed ? (int)(atomicAdd(ra.sy.ticket, 1u) % (unsigned)ra.nwg) : blockIdx.x;
  }
  __syncthreads();
  const int wg = __builtin_amdgcn_readfirstlane(sh_wg);
  const int sys = ra.wg_sys[wg];
  const int g0 = ra.sys_wg[sys], gang = ra.sys_wg[sys + 1] - g0;
  const bool lead = wg == g0 && t == 0;
  SolveState* st = a.st + sys;
  unsigned e = __hip_atomic_load(ra.sy.epoch + ra.ep * ra.nsys + sys, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
  // (no workgroup writes a field that another may still have to read here: a
  // solve that stops without a meeting would race with a late workgroup)
  const bool skip = load_relaxed(&st->zero_rhs) || (a.inner && !load_relaxed(&st->fresh)) ||
                    load_relaxed(ra.sy.abort);
  if (skip) {
    if (load_relaxed(ra.sy.abort)) store_relaxed(&st->gave_up, 1);
    if (lead)
      __hip_atomic_store(ra.sy.epoch + (1 - ra.ep) * ra.nsys + sys, e, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const Deadline dl = {(u64)wall_clock64(), ra.sy.ticks, ra.sy.abort};
  const int r0 = ra.wg_row0[wg];
  const uint16_t* rowpos = ra.rowpos + (size_t)wg * R * kSlab;
  const int h0 = ra.halo_off[wg], nh = ra.halo_off[wg + 1] - h0;
  const int x0 = ra.exp_off[wg], nx = ra.exp_off[wg + 1] - x0;
  T* ds = reinterpret_cast<T*>(smem_raw);  // D: own rows, then halo
  T* dh = ds + R * kSlab;
  T* ah = dh + nh;                         // A D of the halo as it arrives
  T* rh = ah + nh;                         // R of the halo
  T* as = rh + nh;                         // A D of own rows

  // ||r0||^2: the state's, or the partial sums per node block
  double rr;
  if (a.part_rr) {
    const int pb0 = a.sys_blocks ? a.sys_blocks[sys] : 0;
    const int pb1 = a.sys_blocks ? a.sys_blocks[sys + 1] : a.nblocks;
    double p = 0.0;
    for (int i = pb0 + t; i < pb1; i += kSlab) p += a.part_rr[i];
    const double s = tree_sum<1, 1>([&](int) { return Sums<1>{{p}}; }, sh_sum);
    if (t == 0) sh_in[0] = s;
    __syncthreads();
    rr = sh_in[0];
    __syncthreads();
  } else {
    rr = ld_f64(&st->rr0);
  }
  int m = load_relaxed(&st->m[1]) + 1;
  double rr_prev = ld_f64(&st->rr[1]);
  const double thr = ld_f64(&st->eps2xl) * (load_relaxed(&st->use_rr0) ? ld_f64(&st->rr0) : 1.0);
  const int nitmax = load_relaxed(&st->nitmax);

  // the coefficients of small partitions stay in registers for the whole solve
  constexpr bool kKeep = R * sizeof(T) <= 16;
  RowFront<T> front[kKeep ? R : 1];
  int wid[kKeep ? R : 1];
  // the slice of this wave's k-th rows: its coefficients, id words and width
  auto slice = [&](int k, const T*& v, const unsigned*& id) -> int {
    const int q = __builtin_amdgcn_readfirstlane((wg * R + k) * kSlices + wave);
    const int o = ra.slice_off[q];
    v = val + (size_t)o * 64;
    id = ra.ids + (size_t)ra.pair_off[q] * 64;
    return ra.slice_off[q + 1] - o;
  };
  unsigned have = 0;  // bit k: this thread has a k-th row
  T rv[R], xv[R], dq[DQ ? R : 1];
  const double beta0 = m == 0 ? 0.0 : rr / rr_prev;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    // (a few rows' addresses at a time)
    if constexpr (R >= 4) __builtin_amdgcn_sched_barrier(0);
    rv[k] = xv[k] = (T)0;
    if constexpr (DQ) dq[k] = (T)0;
    T d = (T)0;
    const int p = rowpos[k * kSlab + t];
    if (p != 0xffff) {
      const int row = r0 + p;
      have |= 1u << k;
      rv[k] = a.r0[row];
      if (a.x0) xv[k] = a.x0[row];
      if constexpr (DQ) dq[k] = a.diag[row];
      d = rv[k];
      if (m > 0) d += (T)beta0 * a.dlast[row];
    }
    ds[k * kSlab + t] = d;
    if constexpr (kKeep) {
      const T* v;
      const unsigned* id;
      wid[k] = slice(k, v, id);
      load_front(front[k], v, id, lane, wid[k]);
    }
  }
  for (int h = t; h < nh; h += kSlab) {
    const int g = ra.halo_row[h0 + h];
    T d = a.r0[g];
    rh[h] = d;
    if (m > 0) d += (T)beta0 * a.dlast[g];
    dh[h] = d;
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
    int n = 0;
    while (need_s || need_h) {
      if (need_s) need_s = !look(sp, 1, e, p);
      if constexpr (halo.value)
        if (need_h) need_h = !look(hp, ra.nexp, e, hv);
      if ((need_s || need_h) && dl.past(n)) break;
    }
    bool ok = !(need_s || need_h);
    if constexpr (halo.value) {
      if (tt < nh) ah[tt] = hv;
      for (int h = tt + kSlab; h < nh && ok; h += kSlab) {
        T v2;
        while (!look(xch + ra.halo_src[h0 + h], ra.nexp, e, v2))
          if (dl.past(n)) {
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

  // stop test (gracjg.F:306-324; strict for the initial residual, :219)
  bool stop = m == 0 ? rr < thr : rr <= thr;
  int status = ST_CONVERGED;
  while (!stop) {
    // AD
    if constexpr (kKeep) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        T s = front_dot(front[k], ds);
        if (wid[k] > kFront) {
          const T* v;
          const unsigned* id;
          slice(k, v, id);
          s += slice_dot<4>(v, id, lane, kFront, wid[k], ds);
        }
        as[k * kSlab + t] = s;
        // (one slab's gathers at a time, as above)
        if constexpr (R >= 2) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma nounroll
      for (int k = 0; k < R; ++k) {
        const T* v;
        const unsigned* id;
        const int w = slice(k, v, id);
        as[k * kSlab + t] = slice_dot<8>(v, id, lane, 0, w, ds);
      }
    }
    if constexpr (DQ) {
#pragma unroll
      for (int k = 0; k < R; ++k)
        as[k * kSlab + t] += dq[k] * ds[k * kSlab + t];
    } else {
#pragma unroll
      for (int k = 0; k < R; ++k)
        as[k * kSlab + t] += ds[k * kSlab + t];
    }
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
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (have >> k & 1) {
      const int row = r0 + rowpos[k * kSlab + t];
      a.x[row] = xv[k];
      if (a.dlast) a.dlast[row] = ds[k * kSlab + t];
    }
  if (lead) {
    st->final_m = m;
    st->final_rr = rr;
    // the ||R||^2 that built the last direction (continued solves)
    st->rr[0] = rr_prev;
    st->rr[1] = rr_prev;
    st->t_done = wall_clock64();
    store_relaxed(&st->done1, (m << 2) | status);
    store_relaxed(&st->done, status);
    store_relaxed(&st->stop, 1);
    __hip_atomic_store(ra.sy.epoch + (1 - ra.ep) * ra.nsys + sys, e, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------------------
// D A D and assembly of one node block: its coefficients are scaled, written
// back and kept in LDS, where the block's 16 slices sum them. A gather from
// memory instead takes a cache line per coefficient (k_rows_assemble: 138 us
// for 2M nodes in FP64, after 49 us for the scaling alone). Bound by memory:
// 105 us for 2M nodes in FP64 (450 MB, 4.3 TB/s), 48 us for 1M in FP32. 512
// threads: two blocks per CU, one gathers while the other loads.
// ---------------------------------------------------------------------------
constexpr int kDmdThreads = 512;
template <int NDP, bool Q, typename T>
__global__ void __launch_bounds__(kDmdThreads)
k_dmd_rows(RowsDmd a, T* __restrict__ val, const int32_t* __restrict__ slice_off,
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
    for (int l = t; l < nloc; l += kDmdThreads)
      ds[l] = a.d[l < nown ? n0 + l : a.halo[h0 + l - nown]];
    __syncthreads();
  }
  for (int i = t; i < ns; i += kDmdThreads) {
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
  for (int i = wave; i < kSlices; i += kDmdThreads / 64) {
    const int q = __builtin_amdgcn_readfirstlane(q0 + i % group * kSlices + i / group);
    const int c1 = ref_off[q + 1];
    T* out = val + (size_t)slice_off[q] * 64;
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
k_rows_assemble(T* __restrict__ val, const double* __restrict__ xa,
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

__global__ void k_zero_words(u64* p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    p[i] = 0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <typename T>
struct Buf {
  T* p = nullptr;
  ~Buf() {
    if (p) (void)hipFree(p);
  }
  hipError_t alloc(size_t n) {
    return hipMalloc((void**)&p, std::max<size_t>(n, 1) * sizeof(T));
  }
  hipError_t put(const std::vector<T>& v, hipStream_t s) {
    hipError_t e = alloc(v.size());
    if (e == hipSuccess && !v.empty())
      e = hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s);
    return e;
  }
};

struct RowsDev {
  int nslice = 0, group = 1, nwg = 0, nsys = 1, max_halo = 0;
  int64_t nent = 0;
  int ncu = 0, nexp = 0;
  Buf<int32_t> wg_row0, slice_off, pair_off, ref_off, refs, wg_sys, sys_wg, halo_off, halo_row, halo_src,
      exp_off;
  Buf<uint16_t> rowpos, ids, exp_loc, refs16;
  Buf<int32_t> slab_slice;  // by_block: first slice of each block's slab
  bool by_block = false;
  int max_slots = 0, lds_max = 0;
  Buf<uint8_t> ref_end;
  Buf<double> v64;
  Buf<float> v32;
  Buf<u64> words;
  SyncWords sy[2];  // FP64, FP32
  int ep[2] = {0, 0};
};

static size_t cg_lds(const RowsDev& r, int bytes) {
  // D and A D of own rows; D, A D and R of the halo
  return ((size_t)2 * r.group * kSlab + (size_t)3 * r.max_halo) * bytes;
}

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
  const size_t lds = cg_lds(r, sizeof(T));
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

RowsDev* rows_create(const Layout& L, int nsys, const int64_t* node_off, hipStream_t stream,
                     hipError_t* err) {
  *err = hipSuccess;
  int dev = 0, ncu = 0, lds_max = 0;
  if ((*err = hipGetDevice(&dev)) != hipSuccess) return nullptr;
  if ((*err = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) !=
      hipSuccess)
    return nullptr;
  if ((*err = hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) !=
      hipSuccess)
    return nullptr;
  RowLayout R;
  if (!build_rows(L, nsys, node_off, ncu, R)) return nullptr;
  // the kernels may read one entry column past the last slice (load_front)
  R.ids.resize(R.ids.size() + 128, 0);
  std::unique_ptr<RowsDev> r(new RowsDev());
  r->nslice = R.nslice;
  r->group = R.group;
  r->nwg = R.nwg;
  r->nsys = nsys;
  r->max_halo = R.max_halo;
  r->by_block = R.by_block;
  r->max_slots = R.max_slots;
  r->lds_max = lds_max;
  r->nent = R.nent + 64;
  r->ncu = ncu;
  r->nexp = (int)R.exp_loc.size();
  lds_max -= 2048;  // the kernels' static LDS: their sums
  if (cg_lds(*r, sizeof(double)) > (size_t)lds_max) return nullptr;
  bool fits = true;
  if ((*err = cg_fits<double>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if ((*err = cg_fits<float>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if (!fits) return nullptr;
  auto ok = [&](hipError_t e) {
    if (e != hipSuccess) *err = e;
    return e == hipSuccess;
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
  if (!ok(r->wg_row0.put(R.wg_row0, stream)) || !ok(r->refs16.put(R.refs16, stream)) ||
      !ok(r->slab_slice.put(slab_slice, stream)) || !ok(r->slice_off.put(R.slice_off, stream)) ||
      !ok(r->pair_off.put(R.pair_off, stream)) ||
      !ok(r->refs.put(R.refs, stream)) ||
      !ok(r->wg_sys.put(R.wg_sys, stream)) || !ok(r->sys_wg.put(R.sys_wg, stream)) ||
      !ok(r->halo_off.put(R.halo_off, stream)) || !ok(r->halo_row.put(R.halo_row, stream)) ||
      !ok(r->halo_src.put(R.halo_src, stream)) || !ok(r->exp_off.put(R.exp_off, stream)) ||
      !ok(r->rowpos.put(R.rowpos, stream)) || !ok(r->ids.put(R.ids, stream)) ||
      !ok(r->exp_loc.put(R.exp_loc, stream)) || !ok(r->ref_end.put(R.ref_end, stream)) ||
      !ok(r->ref_off.put(R.ref_off, stream)) || !ok(r->v64.alloc(r->nent)))
    return nullptr;
  // sync words: per precision sums and exchange, then the counters
  const size_t nslot = (size_t)2 * kReplicas * kSums * R.nwg * 2, nexp = R.exp_loc.size();
  const size_t nepoch = (2 * (size_t)nsys + 1) / 2 + 1;  // in 64-bit words
  const size_t one = nslot + 4 * nexp + nepoch + 2;
  if (!ok(r->words.alloc(2 * one))) return nullptr;
  u64 ticks = kWaitTicks;
  if (const char* ev = getenv("BHIP_ROWS_WAIT")) ticks = strtoull(ev, nullptr, 10);
  for (int k = 0; k < 2; ++k) {
    u64* p = r->words.p + k * one;
    r->sy[k].slots = p;
    r->sy[k].xch = p + nslot;
    r->sy[k].epoch = reinterpret_cast<unsigned*>(p + nslot + 4 * nexp);
    r->sy[k].abort = reinterpret_cast<int*>(p + one - 2);
    r->sy[k].ticket = reinterpret_cast<unsigned*>(p + one - 1);
    r->sy[k].ticks = ticks;
  }
  hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, stream, r->words.p, (long)(2 * one));
  if (!ok(hipGetLastError()) || !ok(hipStreamSynchronize(stream))) return nullptr;
  return r.release();
}

void rows_destroy(RowsDev* r) { delete r; }

hipError_t rows_reserve(RowsDev* r, int bytes) {
  if (bytes == 8) return r->v64.p ? hipSuccess : r->v64.alloc(r->nent);
  return r->v32.p ? hipSuccess : r->v32.alloc(r->nent);
}

hipError_t rows_assemble(RowsDev* r, int bytes, const double* xa, int nslot_pad, int npair,
                         bool nonsym, hipStream_t stream) {
  const int nslice = r->nslice;
  const unsigned lower = nonsym ? (unsigned)npair * (unsigned)nslot_pad : 0u;
  const dim3 grid((nslice + 3) / 4), block(256);
  if (bytes == 8)
    hipLaunchKernelGGL(k_rows_assemble<double>, grid, block, 0, stream, r->v64.p, xa,
                       r->slice_off.p, r->ref_off.p, r->ref_end.p, r->refs.p, nslice, lower);
  else
    hipLaunchKernelGGL(k_rows_assemble<float>, grid, block, 0, stream, r->v32.p, xa,
                       r->slice_off.p, r->ref_off.p, r->ref_end.p, r->refs.p, nslice, lower);
  return hipGetLastError();
}

bool rows_by_block(const RowsDev* r) { return r->by_block; }

hipError_t rows_dmd(RowsDev* r, int bytes, const RowsDmd& a, hipStream_t stream) {
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
    hipLaunchKernelGGL(kern, dim3(a.nblocks), dim3(kDmdThreads), lds, stream, a, val,
                       r->slice_off.p, r->ref_off.p, r->ref_end.p, r->refs16.p, r->slab_slice.p,
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

static RowArgs row_args(const RowsDev* r, int k) {
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
  a.sy = r->sy[k];
  a.ep = r->ep[k];
  a.ticketed = r->nwg > r->ncu;
  return a;
}

template <typename T>
hipError_t rows_cg(RowsDev* r, const RowsCg<T>& a, hipStream_t stream) {
  const int k = sizeof(T) == 4;
  const RowArgs ra = row_args(r, k);
  r->ep[k] ^= 1;
  const T* val;
  if constexpr (sizeof(T) == 8)
    val = r->v64.p;
  else
    val = r->v32.p;
  if (ra.ticketed) {
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(64), 0, stream,
                       reinterpret_cast<u64*>(ra.sy.ticket), 1L);
  }
  return with_cg_kernel<T>(r->group, a.diag != nullptr, [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(r->nwg), dim3(kSlab), cg_lds(*r, sizeof(T)), stream, ra, val, a);
    return hipGetLastError();
  });
}
template hipError_t rows_cg<double>(RowsDev*, const RowsCg<double>&, hipStream_t);
template hipError_t rows_cg<float>(RowsDev*, const RowsCg<float>&, hipStream_t);

}  // namespace bhip
