// Persistent Krylov kernels on assembled rows (rows.h), MI355X.
//
// One launch runs a whole CG solve. Each workgroup (one per CU, 1024 threads)
// keeps the residual, the solution and A D of its rows in registers, one row
// of each of its slabs per thread, and the direction D of its rows and halo in
// LDS; only the matrix is read again each iteration, and at most 2M rows of it
// (120 MB in FP64) stay in the last-level cache.
//
// Workgroups meet twice per iteration (D.AD; ||R||^2 together with the
// exchange of halo residuals). There are no fences: every word that crosses
// workgroups is written and read with 64-bit relaxed atomics at agent scope
// and carries the number of the meeting in its low half (a double travels as
// two such words), so reading the right number is the synchronisation. Each
// workgroup writes its sum to kReplicas places and reads all sums of its
// system from one of them, which spreads the readers over the memory
// channels. Measured per meeting on 8 XCDs: 1.35 us for 16 workgroups, 1.6
// for 64, 2.0 for 128, 2.8 for 256 (one place instead of 8: 4.0 for 256; two
// levels of 16: 3.5).
//
// Sums are binary trees over rows aligned on powers of two, so they do not
// depend on how many slabs a workgroup holds: a system gives the same bits
// alone and in an ensemble.
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

#include <cstdlib>
#include <memory>
#include <vector>

namespace bhip {

typedef unsigned long long u64;

constexpr int kReplicas = 8;
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
template <typename T>
constexpr int kWords = sizeof(T) / 4;
__device__ inline void post(u64* p, unsigned e, double v) {
  const u64 b = __double_as_longlong(v);
  st_word(p, (b & 0xffffffff00000000ull) | e);
  st_word(p + 1, (b << 32) | e);
}
__device__ inline void post(u64* p, unsigned e, float v) {
  st_word(p, ((u64)__float_as_uint(v) << 32) | e);
}
// waits for the value numbered e; false after the deadline
struct Deadline {
  u64 t0, ticks;
  const int* abort;
  __device__ bool past(int& n) const {
    return ((++n & 255) == 0 || ticks == 0) &&
           ((u64)wall_clock64() - t0 >= ticks || load_relaxed(abort));
  }
};
__device__ inline bool await(const u64* p, unsigned e, double& v, const Deadline& dl) {
  u64 a, b;
  for (int n = 0;;) {
    a = ld_word(p);
    b = ld_word(p + 1);
    if ((unsigned)a == e && (unsigned)b == e) break;
    if (dl.past(n)) return false;
  }
  v = __longlong_as_double((a & 0xffffffff00000000ull) | (b >> 32));
  return true;
}
__device__ inline bool await(const u64* p, unsigned e, float& v, const Deadline& dl) {
  u64 a;
  for (int n = 0;;) {
    a = ld_word(p);
    if ((unsigned)a == e) break;
    if (dl.past(n)) return false;
  }
  v = __uint_as_float((unsigned)(a >> 32));
  return true;
}

// the sync words of one precision
struct SyncWords {
  u64* slots;       // [2][kReplicas][nwg][2] sums, by parity of the meeting
  u64* xch;         // [exported rows][kWords]
  unsigned* epoch;  // [2][nsys] number of the last meeting, by parity of the launch
  int* abort;       // a launch has given up
  unsigned* ticket; // workgroups started (launches larger than the GPU)
  u64 ticks;        // longest wait
};

struct RowArgs {
  const int32_t* slice_off;
  const uint16_t* ids;
  const uint16_t* rowpos;
  const int32_t* slab_row0;
  const int32_t* wg_slab0;
  const int32_t* wg_sys;
  const int32_t* sys_wg;
  const int32_t* halo_off;
  const int32_t* halo_row;
  const int32_t* halo_src;
  const int32_t* exp_off;
  const uint16_t* exp_loc;
  int nwg, nsys, nslab;
  SyncWords sy;
  int ep;        // parity of the launch
  int ticketed;  // workgroup numbers by order of start
};

// ---------------------------------------------------------------------------
// sums
// ---------------------------------------------------------------------------
__device__ inline double lane_tree(double v, int from) {
  for (int m = from; m < 64; m <<= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// the workgroup's sum of v[k] over threads and slabs, as an aligned binary
// tree over rows (slab k, thread t). Valid in wave 0. sh: [R * kRowWaves].
// Ends with nothing pending on sh that the next call's first barrier does not
// cover (one barrier between two calls is enough).
template <int R>
__device__ inline double tree_sum(const double (&v)[R], double* sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // lanes halve the slabs they carry while summing over lane pairs
  double a[R];
#pragma unroll
  for (int k = 0; k < R; ++k) a[k] = v[k];
  int slab = 0, mask = 1;
#pragma unroll
  for (int h = R / 2; h >= 1; h >>= 1) {
    const bool up = lane & mask;
#pragma unroll
    for (int k = 0; k < h; ++k) {
      const double keep = up ? a[k + h] : a[k];
      const double give = up ? a[k] : a[k + h];
      a[k] = keep + __shfl_xor(give, mask, 64);
    }
    slab += up ? h : 0;
    mask <<= 1;
  }
  const double s = lane_tree(a[0], R);
  if (lane < R) sh[slab * kRowWaves + w] = s;
  __syncthreads();
  double t = 0.0;
  if (w == 0) {
    const int wl = lane & 15, g = lane >> 4;
    if constexpr (R == 8) {
      double p = sh[(2 * g) * kRowWaves + wl], q = sh[(2 * g + 1) * kRowWaves + wl];
      for (int m = 1; m < 16; m <<= 1) {
        p += __shfl_xor(p, m, 64);
        q += __shfl_xor(q, m, 64);
      }
      t = p + q;
    } else {
      t = g < R ? sh[g * kRowWaves + wl] : 0.0;
      for (int m = 1; m < 16; m <<= 1) t += __shfl_xor(t, m, 64);
    }
    t += __shfl_xor(t, 16, 64);
    t += __shfl_xor(t, 32, 64);
  }
  return t;
}

// ---------------------------------------------------------------------------
// row products
// ---------------------------------------------------------------------------
// sum of W entries of this lane's row of a slice whose entries start at v, id
// (the same in the whole wave: scalar bases, one 32-bit offset per lane)
template <typename T, int W>
__device__ inline T row_dot(const T* __restrict__ v, const uint16_t* __restrict__ id,
                            unsigned lane, const T* ys) {
  T c[W];
  int i[W];
#pragma unroll
  for (int j = 0; j < W; ++j) {
    c[j] = v[j * 64 + lane];
    i[j] = id[j * 64 + lane];
  }
  T s = c[0] * ys[i[0]];
#pragma unroll
  for (int j = 1; j < W; ++j) s += c[j] * ys[i[j]];
  return s;
}

// sum over the w entries (w the same in the whole wave), eight in flight
template <typename T>
__device__ inline T slice_dot(const T* __restrict__ v, const uint16_t* __restrict__ id,
                              unsigned lane, int w, const T* ys) {
  T s = (T)0;
  while (w >= 8) {
    s += row_dot<T, 8>(v, id, lane, ys);
    v += 8 * 64;
    id += 8 * 64;
    w -= 8;
  }
  switch (w) {
    case 7: s += row_dot<T, 7>(v, id, lane, ys); break;
    case 6: s += row_dot<T, 6>(v, id, lane, ys); break;
    case 5: s += row_dot<T, 5>(v, id, lane, ys); break;
    case 4: s += row_dot<T, 4>(v, id, lane, ys); break;
    case 3: s += row_dot<T, 3>(v, id, lane, ys); break;
    case 2: s += row_dot<T, 2>(v, id, lane, ys); break;
    case 1: s += row_dot<T, 1>(v, id, lane, ys); break;
    default: break;
  }
  return s;
}

// ---------------------------------------------------------------------------
// CG
// ---------------------------------------------------------------------------
template <typename T, int R, bool DQ>
__global__ void __launch_bounds__(kSlab)
k_cg_rows(RowArgs ra, const T* __restrict__ val, RowsCg<T> a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double sh_sum[R * kRowWaves];
  __shared__ double sh_in[4];
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
  const int k0 = ra.wg_slab0[wg], nk = ra.wg_slab0[wg + 1] - k0;
  const int h0 = ra.halo_off[wg], nh = ra.halo_off[wg + 1] - h0;
  const int x0 = ra.exp_off[wg], nx = ra.exp_off[wg + 1] - x0;
  T* ds = reinterpret_cast<T*>(smem_raw);  // D: own rows, then halo
  T* dh = ds + R * kSlab;
  T* hr = dh + nh;                         // halo residuals as they arrive
  // also holds the exported residuals of the workgroup (by LDS index) while
  // they are posted: the residuals themselves live in registers
  T* rs = hr + nh;

  // ||r0||^2: the state's, or the partial sums per node block
  double rr;
  if (a.part_rr) {
    const int pb0 = a.sys_blocks ? a.sys_blocks[sys] : 0;
    const int pb1 = a.sys_blocks ? a.sys_blocks[sys + 1] : a.nblocks;
    double p[1] = {0.0};
    for (int i = pb0 + t; i < pb1; i += kSlab) p[0] += a.part_rr[i];
    const double s = tree_sum<1>(p, sh_sum);
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

  int off[R];         // slices of this wave: first entries and widths (scalars)
  int wid[R];
  unsigned have = 0;  // bit k: this thread has a row in slab k
  T rv[R], xv[R], ad[R], dq[DQ ? R : 1];
  const double beta0 = m == 0 ? 0.0 : rr / rr_prev;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    off[k] = wid[k] = 0;
    rv[k] = xv[k] = ad[k] = (T)0;
    if constexpr (DQ) dq[k] = (T)0;
    T d = (T)0;
    if (k < nk) {
      const int q = (k0 + k) * kSlices + wave;
      off[k] = __builtin_amdgcn_readfirstlane(ra.slice_off[q]);
      wid[k] = __builtin_amdgcn_readfirstlane(ra.slice_off[q + 1]) - off[k];
      const int p = ra.rowpos[(size_t)(k0 + k) * kSlab + t];
      if (p != 0xffff) {
        const int row = ra.slab_row0[k0 + k] + p;
        have |= 1u << k;
        rv[k] = a.r0[row];
        if (a.x0) xv[k] = a.x0[row];
        if constexpr (DQ) dq[k] = a.diag[row];
        d = rv[k];
        if (m > 0) d += (T)beta0 * a.dlast[row];
      }
    }
    ds[k * kSlab + t] = d;
  }
  for (int h = t; h < nh; h += kSlab) {
    const int g = ra.halo_row[h0 + h];
    T d = a.r0[g];
    if (m > 0) d += (T)beta0 * a.dlast[g];
    dh[h] = d;
  }
  __syncthreads();

  // a meeting: the system's sum of v (and, in `halo`, the halo residuals of
  // rv into hr); false when it gave up
  auto meet = [&](const double (&v)[R], bool halo, double& sum) -> bool {
    ++e;
    if (gang > 1 && halo) {
#pragma unroll
      for (int k = 0; k < R; ++k) rs[k * kSlab + t] = rv[k];
    }
    const double s = tree_sum<R>(v, sh_sum);
    if (gang == 1) {
      if (t == 0) sh_in[0] = s;
      __syncthreads();
      sum = sh_in[0];
      return true;
    }
    u64* slots = ra.sy.slots + (size_t)(e & 1) * kReplicas * ra.nwg * 2;
    if (t < kReplicas) post(slots + ((size_t)t * ra.nwg + wg) * 2, e, s);
    if (halo) {
      // (rs is complete: tree_sum's barrier)
      for (int i = t; i < nx; i += kSlab)
        post(ra.sy.xch + (size_t)(x0 + i) * kWords<T>, e, rs[ra.exp_loc[x0 + i]]);
    }
    bool ok = true;
    if (wave < 4) {
      double p = 0.0;
      if (t < gang)
        ok = await(slots + ((size_t)(wg & (kReplicas - 1)) * ra.nwg + g0 + t) * 2, e, p, dl);
      p = lane_tree(p, 1);
      if (lane == 0) sh_in[wave] = p;
    }
    if (halo) {
      // waves 4 and up first, so that the sums and most halos are read at once
      for (int h = (t + kSlab - 256) & (kSlab - 1); h < nh && ok; h += kSlab) {
        T v2;
        ok = await(ra.sy.xch + (size_t)ra.halo_src[h0 + h] * kWords<T>, e, v2, dl);
        if (ok) hr[h] = v2;
      }
    }
    if (!ok) sh_bad = 1;
    __syncthreads();
    if (sh_bad) {
      if (t == 0) {
        store_relaxed(ra.sy.abort, 1);
        store_relaxed(&st->gave_up, 1);
      }
      return false;
    }
    sum = (sh_in[0] + sh_in[1]) + (sh_in[2] + sh_in[3]);
    return true;
  };

  int status;
  for (;;) {
    // stop test (gracjg.F:306-324; strict for the initial residual, :219)
    if (m == 0 ? rr < thr : rr <= thr) {
      status = ST_CONVERGED;
      break;
    }
    // AD, D.AD
    double part[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      // (opaque, or the base addresses of all slabs are kept over the loop)
      int o = off[k];
      asm volatile("" : "+s"(o));
      const T s = slice_dot<T>(val + (size_t)o * 64, ra.ids + (size_t)o * 64, lane, wid[k], ds);
      const T d = ds[k * kSlab + t];
      ad[k] = s + (DQ ? dq[k] * d : d);
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
      part[k] = (have >> k & 1) ? (double)ds[k * kSlab + t] * (double)ad[k] : 0.0;
    double dad;
    if (!meet(part, false, dad)) return;
    // RO, X -= RO D (gracjg.F:380-388); after iteration NITMAX no more
    const double rho = rr / dad;
    const T rhot = (T)rho;
#pragma unroll
    for (int k = 0; k < R; ++k) xv[k] -= rhot * ds[k * kSlab + t];
    if (m >= nitmax) {
      status = ST_MAXITER;
      break;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
      rv[k] -= rhot * ad[k];
      part[k] = (have >> k & 1) ? (double)rv[k] * (double)rv[k] : 0.0;
    }
    rr_prev = rr;
    if (!meet(part, true, rr)) return;
    ++m;
    // D = R + BETA D, halo included
    const T beta = (T)(rr / rr_prev);
    if (!(rr <= thr)) {
#pragma unroll
      for (int k = 0; k < R; ++k) ds[k * kSlab + t] = rv[k] + beta * ds[k * kSlab + t];
      for (int h = (t + kSlab - 256) & (kSlab - 1); h < nh; h += kSlab)
        dh[h] = hr[h] + beta * dh[h];
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (have >> k & 1) {
      const int row = ra.slab_row0[k0 + k] + ra.rowpos[(size_t)(k0 + k) * kSlab + t];
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
// assembly: one wave per slice
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
k_rows_assemble(T* __restrict__ val, const double* __restrict__ xa,
                const int32_t* __restrict__ slice_off, const uint8_t* __restrict__ cnt,
                const int64_t* __restrict__ ref_off, const int32_t* __restrict__ refs,
                int nslice, unsigned lower) {
  // each XCD takes a contiguous range of slices: a block's coefficients are
  // read by the slices of its rows
  const int nb = gridDim.x;
  const int b = xcd_block(blockIdx.x, nb);
  const int q = b * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (q >= nslice) return;
  const int o0 = __builtin_amdgcn_readfirstlane(slice_off[q]);
  const int o1 = __builtin_amdgcn_readfirstlane(slice_off[q + 1]);
  const int32_t* r = refs + ref_off[q] * 64 + lane;
  for (int j = o0; j < o1; ++j) {
    const int c = __builtin_amdgcn_readfirstlane(cnt[j]);
    double s = 0.0;
    for (int i = 0; i < c; ++i, r += 64) {
      const int f = *r;
      if (f != -1) s += xa[(size_t)(f & 0x7fffffff) + (f < 0 ? lower : 0u)];
    }
    val[(size_t)j * 64 + lane] = (T)s;
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
  int nslab = 0, group = 1, nwg = 0, nsys = 1, max_halo = 0;
  int64_t nent = 0;
  int ncu = 0;
  Buf<int32_t> slab_row0, slice_off, refs, wg_slab0, wg_sys, sys_wg, halo_off, halo_row, halo_src,
      exp_off;
  Buf<uint16_t> rowpos, ids, exp_loc;
  Buf<uint8_t> cnt;
  Buf<int64_t> ref_off;
  Buf<double> v64;
  Buf<float> v32;
  Buf<u64> words;
  SyncWords sy[2];  // FP64, FP32
  int ep[2] = {0, 0};
};

static size_t cg_lds(const RowsDev& r, int bytes) {
  // D of own rows and halo, halo residuals, own residuals for the exchange
  return ((size_t)2 * r.group * kSlab + (size_t)2 * r.max_halo) * bytes;
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
  std::unique_ptr<RowsDev> r(new RowsDev());
  r->nslab = R.nslab;
  r->group = R.group;
  r->nwg = R.nwg;
  r->nsys = nsys;
  r->max_halo = R.max_halo;
  r->nent = R.nent;
  r->ncu = ncu;
  lds_max -= 4096;  // the kernels' static LDS: their sums
  if (cg_lds(*r, sizeof(double)) > (size_t)lds_max) return nullptr;
  bool fits = true;
  if ((*err = cg_fits<double>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if ((*err = cg_fits<float>(*r, lds_max, &fits)) != hipSuccess) return nullptr;
  if (!fits) return nullptr;
  auto ok = [&](hipError_t e) {
    if (e != hipSuccess) *err = e;
    return e == hipSuccess;
  };
  if (!ok(r->slab_row0.put(R.slab_row0, stream)) || !ok(r->slice_off.put(R.slice_off, stream)) ||
      !ok(r->refs.put(R.refs, stream)) || !ok(r->wg_slab0.put(R.wg_slab0, stream)) ||
      !ok(r->wg_sys.put(R.wg_sys, stream)) || !ok(r->sys_wg.put(R.sys_wg, stream)) ||
      !ok(r->halo_off.put(R.halo_off, stream)) || !ok(r->halo_row.put(R.halo_row, stream)) ||
      !ok(r->halo_src.put(R.halo_src, stream)) || !ok(r->exp_off.put(R.exp_off, stream)) ||
      !ok(r->rowpos.put(R.rowpos, stream)) || !ok(r->ids.put(R.ids, stream)) ||
      !ok(r->exp_loc.put(R.exp_loc, stream)) || !ok(r->cnt.put(R.cnt, stream)) ||
      !ok(r->ref_off.put(R.ref_off, stream)) || !ok(r->v64.alloc(R.nent)))
    return nullptr;
  // sync words: per precision sums and exchange, then the counters
  const size_t nslot = (size_t)2 * kReplicas * R.nwg * 2, nexp = R.exp_loc.size();
  const size_t nepoch = (2 * (size_t)nsys + 1) / 2 + 1;  // in 64-bit words
  const size_t one = nslot + 2 * nexp + nepoch + 2;
  if (!ok(r->words.alloc(2 * one))) return nullptr;
  u64 ticks = kWaitTicks;
  if (const char* ev = getenv("BHIP_ROWS_WAIT")) ticks = strtoull(ev, nullptr, 10);
  for (int k = 0; k < 2; ++k) {
    u64* p = r->words.p + k * one;
    r->sy[k].slots = p;
    r->sy[k].xch = p + nslot;
    r->sy[k].epoch = reinterpret_cast<unsigned*>(p + nslot + 2 * nexp);
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
  const int nslice = r->nslab * kSlices;
  const unsigned lower = nonsym ? (unsigned)npair * (unsigned)nslot_pad : 0u;
  const dim3 grid((nslice + 3) / 4), block(256);
  if (bytes == 8)
    hipLaunchKernelGGL(k_rows_assemble<double>, grid, block, 0, stream, r->v64.p, xa,
                       r->slice_off.p, r->cnt.p, r->ref_off.p, r->refs.p, nslice, lower);
  else
    hipLaunchKernelGGL(k_rows_assemble<float>, grid, block, 0, stream, r->v32.p, xa,
                       r->slice_off.p, r->cnt.p, r->ref_off.p, r->refs.p, nslice, lower);
  return hipGetLastError();
}

static RowArgs row_args(const RowsDev* r, int k) {
  RowArgs a;
  a.slice_off = r->slice_off.p;
  a.ids = r->ids.p;
  a.rowpos = r->rowpos.p;
  a.slab_row0 = r->slab_row0.p;
  a.wg_slab0 = r->wg_slab0.p;
  a.wg_sys = r->wg_sys.p;
  a.sys_wg = r->sys_wg.p;
  a.halo_off = r->halo_off.p;
  a.halo_row = r->halo_row.p;
  a.halo_src = r->halo_src.p;
  a.exp_off = r->exp_off.p;
  a.exp_loc = r->exp_loc.p;
  a.nwg = r->nwg;
  a.nsys = r->nsys;
  a.nslab = r->nslab;
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
