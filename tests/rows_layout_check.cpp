// Host-side check of the assembled row storage: prints "ok" or what is wrong.
// Arguments: workgroups that fit, nodes per block, then per system its nodes (in
// segment storage, a chain of neighbours, or `far`: two halves joined only with
// each other). CHECK_FAIL in the environment: "threads", no thread can be
// started; "memory=<n>", the n-th allocation of build_rows fails (and "bad_alloc"
// is printed). CHECK_PRINT: the slabs per workgroup are printed, nothing else.
#include "rows.h"

#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <random>

using namespace bhip;

static bool no_threads = false;
static std::atomic<long> allocations_left{-1};  // negative: no limit

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* p) {
  typedef int (*Real)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Real real = (Real)dlsym(RTLD_NEXT, "pthread_create");
  return no_threads ? EAGAIN : real(t, a, f, p);
}
void* operator new(size_t n) {
  if (allocations_left >= 0 && allocations_left-- == 0) throw std::bad_alloc();
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
// (std::stable_sort does without its buffer)
void* operator new(size_t n, const std::nothrow_t&) noexcept { return malloc(n ? n : 1); }
void operator delete(void* p, const std::nothrow_t&) noexcept { free(p); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static int wrong(const char* what, int at) {
  printf("%s (%d)\n", what, at);
  return 1;
}

int main(int argc, char** argv) {
  const size_t max_lds = 158 << 10;
  const int max_wg = atoi(argv[1]), block_nodes = atoi(argv[2]);
  std::vector<int> np, ne;
  std::vector<int32_t> ikle;
  std::vector<double> x, y;
  for (int a = 3; a < argc; ++a) {
    const bool far = strncmp(argv[a], "far", 3) == 0;
    const int n = atoi(argv[a] + (far ? 3 : 0)), h = n / 2;
    std::vector<int32_t> p, q;
    for (int i = 0; i < n; ++i) {
      const int k = far ? i % h : i;
      x.push_back((far && i >= h ? 1e5 : 0.0) + k % 32);
      y.push_back((far && i >= h ? 1e5 : 0.0) + k / 32);
    }
    if (far)
      for (int d = 0; d < 2; ++d)
        for (int i = 0; i < h; ++i) {
          p.push_back(i);
          q.push_back(h + (i + 7 * d) % h);
        }
    else
      for (int i = 0; i + 1 < n; ++i) {
        p.push_back(i);
        q.push_back(i + 1);
      }
    np.push_back(n);
    ne.push_back((int)p.size());
    ikle.insert(ikle.end(), p.begin(), p.end());
    ikle.insert(ikle.end(), q.begin(), q.end());
  }
  const int nsys = (int)np.size();
  Layout L;
  std::vector<int32_t> blocks, all;
  const std::string err = build_layout_multi(nsys, np.data(), ne.data(), 2, ikle.data(), x.data(),
                                             y.data(), block_nodes, L, blocks, all);
  if (!err.empty()) return wrong(err.c_str(), 0);
  std::vector<int64_t> off(1, 0);
  for (int n : np) off.push_back(off.back() + n);
  RowLayout R;
  if (const char* f = getenv("CHECK_FAIL")) {
    no_threads = strcmp(f, "threads") == 0;
    if (strncmp(f, "memory=", 7) == 0) {
      allocations_left = atol(f + 7);
      try {
        const bool built = build_rows(L, nsys, off.data(), max_wg, max_lds, R);
        allocations_left = -1;
        printf("%s\n", built ? "built" : "no rows");
      } catch (const std::bad_alloc&) {
        allocations_left = -1;
        printf("bad_alloc\n");
      }
      return 0;
    }
  }
  if (!build_rows(L, nsys, off.data(), max_wg, max_lds, R)) return wrong("no rows", 0);
  if (cg_lds(R.group, R.max_halo, 8) > max_lds || cg_lds(R.group, R.max_halo, 4) > max_lds)
    return wrong("more LDS than there is", R.max_halo);
  if (getenv("CHECK_PRINT")) return printf("%d\n", R.group) < 0;
  // launches: whole systems; one of more workgroups than fit has systems of at
  // most an XCD's share (an eighth)
  if (R.launch.front() != 0 || R.launch.back() != R.nwg) return wrong("launches", 0);
  for (size_t i = 0; i + 1 < R.launch.size(); ++i) {
    const int a = R.launch[i], b = R.launch[i + 1];
    if (a >= b) return wrong("empty launch", (int)i);
    if (a > 0 && R.wg_sys[a] == R.wg_sys[a - 1]) return wrong("system cut", (int)i);
    for (int g = a; b - a > max_wg && g < b; ++g)
      if (R.sys_wg[R.wg_sys[g] + 1] - R.sys_wg[R.wg_sys[g]] > max_wg / 8)
        return wrong("system wider than an XCD's share", R.wg_sys[g]);
  }
  const int wrows = R.group * kSlab;
  // every id that the kernels read, a slice's and those load_front reads of a
  // short or empty one, names D of the workgroup's own rows or halo
  for (int q = 0; q < R.nslice; ++q) {
    const int wg = q / (R.group * kSlices), nh = R.halo_off[wg + 1] - R.halo_off[wg];
    const int w = R.slice_off[q + 1] - R.slice_off[q];
    if (R.pair_off[q + 1] - R.pair_off[q] < (w + 1) / 2) return wrong("id words", q);
    for (int j = 0; j < std::max((w + 1) / 2, 1); ++j)
      for (int l = 0; l < 128; ++l) {
        const size_t i = (size_t)(R.pair_off[q] + j) * 128 + l;
        if (i >= R.ids.size()) return wrong("id past the end", q);
        if (R.ids[i] >= wrows + nh) return wrong("id beyond D and its halo", q);
      }
  }
  // a product by rows against one by segments (coefficients by caller element)
  std::mt19937 rng(1);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  std::vector<double> c(L.nelem), v(L.npoin), want(L.npoin, 0.0), xa(L.nslot_pad, 0.0);
  for (double& t : c) t = u(rng);
  for (double& t : v) t = u(rng);
  for (int e = 0; e < L.nelem; ++e) {
    const int i = L.iperm[all[e]], j = L.iperm[all[L.nelem + e]];
    want[i] += c[e] * v[j];
    want[j] += c[e] * v[i];
  }
  for (int s = 0; s < L.nslot; ++s) xa[s] = c[L.slot_elem[s]];
  for (int q = 0; q < R.nslice; ++q) {
    const int wg = q / (R.group * kSlices), r0 = R.wg_row0[wg];
    const uint16_t* rowpos = &R.rowpos[(size_t)wg * wrows];
    std::vector<double> s(64, 0.0), e(64, 0.0);
    int entry = 0;
    for (int k = R.ref_off[q]; k < R.ref_off[q + 1]; ++k) {
      for (int l = 0; l < 64; ++l) {
        int ref;
        if (R.by_block) {
          const int slab = q % (R.group * kSlices) % kSlices * 64 * R.group / kSlab;
          int b = 0;
          while (L.node_start[b + 1] <= r0 + slab * kSlab) ++b;
          const uint16_t f = R.refs16[(size_t)k * 64 + l];
          ref = f == 0xffff ? -1 : (f & 0x7fff) + L.color_off[(size_t)b * (kMaxColors + 1)];
        } else {
          const int32_t f = R.refs[(size_t)k * 64 + l];
          ref = f == -1 ? -1 : f & 0x7fffffff;
        }
        if (ref >= 0) e[l] += xa[ref];
      }
      if (R.ref_end[k / kRefChunk] >> k % kRefChunk & 1) {
        for (int l = 0; l < 64; ++l) {
          const int id = R.ids[((size_t)(R.pair_off[q] + entry / 2) * 64 + l) * 2 + (entry & 1)];
          const int row = id < wrows ? r0 + rowpos[id] : R.halo_row[R.halo_off[wg] + id - wrows];
          if (e[l] != 0.0) s[l] += e[l] * v[row];
          e[l] = 0.0;
        }
        ++entry;
      }
    }
    if (entry != R.slice_off[q + 1] - R.slice_off[q]) return wrong("entries", q);
    for (int l = 0; l < 64; ++l) {
      const int at = rowpos[q % (R.group * kSlices) * 64 + l];
      if (at == 0xffff) continue;
      double& t = want[r0 + at];
      if (!(std::abs(t - s[l]) < 1e-13)) return wrong("product", r0 + at);
      t = s[l];
    }
  }
  printf("ok\n");
  return 0;
}
