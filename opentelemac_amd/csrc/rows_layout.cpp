// Host-side construction of the assembled row storage (see rows.h).
#include "rows.h"

#include <algorithm>
#include <atomic>
#include <functional>
#include <thread>

namespace bhip {

namespace {

// f(i) for i in [0, n) on a few host threads, each with its own scratch from
// make()
template <typename Make, typename F>
void parallel_for(int n, Make make, F f) {
  const int hw = (int)std::thread::hardware_concurrency();
  const int nt = std::max(1, std::min({hw, 8, n / 16}));
  std::atomic<int> next{0};
  auto work = [&]() {
    auto scratch = make();
    for (int i; (i = next.fetch_add(1)) < n;) f(i, scratch);
  };
  std::vector<std::thread> pool;
  for (int t = 1; t < nt; ++t) pool.emplace_back(work);
  work();
  for (auto& t : pool) t.join();
}

struct Contribution {
  int32_t col, ref;
};
struct Entry {
  int32_t col, first, count;
};
struct SlabScratch {
  std::vector<int32_t> off, fill;
  std::vector<Contribution> con;
  std::vector<std::vector<Entry>> rows;
  std::vector<int> order;
};
// one slab's slices before they are joined
struct SlabOut {
  std::vector<int32_t> width;  // per slice
  std::vector<int32_t> cols;   // per entry (internal node id)
  std::vector<uint8_t> cnt;
  std::vector<int32_t> refs, ref_units;  // per slice: 64-wide reference columns
};

}  // namespace

bool build_rows(const Layout& L, int nsys, const int64_t* node_off, int max_wg, RowLayout& R) {
  R = RowLayout();
  const int ndp = L.ndp;
  const int cap = std::min(max_wg, kMaxGang);
  if (cap < 1) return false;
  // references hold pair * nslot_pad + slot in 31 bits
  if ((int64_t)ndp * (ndp - 1) / 2 * L.nslot_pad >= INT32_MAX) return false;
  // slabs
  std::vector<int32_t> sys_slab(nsys + 1, 0);
  for (int s = 0; s < nsys; ++s) {
    const int64_t n = node_off[s + 1] - node_off[s];
    const int64_t ns = (n + kSlab - 1) / kSlab;
    if (ns > (int64_t)cap * kMaxGroup) return false;
    for (int64_t k = 0; k < ns; ++k) {
      R.slab_row0.push_back((int32_t)(node_off[s] + k * kSlab));
      R.slab_rows.push_back((int32_t)std::min<int64_t>(kSlab, n - k * kSlab));
    }
    sys_slab[s + 1] = (int32_t)R.slab_row0.size();
  }
  R.nslab = (int)R.slab_row0.size();
  // slabs per workgroup: the fewest that let every system be resident at
  // once, or (many systems) as many as a workgroup can hold
  auto wgs = [&](int g) {
    int64_t t = 0;
    for (int s = 0; s < nsys; ++s) t += (sys_slab[s + 1] - sys_slab[s] + g - 1) / g;
    return t;
  };
  R.group = 1;
  while (R.group < kMaxGroup && wgs(R.group) > cap) R.group *= 2;
  R.sys_wg.assign(1, 0);
  for (int s = 0; s < nsys; ++s) {
    for (int k = sys_slab[s]; k < sys_slab[s + 1]; k += R.group) {
      R.wg_slab0.push_back(k);
      R.wg_sys.push_back(s);
    }
    R.sys_wg.push_back((int32_t)R.wg_sys.size());
    R.max_gang = std::max(R.max_gang, R.sys_wg[s + 1] - R.sys_wg[s]);
  }
  R.nwg = (int)R.wg_sys.size();
  R.wg_slab0.push_back(R.nslab);

  // ---- rows of each slab ---------------------------------------------------
  std::vector<SlabOut> out(R.nslab);
  R.rowpos.assign((size_t)R.nslab * kSlab, 0xffff);
  std::vector<uint16_t> pos_of((size_t)L.npoin);  // position of a row in its slab
  int pair_idx[6][6];
  for (int i = 0, q = 0; i < ndp; ++i)
    for (int j = i + 1; j < ndp; ++j, ++q) pair_idx[i][j] = pair_idx[j][i] = q;
  parallel_for(R.nslab, [] { return SlabScratch(); }, [&](int k, SlabScratch& w) {
    const int r0 = R.slab_row0[k], nr = R.slab_rows[k], r1 = r0 + nr;
    const int b0 = (int)(std::upper_bound(L.node_start.begin(), L.node_start.end(), r0) -
                         L.node_start.begin()) - 1;
    // every (row, column, coefficient) of the blocks that own these rows, in
    // slot order: counted, then filled
    auto visit = [&](auto&& f) {
      for (int b = b0; b < L.nblocks && L.node_start[b] < r1; ++b) {
        const int n0 = L.node_start[b], nown = L.node_start[b + 1] - n0, h0 = L.halo_start[b];
        const int32_t* co = &L.color_off[(size_t)b * (kMaxColors + 1)];
        for (int s = co[0]; s < co[kMaxColors]; ++s) {
          int g[6];
          for (int a = 0; a < ndp; ++a) {
            const int l = L.lid[(size_t)a * L.nslot_pad + s];
            g[a] = l < nown ? n0 + l : L.halo[h0 + l - nown];
          }
          for (int a = 0; a < ndp; ++a) {
            // rows this block owns (a halo node's row belongs to another block)
            if (g[a] < r0 || g[a] >= r1 || g[a] < n0 || g[a] >= n0 + nown) continue;
            f(s, a, g);
          }
        }
      }
    };
    w.off.assign(nr + 1, 0);
    visit([&](int, int a, const int* g) { w.off[g[a] - r0 + 1] += ndp - 1; });
    for (int i = 0; i < nr; ++i) w.off[i + 1] += w.off[i];
    w.con.resize(w.off[nr]);
    w.fill.assign(w.off.begin(), w.off.end() - 1);
    visit([&](int s, int a, const int* g) {
      for (int j = 0; j < ndp; ++j) {
        if (j == a) continue;
        const uint32_t ref = (uint32_t)pair_idx[a][j] * (uint32_t)L.nslot_pad + (uint32_t)s;
        w.con[w.fill[g[a] - r0]++] = {g[j], (int32_t)(ref | (a > j ? 0x80000000u : 0u))};
      }
    });
    w.rows.resize(kSlab);
    w.order.resize(nr);
    for (int i = 0; i < nr; ++i) {
      auto first = w.con.begin() + w.off[i], last = w.con.begin() + w.off[i + 1];
      std::stable_sort(first, last,
                       [](const Contribution& p, const Contribution& q) { return p.col < q.col; });
      auto& e = w.rows[i];
      e.clear();
      for (auto it = first; it != last; ++it) {
        if (e.empty() || e.back().col != it->col)
          e.push_back({it->col, (int32_t)(it - w.con.begin()), 0});
        e.back().count++;
      }
      // entries with many contributions first, so that the lanes of a slice
      // agree on the count of each entry column
      std::stable_sort(e.begin(), e.end(),
                       [](const Entry& p, const Entry& q) { return p.count > q.count; });
      w.order[i] = i;
    }
    std::stable_sort(w.order.begin(), w.order.end(),
                     [&](int p, int q) { return w.rows[p].size() > w.rows[q].size(); });
    SlabOut& o = out[k];
    o.width.assign(kSlices, 0);
    o.ref_units.assign(kSlices, 0);
    for (int p = 0; p < nr; ++p) {
      R.rowpos[(size_t)k * kSlab + p] = (uint16_t)w.order[p];
      pos_of[r0 + w.order[p]] = (uint16_t)p;
    }
    for (int q = 0; q < kSlices; ++q) {
      const int p0 = q * 64, p1 = std::min(nr, p0 + 64);
      int width = 0;
      for (int p = p0; p < p1; ++p) width = std::max(width, (int)w.rows[w.order[p]].size());
      o.width[q] = width;
      for (int j = 0; j < width; ++j) {
        int c = 0;
        for (int p = p0; p < p1; ++p) {
          const auto& e = w.rows[w.order[p]];
          if (j < (int)e.size()) c = std::max(c, e[j].count);
        }
        o.cnt.push_back((uint8_t)std::min(c, 255));
        o.ref_units[q] += c;
        const size_t base = o.refs.size(), cb = o.cols.size();
        o.refs.resize(base + (size_t)c * 64, -1);
        o.cols.resize(cb + 64, -1);
        for (int p = p0; p < p1; ++p) {
          const auto& e = w.rows[w.order[p]];
          // padding names the row itself (its coefficient stays 0)
          o.cols[cb + p - p0] = j < (int)e.size() ? e[j].col : r0 + w.order[p];
          for (int t = 0; j < (int)e.size() && t < e[j].count; ++t)
            o.refs[base + (size_t)t * 64 + p - p0] = w.con[e[j].first + t].ref;
        }
      }
    }
  });
  // ---- joined --------------------------------------------------------------
  R.slice_off.assign((size_t)R.nslab * kSlices + 1, 0);
  R.ref_off.assign((size_t)R.nslab * kSlices, 0);
  int64_t units = 0, runits = 0;
  for (int k = 0; k < R.nslab; ++k)
    for (int q = 0; q < kSlices; ++q) {
      const size_t i = (size_t)k * kSlices + q;
      R.ref_off[i] = runits;
      units += out[k].width[q];
      runits += out[k].ref_units[q];
      R.slice_off[i + 1] = (int32_t)units;
      for (int j = 0; j < out[k].width[q]; ++j)
        if (units > INT32_MAX / 64) {
          R = RowLayout();
          return false;
        }
    }
  R.nent = units * 64;
  R.nref = runits * 64;
  for (const auto& o : out)
    for (uint8_t c : o.cnt)
      if (c == 255) {  // a pair shared by 255 elements: not a mesh this storage is for
        R = RowLayout();
        return false;
      }
  R.ids.resize(R.nent);
  R.refs.resize(R.nref);
  R.cnt.resize(units);
  // ---- workgroups: halo, then local ids ---------------------------------------
  struct Marks {
    std::vector<int32_t> wg, idx;
  };
  std::vector<std::vector<int32_t>> halo(R.nwg);
  std::atomic<bool> fits{true};
  parallel_for(R.nwg, [&] { return Marks{std::vector<int32_t>(L.npoin, -1),
                                         std::vector<int32_t>(L.npoin, 0)}; },
               [&](int g, Marks& m) {
    const int k0 = R.wg_slab0[g], k1 = R.wg_slab0[g + 1];
    const int r0 = R.slab_row0[k0], r1 = R.slab_row0[k1 - 1] + R.slab_rows[k1 - 1];
    auto& h = halo[g];
    for (int k = k0; k < k1; ++k)
      for (int c : out[k].cols)
        if (c >= 0 && (c < r0 || c >= r1) && m.wg[c] != g) {
          m.wg[c] = g;
          h.push_back(c);
        }
    std::sort(h.begin(), h.end());
    for (size_t i = 0; i < h.size(); ++i) m.idx[h[i]] = (int32_t)i;
    if (R.group * kSlab + h.size() > 65535) fits = false;
    for (int k = k0; k < k1; ++k) {
      const int64_t e0 = (int64_t)R.slice_off[(size_t)k * kSlices] * 64;
      const auto& cols = out[k].cols;
      for (size_t i = 0; i < cols.size(); ++i) {
        const int c = cols[i];
        int id = 0;  // a lane without a row: any index, its coefficient is 0
        if (c >= r0 && c < r1)
          id = (c - r0) / kSlab * kSlab + pos_of[c];
        else if (c >= 0)
          id = R.group * kSlab + m.idx[c];
        R.ids[e0 + i] = (uint16_t)id;
      }
      std::copy(out[k].refs.begin(), out[k].refs.end(),
                R.refs.begin() + R.ref_off[(size_t)k * kSlices] * 64);
      std::copy(out[k].cnt.begin(), out[k].cnt.end(), R.cnt.begin() + e0 / 64);
    }
  });
  if (!fits) {
    R = RowLayout();
    return false;
  }
  // ---- exported rows ---------------------------------------------------------
  std::vector<int32_t> rank(L.npoin, -1);
  for (const auto& h : halo)
    for (int c : h) rank[c] = 0;
  R.exp_off.assign(1, 0);
  for (int g = 0; g < R.nwg; ++g) {
    for (int k = R.wg_slab0[g]; k < R.wg_slab0[g + 1]; ++k)
      for (int p = 0; p < R.slab_rows[k]; ++p) {
        const int row = R.slab_row0[k] + R.rowpos[(size_t)k * kSlab + p];
        if (rank[row] < 0) continue;
        rank[row] = (int32_t)R.exp_loc.size();
        R.exp_loc.push_back((uint16_t)((k - R.wg_slab0[g]) * kSlab + p));
      }
    R.exp_off.push_back((int32_t)R.exp_loc.size());
  }
  R.halo_off.assign(1, 0);
  for (int g = 0; g < R.nwg; ++g) {
    for (int c : halo[g]) {
      R.halo_row.push_back(c);
      R.halo_src.push_back(rank[c]);
    }
    R.halo_off.push_back((int32_t)R.halo_row.size());
    R.max_halo = std::max(R.max_halo, (int)halo[g].size());
  }
  return true;
}

}  // namespace bhip
