// Host-side construction of the assembled row storage (see rows.h).
#include "rows.h"

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>

namespace bhip {

namespace {

// f(i) for i in [0, n) on a few host threads, each with its own scratch from
// make(). An exception of any of them is thrown here, once all have ended; where
// no (more) threads can be started, those that are there do the work.
template <typename Make, typename F>
void parallel_for(int n, Make make, F f) {
  const int hw = (int)std::thread::hardware_concurrency();
  const int nt = std::max(1, std::min({hw, 8, n / 2}));
  std::atomic<int> next{0};
  std::exception_ptr failed;
  std::mutex mu;
  auto work = [&]() {
    try {
      auto scratch = make();
      for (int i; (i = next.fetch_add(1)) < n;) f(i, scratch);
    } catch (...) {
      std::lock_guard<std::mutex> one(mu);
      failed = std::current_exception();
      next = n;
    }
  };
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < nt; ++t) pool.emplace_back(work);
  } catch (...) {
  }
  work();
  for (auto& t : pool) t.join();
  if (failed) std::rethrow_exception(failed);
}

struct Contribution {
  int32_t col, ref;
};
struct Entry {
  int32_t col, first, count;
};
struct Scratch {
  std::vector<int32_t> off, fill, order, row_at;
  std::vector<Contribution> con;
  std::vector<std::vector<Entry>> rows;
  std::vector<int32_t> mark;  // per row: the last workgroup that saw it
};
// one workgroup's slices before they are joined
struct WgOut {
  std::vector<int32_t> width;  // per slice
  std::vector<int32_t> cols;   // per entry (internal node id, -1: none)
  std::vector<uint8_t> ref_end;
  std::vector<int32_t> refs, ref_cols;  // per slice: reference columns
  std::vector<int32_t> halo;
};

}  // namespace

bool build_rows(const Layout& L, int nsys, const int64_t* node_off, int max_wg, size_t max_lds,
                RowLayout& R) {
  R = RowLayout();
  const int ndp = L.ndp;
  const int cap = std::min(max_wg, kMaxGang);
  if (cap < 1) return false;
  // references hold pair * nslot_pad + slot in 31 bits
  if ((int64_t)ndp * (ndp - 1) / 2 * L.nslot_pad >= INT32_MAX) return false;
  std::vector<int64_t> slabs(nsys);
  for (int s = 0; s < nsys; ++s) {
    slabs[s] = (node_off[s + 1] - node_off[s] + kSlab - 1) / kSlab;
    if (slabs[s] > (int64_t)cap * kMaxGroup) return false;
  }
  // slabs per workgroup: the fewest that let every system be resident at once,
  // or (many systems) more while that saves a fifth of the workgroups: one with
  // empty slabs costs a round on its CU like any other, and more of a thread's
  // rows mean fewer coefficients in its registers. us per solve, FP64 / mixed,
  // with 1, 2, 4, 8 slabs: 2,000 systems of 500 nodes 326/423, 383/519, 606/823,
  // 868/1336; 300 of 2,000 nodes 212/254, 140/183, 201/241, 289/334; 256 of 5k to
  // 200k nodes -, 3936/5246, 3835/4056, 3665/3925. Two instead of one already
  // past half of the workgroups: a meeting of 256 workgroups takes 1 us longer
  // than one of 128, a second slab kept in registers less
  auto wgs = [&](int g) {
    int64_t t = 0;
    for (int s = 0; s < nsys; ++s) t += (slabs[s] + g - 1) / g;
    return t;
  };
  const int64_t widest = *std::max_element(slabs.begin(), slabs.end());
  auto wants_more = [&](int g) {
    if (widest > (int64_t)cap * g) return true;
    return wgs(g) > (g == 1 ? cap / 2 : cap) && 5 * wgs(2 * g) <= 4 * wgs(g);
  };
  R.group = 1;
  while (R.group < kMaxGroup && wants_more(R.group)) R.group *= 2;
  const int G = R.group, wrows = G * kSlab;
  // slabs and node blocks are the same rows when both start anew with each
  // system and hold kSlab of them
  auto block_slots = [&](int b) {
    const int32_t* co = &L.color_off[(size_t)b * (kMaxColors + 1)];
    return co[kMaxColors] - co[0];
  };
  for (int b = 0; b < L.nblocks; ++b) R.max_slots = std::max(R.max_slots, block_slots(b));
  R.by_block = ndp <= 3 && L.block_nodes == kSlab &&
               R.max_slots * (ndp * (ndp - 1) / 2) < 0x7fff &&
               // k_dmd_rows keeps a block's coefficients and D in LDS
               ((size_t)ndp * (ndp - 1) * R.max_slots + L.max_local + 1) * 8 <= kSlabLds;
  R.sys_wg.assign(1, 0);
  std::vector<int32_t> nrows;  // of each workgroup
  for (int s = 0; s < nsys; ++s) {
    for (int64_t k = 0; k < slabs[s]; k += G) {
      const int64_t r0 = node_off[s] + k * kSlab;
      R.wg_row0.push_back((int32_t)r0);
      nrows.push_back((int32_t)std::min<int64_t>(wrows, node_off[s + 1] - r0));
      R.wg_sys.push_back(s);
    }
    R.sys_wg.push_back((int32_t)R.wg_sys.size());
    R.max_gang = std::max(R.max_gang, R.sys_wg[s + 1] - R.sys_wg[s]);
  }
  R.nwg = (int)R.wg_sys.size();
  R.launch.assign(1, 0);
  if (R.nwg > max_wg && R.max_gang > max_wg / kXcds)
    for (int s = 0; s < nsys; ++s)
      if (R.sys_wg[s + 1] - R.launch.back() > max_wg) R.launch.push_back(R.sys_wg[s]);
  R.launch.push_back(R.nwg);
  const int wslices = G * kSlices;  // slices of a workgroup
  R.nslice = R.nwg * wslices;

  // ---- rows of each workgroup ------------------------------------------------
  std::vector<WgOut> out(R.nwg);
  R.rowpos.assign((size_t)R.nwg * wrows, 0xffff);
  std::vector<uint16_t> lid_of((size_t)L.npoin);  // LDS index of a row in its workgroup
  int pair_idx[6][6];
  for (int i = 0, q = 0; i < ndp; ++i)
    for (int j = i + 1; j < ndp; ++j, ++q) pair_idx[i][j] = pair_idx[j][i] = q;
  auto fits = [&](size_t nh) {
    return wrows + nh <= 65535 && cg_lds(G, nh, 8) <= max_lds && cg_lds(G, nh, 4) <= max_lds;
  };
  std::atomic<bool> refused{false};  // by one of them: the others are not wanted
  parallel_for(R.nwg, [] { return Scratch(); }, [&](int wg, Scratch& w) {
    if (refused) return;
    const int r0 = R.wg_row0[wg], nr = nrows[wg], r1 = r0 + nr;
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
    w.rows.resize(wrows);
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
    }
    // leaves, half a slab at a time; row_at[LDS index]
    w.row_at.assign(wrows, -1);
    static const int kRun[8] = {0, 4, 1, 5, 2, 6, 3, 7};
    constexpr int kHalf = kSlab / 2;
    static_assert(kHalf == 8 * 64, "eight runs of 64 ranks");
    for (int h = 0; h < nr; h += kHalf) {
      const int n = std::min(kHalf, nr - h);
      w.order.resize(n);
      for (int i = 0; i < n; ++i) w.order[i] = h + i;
      std::stable_sort(w.order.begin(), w.order.end(),
                       [&](int p, int q) { return w.rows[p].size() > w.rows[q].size(); });
      for (int i = 0; i < n; ++i) {
        const int leaf = h + 8 * (i % 64) + kRun[i / 64];
        const int id = leaf % G * kSlab + leaf / G;
        w.row_at[id] = w.order[i];
        lid_of[r0 + w.order[i]] = (uint16_t)id;
      }
    }
    for (int id = 0; id < wrows; ++id)
      if (w.row_at[id] >= 0) R.rowpos[(size_t)wg * wrows + id] = (uint16_t)w.row_at[id];
    WgOut& o = out[wg];
    o.width.assign(wslices, 0);
    o.ref_cols.assign(wslices, 0);
    for (int q = 0; q < wslices; ++q) {
      const int32_t* at = &w.row_at[(size_t)q * 64];  // (k * kSlab + wave * 64)
      int width = 0;
      for (int l = 0; l < 64; ++l)
        if (at[l] >= 0) width = std::max(width, (int)w.rows[at[l]].size());
      o.width[q] = width;
      for (int j = 0; j < width; ++j) {
        int c = 0;
        for (int l = 0; l < 64; ++l)
          if (at[l] >= 0 && j < (int)w.rows[at[l]].size())
            c = std::max(c, w.rows[at[l]][j].count);
        for (int t = 0; t < c; ++t) {
          const int col = o.ref_cols[q]++;
          if (col % kRefChunk == 0) o.ref_end.push_back(0);
          if (t == c - 1) o.ref_end.back() |= (uint8_t)(1 << col % kRefChunk);
        }
        const size_t base = o.refs.size(), cb = o.cols.size();
        o.refs.resize(base + (size_t)c * 64, -1);
        o.cols.resize(cb + 64, -1);
        for (int l = 0; l < 64; ++l) {
          if (at[l] < 0) continue;
          const auto& e = w.rows[at[l]];
          // padding names the row itself (its coefficient stays 0)
          o.cols[cb + l] = j < (int)e.size() ? e[j].col : r0 + at[l];
          for (int t = 0; j < (int)e.size() && t < e[j].count; ++t)
            o.refs[base + (size_t)t * 64 + l] = w.con[e[j].first + t].ref;
        }
      }
      o.ref_cols[q] = (o.ref_cols[q] + kRefChunk - 1) / kRefChunk * kRefChunk;
      size_t total = 0;
      for (int i = 0; i <= q; ++i) total += o.ref_cols[i];
      o.refs.resize(total * 64, -1);
    }
    // halo: the other workgroups' rows these entries name, by row
    if (w.mark.empty()) w.mark.assign(L.npoin, -1);
    for (int c : o.cols)
      if (c >= 0 && (c < r0 || c >= r1) && w.mark[c] != wg) {
        w.mark[c] = wg;
        o.halo.push_back(c);
      }
    std::sort(o.halo.begin(), o.halo.end());
    if (!fits(o.halo.size())) refused = true;
  });
  if (refused) {
    R = RowLayout();
    return false;
  }
  for (const auto& o : out) R.max_halo = std::max(R.max_halo, (int)o.halo.size());
  // ---- joined --------------------------------------------------------------
  R.slice_off.assign(R.nslice + 1, 0);
  R.pair_off.assign(R.nslice + 1, 0);
  R.ref_off.assign(R.nslice + 1, 0);
  int64_t units = 0, runits = 0;
  for (int g = 0; g < R.nwg; ++g)
    for (int q = 0; q < wslices; ++q) {
      const size_t i = (size_t)g * wslices + q;
      units += out[g].width[q];
      runits += out[g].ref_cols[q];
      if (runits > INT32_MAX || units > INT32_MAX / 128) {
        R = RowLayout();
        return false;
      }
      R.ref_off[i + 1] = (int32_t)runits;
      R.slice_off[i + 1] = (int32_t)units;
      // (an id word per lane for an empty slice too: load_front reads one, and
      // the next slice's would name another workgroup's halo)
      R.pair_off[i + 1] = R.pair_off[i] + std::max((out[g].width[q] + 1) / 2, 1);
    }
  R.nent = units * 64;
  R.nref = runits * 64;
  R.ids.assign((size_t)R.pair_off.back() * 128, 0);
  if (!R.by_block) R.refs.resize(R.nref);
  R.ref_end.resize(runits / kRefChunk);
  if (R.by_block) R.refs16.resize(R.nref);
  parallel_for(R.nwg, [] { return 0; }, [&](int g, int&) {
    const int r0 = R.wg_row0[g], r1 = r0 + nrows[g];
    const WgOut& o = out[g];
    const size_t q0 = (size_t)g * wslices;
    size_t i = 0;
    for (int q = 0; q < wslices; ++q) {
      uint16_t* id = R.ids.data() + (size_t)R.pair_off[q0 + q] * 128;
      for (int j = 0; j < o.width[q]; ++j)
        for (int l = 0; l < 64; ++l, ++i) {
          const int c = o.cols[i];
          int v = 0;  // a lane without a row: any index, its coefficient is 0
          if (c >= r0 && c < r1)
            v = lid_of[c];
          else if (c >= 0)
            v = wrows + (int)(std::lower_bound(o.halo.begin(), o.halo.end(), c) - o.halo.begin());
          id[((size_t)(j / 2) * 64 + l) * 2 + (j & 1)] = (uint16_t)v;
        }
    }
    if (R.by_block) {
      // slice by slice: its rows lie in one slab, so in one block
      size_t i = 0;
      for (int q = 0; q < wslices; ++q) {
        const int leaf = q % kSlices * 64 * G;  // first leaf of the slice's first lane
        const int row = r0 + leaf / kSlab * kSlab;
        const int b = (int)(std::upper_bound(L.node_start.begin(), L.node_start.end(), row) -
                            L.node_start.begin()) - 1;
        const int s0 = b < L.nblocks ? L.color_off[(size_t)b * (kMaxColors + 1)] : 0;
        const int ns = b < L.nblocks ? block_slots(b) : 1;
        uint16_t* to = R.refs16.data() + (size_t)R.ref_off[q0 + q] * 64;
        for (int c = 0; c < o.ref_cols[q] * 64; ++c, ++i) {
          const uint32_t f = (uint32_t)o.refs[i], low = f & 0x7fffffffu;
          to[c] = o.refs[i] == -1 ? 0xffff
                                  : (uint16_t)((f >> 31 << 15) | (low / L.nslot_pad * ns +
                                                                  low % L.nslot_pad - s0));
        }
      }
    } else {
      std::copy(o.refs.begin(), o.refs.end(), R.refs.begin() + (size_t)R.ref_off[q0] * 64);
    }
    std::copy(o.ref_end.begin(), o.ref_end.end(), R.ref_end.begin() + R.ref_off[q0] / kRefChunk);
  });
  std::vector<std::vector<int32_t>> halo(R.nwg);
  for (int g = 0; g < R.nwg; ++g) halo[g] = std::move(out[g].halo);
  // ---- exported rows ---------------------------------------------------------
  std::vector<int32_t> rank(L.npoin, -1);
  for (const auto& h : halo)
    for (int c : h) rank[c] = 0;
  R.exp_off.assign(1, 0);
  for (int g = 0; g < R.nwg; ++g) {
    for (int id = 0; id < wrows; ++id) {
      const int at = R.rowpos[(size_t)g * wrows + id];
      if (at == 0xffff || rank[R.wg_row0[g] + at] < 0) continue;
      rank[R.wg_row0[g] + at] = (int32_t)R.exp_loc.size();
      R.exp_loc.push_back((uint16_t)id);
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
  }
  return true;
}

}  // namespace bhip
