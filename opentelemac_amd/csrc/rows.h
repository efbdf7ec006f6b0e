// Assembled row storage of an EBE (or segment) matrix and its partition over
// the workgroups of the persistent Krylov kernels (rows.hip).
//
// Rows (nodes, internal order) are cut into slabs of kSlab consecutive rows of
// one system. Inside a slab rows are sorted by their number of off-diagonal
// entries, so that the 64 rows of a wave (a slice) have nearly the same count
// and padding stays at a few per cent. A slice stores its entries entry by
// entry, 64 lanes wide (coalesced): entry j of lane l of slice q is
// (slice_off[q] + j) * 64 + l.
//
// A workgroup owns `group` consecutive slabs (a power of two, the same for
// the whole context). It holds the multiplied vector of its own rows and of
// its halo (rows of other workgroups that its entries name) in LDS; ids[] are
// indices into that array: own row at position p of the workgroup's k-th slab
// is k * kSlab + p, halo entry h is group * kSlab + h. Between products each
// workgroup hands the rows that others need (exp_loc) to them through global
// memory.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "layout.h"

namespace bhip {

constexpr int kSlab = 1024;          // rows of a slab, threads of a workgroup
constexpr int kSlices = kSlab / 64;  // slices (waves) of a slab
constexpr int kMaxGroup = 8;         // slabs of one workgroup
constexpr int kMaxGang = 256;        // workgroups of one system

struct RowLayout {
  int nslab = 0, group = 1, nwg = 0;
  int max_halo = 0, max_gang = 0;
  int64_t nent = 0;                  // entries, 64 per unit of slice_off
  int64_t nref = 0;
  std::vector<int32_t> slab_row0;    // [nslab] first row (internal node id)
  std::vector<int32_t> slab_rows;    // [nslab] rows of the slab
  std::vector<uint16_t> rowpos;      // [nslab * kSlab] row - slab_row0 at position p, 0xffff: none
  std::vector<int32_t> slice_off;    // [nslab * kSlices + 1]
  std::vector<uint16_t> ids;         // [nent] LDS index of the entry's column
  // assembly: entry column j of slice q sums cnt[slice_off[q] + j] coefficients,
  // whose references start at ref_off[q] * 64, 64 lanes wide, column by column.
  // A reference is pair * nslot_pad + slot, its top bit set for a term below
  // the element's diagonal (the second half of a non-symmetric matrix), or -1
  std::vector<uint8_t> cnt;
  std::vector<int64_t> ref_off;      // [nslab * kSlices]
  std::vector<int32_t> refs;
  // workgroups
  std::vector<int32_t> wg_slab0;     // [nwg + 1]
  std::vector<int32_t> wg_sys;       // [nwg]
  std::vector<int32_t> sys_wg;       // [nsys + 1]
  std::vector<int32_t> halo_off;     // [nwg + 1]
  std::vector<int32_t> halo_row;     // internal node id
  std::vector<int32_t> halo_src;     // index into the exported values
  std::vector<int32_t> exp_off;      // [nwg + 1]
  std::vector<uint16_t> exp_loc;     // LDS index of the exported row
};

// Rows of the layout's matrix for nsys systems of node_off[nsys + 1] nodes.
// max_wg: workgroups that can be resident at once. Returns false (and leaves R
// empty) when a system needs more workgroups than that, or more than kMaxGang.
bool build_rows(const Layout& L, int nsys, const int64_t* node_off, int max_wg, RowLayout& R);

}  // namespace bhip
