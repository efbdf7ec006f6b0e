// Assembled row storage of an EBE (or segment) matrix and its partition over
// the workgroups of the persistent Krylov kernels (rows.hip).
//
// Rows (nodes, internal order) are cut into slabs of kSlab consecutive rows of
// one system; a workgroup owns `group` consecutive slabs (a power of two, the
// same for the whole context), `group` rows per thread. Every row has a leaf
// number in its slab that does not depend on the group, and thread t of a
// workgroup owns the leaves t * group ... t * group + group - 1 of its slabs:
// sums over rows are binary trees over leaves, first within a thread, so they
// do not depend on the group either.
//
// Leaves are given out so that the 64 rows a wave works on at once (a slice:
// the k-th rows of its lanes) have nearly the same number of entries. Each
// half of a slab is sorted by it; rank g * 64 + v becomes leaf 8 v + j(g), j =
// 0, 4, 1, 5, 2, 6, 3, 7: groups of 8 take one run of 64 ranks per slice,
// groups of 4 two neighbouring ones. (Groups of up to 4 keep their rows'
// first entries in registers, where padding costs nothing.)
//
// A slice stores its coefficients entry by entry, 64 lanes wide (coalesced):
// entry j of lane l of slice q is (slice_off[q] + j) * 64 + l. Its column ids
// are stored two entries to a 32-bit word: ids[((pair_off[q] + j / 2) * 64 + l) * 2
// + (j & 1)], at least one word per lane (zeros where the slice is empty). Slice
// k * kSlices + w of workgroup g is q = g * group * kSlices + that.
//
// A workgroup holds the multiplied vector of its own rows and of its halo (rows
// of other workgroups that its entries name) in LDS; ids[] are indices into that
// array: thread t's k-th row is k * kSlab + t, halo entry h is group * kSlab + h.
// With each product the workgroups hand the rows that others need (exp_loc) to
// them through global memory.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "layout.h"

namespace bhip {

constexpr int kSlab = 1024;          // rows of a slab, threads of a workgroup
constexpr int kSlices = kSlab / 64;  // waves of a workgroup, slices of one row per thread
constexpr int kRefChunk = 4;
constexpr size_t kSlabLds = 152 << 10;  // LDS of the fused D A D and assembly (by_block)
constexpr int kMaxGroup = 8;         // slabs of one workgroup
constexpr int kMaxGang = 256;        // workgroups of one system
constexpr int kXcds = 8;             // dies that a launch's workgroups go to in turn

struct RowLayout {
  int group = 1, nwg = 0, nslice = 0;
  int max_halo = 0, max_gang = 0;
  int64_t nent = 0;                  // entries, 64 per unit of slice_off
  int64_t nref = 0;
  std::vector<int32_t> wg_row0;      // [nwg] first row (internal node id)
  std::vector<uint16_t> rowpos;      // [nwg * group * kSlab] row - wg_row0 at LDS index, 0xffff: none
  std::vector<int32_t> slice_off;    // [nslice + 1]
  std::vector<int32_t> pair_off;     // [nslice + 1]
  std::vector<uint16_t> ids;         // LDS index of the entry's column
  // assembly: the coefficients a slice's entries sum, reference column by
  // reference column, 64 lanes wide, entry after entry: column c of slice q is
  // refs[(ref_off[q] + c) * 64 + lane]. A reference is pair * nslot_pad + slot,
  // its top bit set for a term below the element's diagonal (the second half
  // of a non-symmetric matrix), or -1. Columns come in chunks of kRefChunk
  // (filled up with -1); bit c of a chunk's byte in ref_end says that column c
  // is the last one of its entry.
  std::vector<int32_t> ref_off;      // [nslice + 1], multiples of kRefChunk
  std::vector<uint8_t> ref_end;      // [ref_off / kRefChunk]
  std::vector<int32_t> refs;
  // node blocks that are the slabs (triangles and segments, blocks of kSlab
  // nodes): the references within a block instead, pair * slots of the block +
  // slot - its first slot, top bit as above, 0xffff: none
  bool by_block = false;
  int max_slots = 0;                 // slots of one block
  std::vector<uint16_t> refs16;
  // workgroups
  std::vector<int32_t> wg_sys;       // [nwg]
  std::vector<int32_t> sys_wg;       // [nsys + 1]
  // launches of one solve: first workgroup of each, and nwg. A launch of more
  // than the GPU holds numbers its workgroups as they start, so that the lowest
  // unfinished system has all of its own started, or none but its own starting
  // next. They go to the XCDs in turn, whoever is ahead, so at the end those left
  // may all wait for one XCD: a system must fit on one, else there are several
  // launches, each of whole systems that the GPU holds at once.
  std::vector<int32_t> launch;
  std::vector<int32_t> halo_off;     // [nwg + 1]
  std::vector<int32_t> halo_row;     // internal node id
  std::vector<int32_t> halo_src;     // index into the exported values
  std::vector<int32_t> exp_off;      // [nwg + 1]
  std::vector<uint16_t> exp_loc;     // LDS index of the exported row
};

// LDS of the CG kernel for `bytes` (8 or 4) per value: D and A D of own rows; D,
// A D and R of the halo; mixed: X of both in FP64
inline size_t cg_lds(int group, size_t max_halo, int bytes) {
  return ((size_t)2 * group * kSlab + 3 * max_halo) * bytes +
         (bytes == 4 ? ((size_t)group * kSlab + max_halo + 1) * sizeof(double) : 0);
}

// Rows of the layout's matrix for nsys systems of node_off[nsys + 1] nodes.
// max_wg: workgroups that can be resident at once; max_lds: of one. Returns false
// (and leaves R empty) when a system needs more workgroups than that, or more than
// kMaxGang, or a workgroup's halo more LDS. Throws std::bad_alloc.
bool build_rows(const Layout& L, int nsys, const int64_t* node_off, int max_wg, size_t max_lds,
                RowLayout& R);

}  // namespace bhip
