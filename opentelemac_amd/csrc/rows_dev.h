// Device side of the assembled row storage: the matrix in row form and the
// persistent CG on it (rows.hip).
#pragma once

#include "device_common.h"
#include "rows.h"

namespace bhip {

struct RowsDev;

// The rows of a layout on the current device, or nullptr when they cannot be
// used (build_rows; *err stays hipSuccess then). Work is queued on stream;
// the host arrays are read before it returns.
RowsDev* rows_create(const Layout& L, int nsys, const int64_t* node_off, hipStream_t stream,
                     hipError_t* err);
void rows_destroy(RowsDev* r);

// Row values of precision 8 or 4 bytes: allocated here when first asked for.
hipError_t rows_reserve(RowsDev* r, int bytes);

// Assembles the rows of the precision from the slot coefficients xa (upper
// npair columns, and the lower ones when nonsym), nslot_pad apart.
hipError_t rows_assemble(RowsDev* r, int bytes, const double* xa, int nslot_pad, int npair,
                         bool nonsym, hipStream_t stream);

// OM 'M=DMD' and the assembly in one pass, where node blocks are slabs
// (rows_by_block): the coefficients src times D(i) D(j), written to xa and
// summed into the rows. d nullptr: src as it is, xa not written.
bool rows_by_block(const RowsDev* r);
struct RowsDmd {
  const double* src;
  double* xa;
  const double* d;
  int ndp, nslot_pad, nblocks, max_local;
  bool nonsym;
  const uint16_t* lid;
  const int32_t* node_start;
  const int32_t* halo_start;
  const int32_t* halo;
  const int32_t* color_off;
};
hipError_t rows_dmd(RowsDev* r, int bytes, const RowsDmd& a, hipStream_t stream);

// One CG solve per system of the context (gracjg.F:248-409), from the
// residual r0 to the stop, in one launch. Vectors in internal node order.
template <typename T>
struct RowsCg {
  const T* r0;             // A x - b (FP64), or b - A x of an inner solve (its sign)
  const T* x0;             // initial solution, or nullptr for zero
  T* x;                    // solution (not x0: a launch that gives up leaves x0 as it is)
  const T* diag;           // diagonal, or nullptr for a unit diagonal
  T* dlast;                // the previous direction of a continued solve (read), and the
                           // last direction of this one (written); nullptr: neither
  const double* part_rr;   // partial sums of ||r0||^2 per node block, or nullptr: the
                           // state's rr0
  int nblocks;
  const int32_t* sys_blocks;
  SolveState* st;
  int inner;               // an inner solve: only systems with a fresh start
};
template <typename T>
hipError_t rows_cg(RowsDev* r, const RowsCg<T>& a, hipStream_t stream);

// Restarted GMRES (gmres.f:171-372) of a context of one system: FP64, the
// whole solve in one launch; FP32, one cycle of the mixed solve from the FP64
// residual r0 (nothing where the stop test on it ends the solve). Vectors in
// internal node order.
struct GmState {  // on the device, written by a launch
  double prec;    // ||R0|| / max(||B||, 1)
  int m, products, done, relat;
  int updated;    // x has been written
  int gave_up;    // a launch gave up waiting for its workgroups (never reset)
};
struct RowsGmres {
  const double* x0;  // initial solution
  double* x;         // solution, if updated (not x0: see RowsCg)
  const double* diag;  // diagonal, or nullptr for a unit diagonal
  const double* b;     // FP64
  const double* r0;    // FP32: A x - b, and the partial sums of r0.r0 and b.b
  const double* part_rr;
  const double* part_bb;
  int npart_rr, npart_bb;
  double eps;
  int nitmax, krylov;
  int first;           // first launch of the solve
};
bool rows_gmres_fits(const RowsDev* r, int bytes);
template <typename T>
hipError_t rows_gmres(RowsDev* r, const RowsGmres& a, hipStream_t stream);
hipError_t rows_gmres_state(const RowsDev* r, GmState* host, hipStream_t stream);

}  // namespace bhip
