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

// One CG per system of the context (gracjg.F:189-409) in one launch. Vectors in
// internal node order. FP64: a whole solve of A x = b, from the initial
// solution to the outcome in the state (gave_up is only ever set). FP32: the
// inner solve that the outer test has started, if it has, with its state.
template <typename T>
struct RowsCg {
  const T* b;              // FP64: b; FP32: the residual b - A x the inner solve starts from
                           // (its sign as the mixed solver keeps it)
  const T* diag;           // diagonal, or nullptr for a unit diagonal
  T* x;                    // solution; FP64: at idx[i] (or i), times scale[i] if given (not
                           // x0: a launch that gives up leaves that as it is)
  SolveState* st;
  const T* x0;             // FP64: initial solution
  const T* scale;
  const int32_t* idx;
  double eps;
  int nitmax;
  T* dlast;                // FP32: the previous direction of a continued solve (read), and
                           // the last direction of this one (written)
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
