// Device side of the assembled row storage: the matrix in row form and the
// persistent CG on it (rows.hip).
#pragma once

#include "device_common.h"
#include "rows.h"

namespace bhip {

struct RowsDev;

// The rows of a layout on the current device, or nullptr when they cannot be
// used (build_rows, or no memory for them; *err stays hipSuccess then). Work is queued on stream;
// the host arrays are read before it returns.
RowsDev* rows_create(const Layout& L, int nsys, const int64_t* node_off, hipStream_t stream,
                     hipError_t* err);
void rows_destroy(RowsDev* r);

// Row values of precision 8 or 4 bytes: those of 4 are allocated here when first
// asked for. hipErrorOutOfMemory: solve without the rows.
hipError_t rows_reserve(RowsDev* r, int bytes);

// whether a launch has workgroups that wait for each other: it must not share the
// GPU with another such launch
bool rows_meet(const RowsDev* r);

// device memory that the rows hold
size_t rows_bytes(const RowsDev* r);

// Assembles the rows of the precision from the slot coefficients xa (upper
// npair columns, and the lower ones when nonsym), nslot_pad apart. both: in
// FP64 too (of 4 bytes).
hipError_t rows_assemble(RowsDev* r, int bytes, bool both, const double* xa, int nslot_pad,
                         int npair, bool nonsym, hipStream_t stream);

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
hipError_t rows_dmd(RowsDev* r, int bytes, bool both, const RowsDmd& a, hipStream_t stream);

// Kinds of launches, each with its own words in device memory for what its
// workgroups tell each other. After a launch that ended without giving up the
// caller says so; any other clears the words at the next launch of the kind.
enum RowsKind { kRowsCg, kRowsCgMixed, kRowsGmres };
void rows_ended(RowsDev* r, RowsKind k);

constexpr int kMaxOuter = 100;  // refinement sweeps of one mixed solve

// SOLVE's CG, one per system of the context, in one launch: from the initial
// solution to the outcome in the state (gave_up is only ever set). FP64
// (gracjg.F:189-409), or mixed: FP64 residuals, each reduced by inner_eps by an
// FP32 CG (the rows in both precisions). Vectors in internal node order.
struct RowsCg {
  const double* b;
  const double* diag;   // diagonal, or nullptr for a unit diagonal
  const double* x0;     // initial solution
  double* x;            // solution, at idx[i] (or i), times scale[i] if given (not x0: a
                        // launch that gives up leaves that as it is)
  const double* scale;
  const int32_t* idx;
  SolveState* st;       // the outcome, one per system; host memory will do: nothing is
                        // read back
  double eps;
  int nitmax;           // iterations (mixed: of all inner solves)
  double inner_eps;
  int inner_nitmax;
  int reliable;         // an inner solve continues the direction of the one before
  double* res;          // (scratch, set by rows_cg)
};
hipError_t rows_cg(RowsDev* r, bool mixed, RowsCg a, hipStream_t stream);

// Restarted GMRES (gmres.f:171-372) of a context of one system, a whole solve
// in one launch: FP64, or mixed (FP32 cycles, FP64 residuals; the rows in both
// precisions). Vectors in internal node order.
struct GmState {
  double prec;    // ||R0|| / max(||B||, 1)
  int m, products, relat;
  int updated;    // x has been written
  int gave_up;    // only ever set
};
struct RowsGmres {
  const double* x0;    // initial solution
  double* x;           // solution, if updated (not x0: see RowsCg)
  const double* diag;  // diagonal, or nullptr for a unit diagonal
  const double* b;
  double eps;
  int nitmax, krylov;
  GmState* st;         // the outcome; host memory will do
};
bool rows_gmres_fits(const RowsDev* r, int bytes);
// (allocates the basis when a larger K is first asked for; hipErrorOutOfMemory
// as of rows_reserve)
template <typename T>
hipError_t rows_gmres(RowsDev* r, const RowsGmres& a, hipStream_t stream);

}  // namespace bhip
