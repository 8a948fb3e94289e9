// Chunk streams of the block-local sweeps (ilu_stream.hip).
#pragma once

#include "ilu_internal.hpp"

namespace pilu {

// Whether the current partition may be swept over a stream with G lanes per
// row: one lane per entry, and no earlier attempt found the block too large
// for the LDS.
bool stream_applies(const lljbash::IluSolver::Ext* e, bool upper, int G);

// Builds the stream (and its values, once factored) where it is missing or
// stale; false where the partition has to be swept otherwise.
bool ensure_stream(lljbash::IluSolver::Ext* e, bool upper, int G);

// Refreshes the values of a current stream from the factors.
void gather_stream(lljbash::IluSolver::Ext* e, bool upper);

// One sweep (ensure_stream has returned true for this direction).  reset, if
// given, is filled with kPending after it.
void sweep_stream(lljbash::IluSolver::Ext* e, bool upper, const double* b, double* out, double* reset, const int* gate,
                  int* ctr, int* err);

// Raised when a sweep structure is missing during a no-allocation apply.
void refuse_if_no_alloc(const lljbash::IluSolver::Ext* e, const char* what);

}  // namespace pilu
