// Sweeps of deep, narrow schedules by one workgroup (ilu_walk.hip).
#pragma once

#include "ilu_internal.hpp"

namespace pilu {

// Builds the pattern part of a direction's stream for G (>= 4) lanes per row;
// false where a level is too wide for the LDS ring or the stream exceeds its
// budget of memory.
bool build_walk(lljbash::IluSolver::Ext* e, bool upper, int G, WalkStream& w);

// Refreshes the values of a built stream from the factors.
void gather_walk(lljbash::IluSolver::Ext* e, bool upper, WalkStream& w);

// One sweep over a stream whose values are current.  reset, if given, is
// filled with kPending after it.
void sweep_walk(lljbash::IluSolver::Ext* e, bool upper, const WalkStream& w, const double* b, double* out, double* reset,
                const int* gate);

// Raised when a sweep structure is missing during a no-allocation apply.
void refuse_if_no_alloc(const lljbash::IluSolver::Ext* e, const char* what);

}  // namespace pilu
