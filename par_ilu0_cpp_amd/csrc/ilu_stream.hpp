// Chunk streams of the block-local sweeps (ilu_stream.hip).
#pragma once

#include "ilu_internal.hpp"

namespace pilu {

// Rows in sweep order and how they are grouped (device arrays): rows of block
// p (processing order) and one local level are perm[loff[g] .. loff[g + 1]),
// g in [blev[p], blev[p + 1]); blev has nblk + 1 entries.
struct StreamSchedule {
    const int *perm, *blev, *loff, *block_of;
    int nblk;
};

// Whether every row of the direction has at most one entry per lane.
bool stream_width_fits(const lljbash::IluSolver::Ext* e, bool upper, int G);

// Builds the pattern part of a stream for G lanes per row
// (stream_width_fits); false, with st.lds == 0, where a block does not fit
// the LDS, a row is imported by more blocks than it has lanes for or the
// stream exceeds its budget of memory.
bool build_stream(lljbash::IluSolver::Ext* e, bool upper, int G, const StreamSchedule& sc, SweepStream& st);

// Refreshes the values of a built stream from the factors.
void gather_stream(lljbash::IluSolver::Ext* e, bool upper, SweepStream& st);

// One sweep over a stream whose values are current.  reset, if given, is
// filled with kPending after it.
void sweep_stream(lljbash::IluSolver::Ext* e, bool upper, const SweepStream& st, const double* b, double* out,
                  double* reset, const int* gate, int* ctr, int* err);

// Raised when a sweep structure is missing during a no-allocation apply.
void refuse_if_no_alloc(const lljbash::IluSolver::Ext* e, const char* what);

}  // namespace pilu
