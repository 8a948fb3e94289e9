// What the chunk stream's kernel (ilu_stream.hip) asks of its buffers, in
// plain C++ so that it can be checked on the host.
#pragma once

#include <cstddef>

namespace pilu {

constexpr int kStSolvers = 8;  // solver waves per workgroup; a block's chunks are a multiple of them
// Requests run kStAhead chunks (of the same wave) ahead for the slots, half
// of that for the values, the diagonal and b, whose address comes with them.
constexpr int kStAhead = 16;
constexpr int kStAheadB = 8;

// Chunks of a stream's buffers past its last one.  A solver wave requests
// kStAhead chunks before its loop and one per turn of it, and turns come in
// multiples of kStAhead: at most kStAhead - 1 more than it has chunks.  So the
// last block's waves request 2 kStAhead - 1 chunks each past its end (values:
// kStAheadB fewer), which have to be there: the moving part of the address is
// the scalar offset of a buffer request, which no range check is documented
// to cover.
constexpr long kStOverrun = kStSolvers * (2L * kStAhead - 1);

// LDS of a block: a word per row and per import, and two for unused lanes and
// rows.  The 160 KiB of a CU also hold the workgroup's ticket, a static word
// that the dynamic part is aligned after.
constexpr size_t kStStaticLds = 16;
constexpr size_t kStMaxLds = 160 * 1024 - kStStaticLds;
constexpr size_t st_block_lds(size_t rows, size_t imports) { return 8 * (rows + imports + 2); }

}  // namespace pilu
