// Which indices of a K-major operand the lanes of a split product's tile hold
// and store (LsCol in linear_split.h).  Plain C++ (no HIP types) so that a host
// compiler can build it on its own; under hipcc these are also the device
// functions that the kernel runs.
//
// A tile starts at index i0 of `count` and holds 16 T of them: lane row r loads
// the run T r .. T r + T - 1 (element t makes tile t's fragment).  A run that
// would pass the last index starts T before the end instead, at `last` -- which
// lies before the tile where fewer than T indices are left of it -- so edge
// tiles take the same vector loads.  Such a run repeats elements of other runs,
// or of the tile before; an index belongs to the run that would have held it
// unmoved, so each index of the operand is stored by one lane of one tile.
#ifndef NOVAQ_SPLIT_INDEX_H
#define NOVAQ_SPLIT_INDEX_H

#ifdef __HIPCC__
#define NOVAQ_SPLIT_HD __host__ __device__
#else
#define NOVAQ_SPLIT_HD
#endif

namespace novaq {
namespace split_detail {

// The latest start of a run, relative to the tile (count >= T; may be negative).
NOVAQ_SPLIT_HD inline int col_last(int T, int count, int i0) { return count - T - i0; }

// Index, relative to the tile, of element t of lane row r's run.
NOVAQ_SPLIT_HD inline int col_index(int T, int last, int t, int r) {
  return (T * r < last ? T * r : last) + t;
}

// Whether lane row r stores that element.
NOVAQ_SPLIT_HD inline bool col_owns(int T, int last, int t, int r) { return t >= T * r - last; }

}  // namespace split_detail
}  // namespace novaq

#endif  // NOVAQ_SPLIT_INDEX_H
