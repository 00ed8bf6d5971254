// tri_strips.hpp -- sparse triangular solves as a pipeline of row strips (see
// tri_strips.hip).
#pragma once

#include <vector>

#include "common.hpp"

namespace tnlmi {

constexpr int kTriGroup = 3;       // steps between two looks at the other waves' flags
// Imported values in LDS.  Before a group of steps the solving wave waits for the
// group's imports while the group before, in progress, still holds its own: two
// groups' imports, three per row, have to fit.
constexpr int kTriImports = 2048;
static_assert( kTriImports >= 2 * kTriGroup * 64 * 3 && ( kTriImports & ( kTriImports - 1 ) ) == 0 );

// One triangular factor prepared for the strip solve.  Rows are taken in solve
// order t (lower: row t, upper: row N - 1 - t); a position is 64 * step + lane
// over all strips.
struct TriStrips
{
   int64_t n = 0;
   int64_t steps = 0;  // of all strips
   int32_t strips = 0;
   int entries = 0;  // off-diagonal entries per row at most (2 or 3)
   bool upper = false;
   DeviceArray< int32_t > table;  // per strip: first step, steps, first import, imports
   DeviceArray< int32_t > need;   // per kGroup steps: the strip's imports used up to and including them
   DeviceArray< int32_t > src;    // per import: position of the value
   DeviceArray< int32_t > row;    // per position: its row (-1: none)
   DeviceArray< int32_t > pos;    // per row: its position
   DeviceArray< char > records;   // per step: addresses, values, pivots and right-hand side of its 64 rows
   uint32_t block = 0, b_at = 0;  // bytes of a step's records; where in them the right-hand side is
   DeviceArray< double > x;       // solution by position
   DeviceArray< int32_t > started;  // workgroups of the solve that have started
   bool used() const { return strips > 0; }
};

// A factor's schedule on the host.
struct TriStripsPlan
{
   int64_t n = 0, steps = 0;
   int32_t strips = 0;  // 0: another solve is expected to be faster
   int entries = 0;
   bool upper = false;
   uint32_t block = 0, b_at = 0;
   std::vector< int32_t > table, need, src, row, pos;
   std::vector< char > records;
};

// Plans the factor in CSR arrays (ILU(0)'s layout: lower rows with their
// strictly lower entries; upper rows reversed, the pivot first), unless
// other_us, the time another solve of the factor is expected to take, is less
// than the strip solve's.  Host work only.
TriStripsPlan tri_strips_plan( int64_t N, const std::vector< int32_t >& ptr, const std::vector< int32_t >& col,
                               const std::vector< double >& val, bool upper, double other_us );
// T from the plan (the plan's arrays are read until s has passed)
void tri_strips_upload( TriStrips& T, const TriStripsPlan& P, hipStream_t s );

// The right-hand side of position p = src[map[p]], T.x[p] = "not solved": what tri_strips_solve starts from.
void tri_strips_load( TriStrips& T, const double* src, const int32_t* map, hipStream_t s );
// the solution by position into T.x
void tri_strips_solve( TriStrips& T, int64_t spin_cap, hipStream_t s );
// x[i] = the solution's row i
void tri_strips_result( const TriStrips& T, double* x, hipStream_t s );

}  // namespace tnlmi
