// A triangular factor's strip plan, for tests/test_tri_strips_plan.py.
#include <algorithm>

#include "tri_strips.hpp"

// strips: 0 where another solve is taken.  Returns the most imports of two
// consecutive groups of steps in one strip.
extern "C" int32_t strips_plan( int64_t n, const int32_t* ptr, const int32_t* col, int upper, double other_us,
                                int32_t* strips )
{
   const std::vector< int32_t > p( ptr, ptr + n + 1 ), c( col, col + ptr[ n ] );
   const std::vector< double > v( c.size(), 1.0 );
   const tnlmi::TriStripsPlan T = tnlmi::tri_strips_plan( n, p, c, v, upper != 0, other_us );
   *strips = T.strips;
   int32_t most = 0;
   for( int32_t k = 0; k < T.strips; k++ ) {
      const int32_t* need = T.need.data() + T.table[ 4 * k ] / tnlmi::kTriGroup;
      const int32_t groups = T.table[ 4 * k + 1 ] / tnlmi::kTriGroup;
      for( int32_t g = 0; g < groups; g++ )
         most = std::max( most, need[ g ] - ( g >= 2 ? need[ g - 2 ] : 0 ) );
   }
   return most;
}

extern "C" int32_t strips_imports()
{
   return tnlmi::kTriImports;
}
