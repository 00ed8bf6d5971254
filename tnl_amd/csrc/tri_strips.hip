// tri_strips.hip -- sparse triangular solves (the ILU(0) preconditioner's,
// ILU0.hpp:99-139) as a pipeline of row strips.
//
// What bounds a triangular solve is its chain of dependent rows.  One
// workgroup for the whole factor pays a barrier or an LDS poll among 16 waves
// per level (0.65 us a level); a launch per level pays several us.  Here the rows
// are cut into strips of consecutive rows, one workgroup each.  Within a strip
// ONE wave solves 64 rows per step, lane = row, in the order of the strip's own
// levels: a dependent value goes from step to step through LDS without any
// barrier (LDS accesses of one wave complete in order).  Values that cross
// strips go through memory, off the solving wave's path: a second wave
// imports them into LDS ahead of their use, a third writes the solved values
// out.  Strips run concurrently, each some steps behind the strip it reads from
// (a grid's strip of 64 lines: 64 steps), so the latency between workgroups is
// paid once per strip and not once per level.
//
// 1024^2 grid, 5-point stencil (2,047 levels each way, 16 strips of 64 lines):
// lower 222 us, upper 276 us, against 1,290 and 1,404 us for one workgroup
// without barriers (tri_flow); an apply 526 us against 2,950 us.  80^3 grid:
// 0.37 against 3.0 ms (a launch per wide level).  What is left is the chain of a
// step, about 0.1 us: an LDS write, the next step's LDS read and its
// multiply-adds, with everything else (record requests, flags) issued while
// LDS answers (0.16 us when these stood in the chain).
//
// Waiting: a strip reads earlier strips only, and workgroups take the strips in
// the order in which they start (a counter: the XCDs start their workgroups
// independently, and other kernels may keep one of them busy), so the strips a
// running one waits for have started.  Every wait is bounded all the same: an
// import that is not there after spin_cap polls ends all waiting of its
// workgroup, whose values become NaN.  "Not there" is a signalling NaN written before the solve, a
// value that no arithmetic gives.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "tri_strips.hpp"

namespace tnlmi {
namespace {

constexpr int kWin = 48;                       // steps whose values stay in LDS (a multiple of kAhead)
constexpr int kImports = kTriImports;          // imported values in LDS
constexpr int kExt = kWin * 64;                // LDS address of the first import
constexpr int kZero = kExt + kImports;         // LDS address of a 0 (an absent entry)
static_assert( 8 * kZero <= 0xffff, "LDS byte addresses of 16 bits" );
constexpr int kAhead = 12;                     // steps whose records are requested ahead
constexpr int kGroup = kTriGroup;              // steps between two looks at the other waves' flags (divides kAhead)
constexpr int kBatches = 8;                    // batches of 64 imports requested together at most
constexpr int kMaxStrips = 256;                // one per CU
// pivots and quotients for which the quotient from the reciprocal is exact to
// rounding (their product and its rounding error are normal numbers)
constexpr double kSmall = 1e-130, kLarge = 1e130;
constexpr uint64_t kUnsolved = 0x7ff4dead5eed0001ull;  // a signalling NaN

// what the model of the strip choice counts: measured on MI355X
constexpr double kStepUs = 0.1;   // a step of the solving wave
constexpr double kLagSteps = 22;  // a value's way to the next strip, in steps
// The last strip may wait for its first value until all others are done, and by
// default a wait is given up after 2^20 polls, about a second: at most 0.2 s of steps.
constexpr double kMostSteps = 2e6;

struct Shared
{
   double v[ kZero + 1 ];
   int32_t solved;   // steps solved
   int32_t used;     // imports used
   int32_t present;  // imports in LDS so far
   int32_t written;  // steps written out
   int32_t failed;
   int32_t strip;
};

// LDS flags: accesses of one wave to LDS complete in order, so a flag written
// after the values it covers is seen after them; the wavefront-scope fences
// only keep the compiler from reordering.
__device__ __forceinline__ void keep_order()
{
   __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
}
__device__ __forceinline__ int32_t flag( const int32_t* p )
{
   return __hip_atomic_load( p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
}
__device__ __forceinline__ void set_flag( int32_t* p, int32_t v )
{
   __hip_atomic_store( p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
}
// waits until *p >= target (or the workgroup has given up); the new value
__device__ __forceinline__ int32_t wait_for( const int32_t* p, int32_t target, Shared& S, int64_t cap )
{
   int32_t v = wave_uniform( flag( p ) );
   for( int64_t n = 0; v < target; n++ ) {
      if( wave_uniform( flag( &S.failed ) ) )
         return target;
      if( n >= cap ) {
         set_flag( &S.failed, 1 );
         return target;
      }
      v = wave_uniform( flag( p ) );
   }
   keep_order();
   return v;
}

// What a row needs besides the values it reads.  A step's 64 records are laid
// out field by field in one block of kBytes (every field at an immediate
// offset of one address): the solving wave issues one instruction at a time,
// so its address arithmetic counts.
template< bool UPPER, int K >
struct Record
{
   using Addr = std::conditional_t< ( K > 2 ), uint64_t, uint32_t >;
   Addr a;      // byte addresses in LDS of the values it reads, 16 bits each
   double2 v;   // the values of entries 0 and 1
   double v2;   // entry 2 (K == 3)
   double2 d;   // pivot and reciprocal (UPPER)
   double b;    // right-hand side
   static constexpr uint32_t kV = 0, kD = 1024, kV2 = kD + ( UPPER ? 1024 : 0 ), kB = kV2 + ( K > 2 ? 512 : 0 ),
                             kA = kB + 512, kBytes = kA + 64 * sizeof( Addr );
};

template< bool UPPER, int K >
__global__ void __launch_bounds__( 192 )
   tri_strips( const int32_t* __restrict__ table, const int32_t* __restrict__ need, const int32_t* __restrict__ src,
               const char* __restrict__ records, double* x, int32_t* started, int64_t spin_cap )
{
   using R = Record< UPPER, K >;
   __shared__ Shared S;
   const int wave = wave_uniform( (int32_t) ( threadIdx.x >> 6 ) ), lane = threadIdx.x & 63;
   if( threadIdx.x == 0 ) {
      S.strip = atomicAdd( started, 1 );
      S.v[ kZero ] = 0.0;
      S.solved = 0;
      S.used = 0;
      S.present = 0;
      S.written = 0;
      S.failed = 0;
   }
   __syncthreads();
   const int32_t strip = wave_uniform( S.strip );
   if( strip >= (int32_t) gridDim.x )
      return;  // (not if tri_strips_load came before)
   const int32_t step0 = table[ 4 * strip ], steps = table[ 4 * strip + 1 ];
   const int32_t src0 = table[ 4 * strip + 2 ], imports = table[ 4 * strip + 3 ];
   // LDS waits end when another wave of the workgroup goes on; their own limit
   // only backs that up
   const int64_t lds_cap = spin_cap * 16;
   if( wave == 0 ) {  // ---- solves
      R st[ kAhead ];
      int32_t nd[ kAhead / kGroup ];
      int64_t next = (int64_t) step0 * R::kBytes, next_need = step0 / kGroup * 4;
      uint32_t zero = 0;
      asm( "" : "+v"( zero ) );  // need[] by a vector load: a scalar one would share the counter that LDS reads wait on
      auto load = [ & ]( R& w ) {  // (unconditional: none waits for another)
         int64_t at = next;
         asm( "" : "+s"( at ) );  // (one scalar address; the lane's offsets stay in registers)
         const char* q = records + at;
         w.a = *(const typename R::Addr*) ( q + lane * (uint32_t) sizeof( typename R::Addr ) + R::kA );
         w.v = *(const double2*) ( q + lane * 16u + R::kV );
         if( K > 2 )
            w.v2 = *(const double*) ( q + lane * 8u + R::kV2 );
         if( UPPER )
            w.d = *(const double2*) ( q + lane * 16u + R::kD );
         w.b = *(const double*) ( q + lane * 8u + R::kB );
         next += R::kBytes;
         __builtin_amdgcn_sched_barrier( 0 );  // stage by stage: the wait for one leaves the later ones in flight
      };
      auto load_need = [ & ]( int32_t& w ) {
         int64_t at = next_need;
         asm( "" : "+s"( at ) );
         w = *(const int32_t*) ( (const char*) need + at + zero );
         next_need += 4;
      };
      int32_t present = 0, written = 0, s0 = 0;
      // before the group of steps that ends before step last: its n imports are
      // there, and the slots of the steps kWin back are written out
      auto group_ready = [ & ]( int32_t n, int32_t last ) {
         if( n > wave_uniform( present ) )
            present = wave_uniform( wait_for( &S.present, n, S, lds_cap ) );
         if( last - kWin > wave_uniform( written ) )
            written = wave_uniform( wait_for( &S.written, last - kWin, S, lds_cap ) );
      };
#pragma unroll
      for( int d = 0; d < kAhead - 1; d++ ) {
         if( d % kGroup == 0 )
            load_need( nd[ d / kGroup ] );
         load( st[ d ] );
      }
      char* const lds = (char*) S.v;
      uint32_t slot = lane * 8u;  // of this lane in the first step of the round
      int32_t used = 0;           // imports used by the groups before this one
      group_ready( wave_uniform( nd[ 0 ] ), kGroup );
      do {  // (steps > 0: a loop that may not run would let the requests above be moved into it)
#pragma unroll
         for( int d = 0; d < kAhead; d++ ) {
            R& w = st[ d ];
            const double x0 = *(const double*) ( lds + ( w.a & 0xffff ) );
            const double x1 = *(const double*) ( lds + ( w.a >> 16 & 0xffff ) );
            const double x2 = K > 2 ? *(const double*) ( lds + ( (uint64_t) w.a >> 32 & 0xffff ) ) : 0.0;
            __builtin_amdgcn_sched_barrier( 0 );
            // while LDS answers: what the chain of steps does not wait for.  The
            // records of the step before are used up: request those kAhead on
            load( st[ ( d + kAhead - 1 ) % kAhead ] );
            if( d % kGroup == 0 && lane == 0 ) {  // the group before is solved
               set_flag( &S.used, used );
               set_flag( &S.solved, s0 + d );
            }
            if( d % kGroup == kGroup - 1 ) {
               constexpr int G = kAhead / kGroup;
               used = wave_uniform( nd[ d / kGroup ] );
               load_need( nd[ d / kGroup ] );
               // (after the last group: the next strip's count)
               group_ready( min( wave_uniform( nd[ ( d / kGroup + 1 ) % G ] ), imports ), s0 + d + 1 + kGroup );
            }
            __builtin_amdgcn_sched_barrier( 0 );
            // the entries in their order, as the level solves
            double t = w.b;
            t -= w.v.x * x0;
            t -= w.v.y * x1;
            if( K > 2 )
               t -= w.v2 * x2;
            if( UPPER ) {
               // t / pivot from the pivot's correctly rounded reciprocal and
               // one correction, which gives the correctly rounded quotient
               // (Markstein 1990) away from the ends of the exponent range;
               // there, and for a pivot whose reciprocal is not safe (stored
               // as 0), the division itself
               double q = t * w.d.y;
               q = fma( fma( -q, w.d.x, t ), w.d.y, q );
               const double m = fabs( q );
               const bool plain = m > kSmall && m < kLarge;
               if( __builtin_expect( __ballot( ! plain ) != 0, 0 ) ) {  // (uniform)
                  asm volatile( "" );  // (a branch: the division is not computed beside the quotient)
                  q = plain ? q : t / w.d.x;
               }
               t = q;
            }
            *(double*) ( lds + slot + d * 512 ) = t;
            keep_order();
         }
         s0 += kAhead;
         slot = slot + kAhead * 512 < kWin * 512 ? slot + kAhead * 512 : lane * 8u;
      } while( s0 < steps );
      if( lane == 0 ) {
         set_flag( &S.used, used );
         set_flag( &S.solved, steps );
      }
   }
   else if( wave == 1 ) {  // ---- imports
      int32_t k = 0;  // imports [0, k) are in LDS
      int64_t polls = 0;
      bool given_up = false;
      // asks for the next NB batches of 64; the leading ones that are there go
      // to LDS.  Returns whether all were there.
      auto fetch = [ & ]( auto nb ) {
         constexpr int NB = decltype( nb )::value;
         // the slot of import i is free once import i - kImports is used
         const int32_t top = min( imports, wave_uniform( flag( &S.used ) ) + kImports );
         int32_t at[ NB ];
         uint64_t v[ NB ];
#pragma unroll
         for( int u = 0; u < NB; u++ )
            at[ u ] = src[ src0 + min( k + u * 64 + lane, imports - 1 ) ];
#pragma unroll
         for( int u = 0; u < NB; u++ )
            v[ u ] = __hip_atomic_load( (const uint64_t*) x + at[ u ], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
         given_up = given_up || wave_uniform( flag( &S.failed ) );
         int32_t got = 0;
         bool more = true;
#pragma unroll
         for( int u = 0; u < NB; u++ )
            if( more ) {  // (uniform)
               const int32_t i = k + u * 64 + lane;
               const uint64_t missing = __ballot( i >= top || ( v[ u ] == kUnsolved && ! given_up ) );
               const int lead = missing ? __builtin_ctzll( missing ) : 64;
               if( lane < lead )
                  S.v[ kExt + ( i & ( kImports - 1 ) ) ] = given_up ? __builtin_nan( "" ) : __longlong_as_double( v[ u ] );
               got += lead;
               more = lead == 64;
            }
         if( got > 0 ) {
            k += got;
            keep_order();
            if( lane == 0 )
               set_flag( &S.present, k );
            keep_order();
            polls = 0;
         }
         // none: a value that an earlier strip has not solved yet, or no free slot
         else if( ++polls >= ( top > k ? spin_cap : lds_cap ) )
            set_flag( &S.failed, 1 );
         return got == NB * 64;
      };
      bool many = false;  // one batch while the values trickle in
      while( k < imports )
         many = many ? fetch( std::integral_constant< int, kBatches >() ) : fetch( std::integral_constant< int, 1 >() );
   }
   else {  // ---- writes the solved values out
      int32_t e = 0;
      while( e < steps ) {
         const int32_t done = min( steps, wait_for( &S.solved, e + 1, S, lds_cap ) );
         const bool given_up = wave_uniform( flag( &S.failed ) );
         for( ; e < done; e++ ) {
            double t = S.v[ ( e % kWin ) * 64 + lane ];
            if( given_up )
               t = __builtin_nan( "" );
            uint64_t bits = (uint64_t) __double_as_longlong( t );
            if( bits == kUnsolved )
               bits |= uint64_t( 1 ) << 51;  // (a right-hand side's own signalling NaN, quiet)
            __hip_atomic_store( (uint64_t*) x + ( (int64_t) ( step0 + e ) * 64 + lane ), bits, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT );
         }
         keep_order();
         if( lane == 0 )
            set_flag( &S.written, e );
         keep_order();
      }
   }
}

// block, at: bytes of a step's records and where in them the right-hand side is
__global__ void __launch_bounds__( 256 )
   strips_load( int64_t n, const int32_t* __restrict__ map, const double* __restrict__ src,
                char* __restrict__ records, uint32_t block, uint32_t at, double* __restrict__ x,
                int32_t* __restrict__ started )
{
   const int64_t p = (int64_t) blockIdx.x * 256 + threadIdx.x;
   if( p >= n )
      return;
   if( p == 0 )
      *started = 0;
   const int32_t i = map[ p ];
   // (an idle lane: not 0, which would take the division)
   *(double*) ( records + ( p >> 6 ) * block + at + ( p & 63 ) * 8 ) = i >= 0 ? src[ i ] : 1.0;
   x[ p ] = __longlong_as_double( (long long) kUnsolved );
}

__global__ void __launch_bounds__( 256 )
   strips_result( int64_t n, const int32_t* __restrict__ pos, const double* __restrict__ xp, double* __restrict__ x )
{
   const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
   if( i < n )
      x[ i ] = xp[ pos[ i ] ];
}

template< typename T >
void upload( DeviceArray< T >& d, const std::vector< T >& h, hipStream_t s )
{
   d.allocate( std::max< int64_t >( 1, (int64_t) h.size() ) );
   if( ! h.empty() )
      TNLMI_HIP( hipMemcpyAsync( d.ptr, h.data(), sizeof( T ) * h.size(), hipMemcpyHostToDevice, s ) );
}

// the factor's rows in solve order
struct Factor
{
   int64_t N;
   const int32_t *ptr, *col;
   const double* val;
   bool upper;
   int32_t begin( int64_t t ) const { return upper ? std::min( ptr[ t ] + 1, ptr[ t + 1 ] ) : ptr[ t ]; }
   int32_t end( int64_t t ) const { return ptr[ t + 1 ]; }
   int64_t dep( int32_t g ) const { return upper ? N - 1 - col[ g ] : col[ g ]; }
};

// Steps of the strip [t0, t1): rows by their level within the strip, 64 to a
// step; slot[t] = 64 * step + lane.  The number of steps, up to a multiple of
// kAhead (the last ones without rows).
int32_t schedule( const Factor& F, int64_t t0, int64_t t1, std::vector< int32_t >& slot, std::vector< int32_t >& count )
{
   count.clear();
   for( int64_t t = t0; t < t1; t++ ) {
      int32_t l = 0;
      for( int32_t g = F.begin( t ); g < F.end( t ); g++ ) {
         const int64_t d = F.dep( g );
         if( d >= t0 )
            l = std::max( l, slot[ d ] + 1 );
      }
      slot[ t ] = l;
      if( l >= (int32_t) count.size() )
         count.push_back( 0 );
      count[ l ]++;
   }
   int32_t steps = 0;
   for( auto& c : count ) {
      const int32_t k = ( c + 63 ) / 64;
      c = 64 * steps;
      steps += k;
   }
   for( int64_t t = t0; t < t1; t++ )
      slot[ t ] = count[ slot[ t ] ]++;
   return (int32_t) ceil_div( steps, kAhead ) * kAhead;
}

// the expected steps from start to end for strips of R rows, from the two strips in the middle
double expected_steps( const Factor& F, int64_t R, std::vector< int32_t >& slot, std::vector< int32_t >& count )
{
   const int64_t ns = ceil_div( F.N, R ), k = ns / 2;
   const int64_t t0 = k * R, t1 = std::min( F.N, t0 + R ), before = std::max< int64_t >( 0, t0 - R );
   if( k > 0 )
      schedule( F, before, t0, slot, count );
   const int32_t steps = schedule( F, t0, t1, slot, count );
   int32_t behind = 0;
   int64_t imports = 0;
   for( int64_t t = t0; t < t1; t++ )
      for( int32_t g = F.begin( t ); g < F.end( t ); g++ ) {
         const int64_t d = F.dep( g );
         if( d < t0 ) {
            imports++;
            if( d >= before )
               behind = std::max( behind, slot[ d ] / 64 + 1 - slot[ t ] / 64 );
         }
         else if( slot[ t ] / 64 - slot[ d ] / 64 >= kWin )
            imports++;  // (not in LDS any more: by way of memory too)
      }
   // (a strip cannot go faster than its imports arrive: about kBatches * 64 per round trip to memory)
   const double rate = std::max< double >( steps, imports * kLagSteps / ( 64.0 * kBatches ) );
   return rate + (double) ( ns - 1 ) * ( behind + kLagSteps );
}

template< typename T >
struct Tag
{
   using type = T;
};
template< typename F >
void with_record( bool upper, int entries, F&& f )
{
   if( upper )
      entries > 2 ? f( Tag< Record< true, 3 > >() ) : f( Tag< Record< true, 2 > >() );
   else
      entries > 2 ? f( Tag< Record< false, 3 > >() ) : f( Tag< Record< false, 2 > >() );
}

}  // namespace

TriStripsPlan tri_strips_plan( int64_t N, const std::vector< int32_t >& ptr, const std::vector< int32_t >& col,
                               const std::vector< double >& val, bool upper, double other_us )
{
   TriStripsPlan T;
   const Factor F{ N, ptr.data(), col.data(), val.data(), upper };
   int widest = 0;
   int64_t reach = 0;  // the farthest dependency, in rows: a grid's line or plane
   for( int64_t t = 0; t < N; t++ ) {
      widest = std::max( widest, F.end( t ) - F.begin( t ) );
      for( int32_t g = F.begin( t ); g < F.end( t ); g++ ) {
         const int64_t d = F.dep( g );
         if( d < 0 || d >= t )
            return T;
         reach = std::max( reach, t - d );
      }
   }
   if( N < 128 || widest > 3 || widest == 0 )
      return T;
   // strips of whole lines or planes where the matrix has such, or of any rows
   std::vector< int32_t > slot( N ), count;
   std::vector< int64_t > sizes;
   for( int64_t c : { 64, 16, 4, 2, 1 } )
      sizes.push_back( c * reach );
   for( int64_t p : { 16, 64, 256 } )
      sizes.push_back( ceil_div( N, p ) );
   int64_t rows = 0;
   double best = 0;
   for( int64_t R : sizes ) {
      if( R < 64 || ceil_div( N, R ) > kMaxStrips || ( 2 * R > N && rows ) || R >= 2 * N )
         continue;
      const double e = expected_steps( F, std::min( R, N ), slot, count );
      if( ! rows || e < best ) {
         best = e;
         rows = std::min( R, N );
      }
   }
   if( ! rows || best * kStepUs > other_us || best > kMostSteps )
      return T;
   // the schedule of every strip
   const int64_t ns = ceil_div( N, rows );
   std::vector< int32_t >& table = T.table;
   table.resize( 4 * ns );
   int64_t steps = 0;
   for( int64_t k = 0; k < ns; k++ ) {
      table[ 4 * k ] = (int32_t) steps;
      table[ 4 * k + 1 ] = schedule( F, k * rows, std::min( N, ( k + 1 ) * rows ), slot, count );
      steps += table[ 4 * k + 1 ];
   }
   if( steps * 64 > 8 * N + 65536 || steps * 64 > INT32_MAX )
      return T;  // thin levels: mostly idle lanes
   std::vector< int32_t >&row = T.row, &pos = T.pos, &src = T.src, &need = T.need;
   std::vector< char >& rec = T.records;
   row.assign( steps * 64, -1 );
   pos.resize( N );
   for( int64_t k = 0; k < ns; k++ )
      for( int64_t t = k * rows; t < std::min( N, ( k + 1 ) * rows ); t++ ) {
         const int32_t p = table[ 4 * k ] * 64 + slot[ t ];
         const int64_t i = upper ? N - 1 - t : t;
         row[ p ] = (int32_t) i;
         pos[ i ] = p;
      }
   T.entries = widest > 2 ? 3 : 2;
   T.upper = upper;
   with_record( upper, T.entries, [ & ]( auto tag ) {
      using R = typename decltype( tag )::type;
      T.block = R::kBytes;
      T.b_at = R::kB;
   } );
   // (the solving wave requests kAhead steps past a strip's end)
   const int64_t asked = steps + kAhead;
   rec.assign( asked * T.block, 0 );
   need.assign( asked / kGroup, 0 );
   with_record( upper, T.entries, [ & ]( auto tag ) {
      using R = typename decltype( tag )::type;
      for( int64_t k = 0; k < ns; k++ ) {
         const int64_t src0 = (int64_t) src.size();
         for( int64_t st = 0; st < table[ 4 * k + 1 ]; st++ ) {
            const int64_t q = table[ 4 * k ] + st;
            char* block = rec.data() + q * R::kBytes;
            for( int lane = 0; lane < 64; lane++ ) {
               uint16_t a[ 4 ] = { 8 * kZero, 8 * kZero, 8 * kZero, 8 * kZero };
               double v[ 3 ] = { 0, 0, 0 }, d[ 2 ] = { 1, 1 };
               if( row[ q * 64 + lane ] >= 0 ) {
                  const int64_t t = upper ? N - 1 - row[ q * 64 + lane ] : row[ q * 64 + lane ];
                  int e = 0;
                  for( int32_t g = F.begin( t ); g < F.end( t ); g++, e++ ) {
                     const int64_t dep = F.dep( g );
                     const int32_t from = pos[ upper ? N - 1 - dep : dep ] - table[ 4 * k ] * 64;  // (in the strip: >= 0)
                     if( dep >= k * rows && st - from / 64 < kWin )
                        a[ e ] = (uint16_t) ( 8 * ( from % ( kWin * 64 ) ) );
                     else {
                        a[ e ] = (uint16_t) ( 8 * ( kExt + ( (int64_t) src.size() - src0 ) % kImports ) );
                        src.push_back( pos[ upper ? N - 1 - dep : dep ] );
                     }
                     v[ e ] = val[ g ];
                  }
                  if( upper ) {
                     d[ 0 ] = ptr[ t ] < ptr[ t + 1 ] ? val[ ptr[ t ] ] : 0.0;  // a row without entries has no pivot
                     const double m = std::fabs( d[ 0 ] );
                     d[ 1 ] = m > kSmall && m < kLarge ? 1.0 / d[ 0 ] : 0.0;
                  }
               }
               memcpy( block + R::kA + lane * sizeof( typename R::Addr ), a, sizeof( typename R::Addr ) );
               memcpy( block + R::kV + lane * 16, v, 16 );
               if( R::kB != R::kV2 )
                  memcpy( block + R::kV2 + lane * 8, v + 2, 8 );
               if( upper )
                  memcpy( block + R::kD + lane * 16, d, 16 );
            }
            need[ q / kGroup ] = (int32_t) ( (int64_t) src.size() - src0 );
         }
         table[ 4 * k + 2 ] = (int32_t) src0;
         table[ 4 * k + 3 ] = (int32_t) ( (int64_t) src.size() - src0 );
      }
   } );
   T.n = N;
   T.steps = steps;
   T.strips = (int32_t) ns;
   return T;
}

void tri_strips_upload( TriStrips& T, const TriStripsPlan& P, hipStream_t s )
{
   T.n = P.n;
   T.steps = P.steps;
   T.entries = P.entries;
   T.upper = P.upper;
   T.block = P.block;
   T.b_at = P.b_at;
   upload( T.table, P.table, s );
   upload( T.need, P.need, s );
   upload( T.src, P.src, s );
   upload( T.row, P.row, s );
   upload( T.pos, P.pos, s );
   upload( T.records, P.records, s );
   T.x.allocate( P.steps * 64 );
   T.started.allocate( 1 );
   T.strips = P.strips;
}

void tri_strips_load( TriStrips& T, const double* src, const int32_t* map, hipStream_t s )
{
   hipLaunchKernelGGL( strips_load, dim3( (unsigned) ceil_div( T.steps * 64, 256 ) ), dim3( 256 ), 0, s, T.steps * 64,
                       map, src, T.records.ptr, T.block, T.b_at, T.x.ptr, T.started.ptr );
}

void tri_strips_solve( TriStrips& T, int64_t spin_cap, hipStream_t s )
{
   auto go = [ & ]( auto kernel ) {
      hipLaunchKernelGGL( kernel, dim3( (unsigned) T.strips ), dim3( 192 ), 0, s, T.table.ptr, T.need.ptr, T.src.ptr,
                          (const char*) T.records.ptr, T.x.ptr, T.started.ptr, spin_cap );
   };
   if( T.upper )
      T.entries > 2 ? go( tri_strips< true, 3 > ) : go( tri_strips< true, 2 > );
   else
      T.entries > 2 ? go( tri_strips< false, 3 > ) : go( tri_strips< false, 2 > );
}

void tri_strips_result( const TriStrips& T, double* x, hipStream_t s )
{
   hipLaunchKernelGGL( strips_result, dim3( (unsigned) ceil_div( T.n, 256 ) ), dim3( 256 ), 0, s, T.n, T.pos.ptr,
                       (const double*) T.x.ptr, x );
}

}  // namespace tnlmi
