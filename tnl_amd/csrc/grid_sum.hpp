// grid_sum.hpp -- sums over all workgroups of a running kernel, and data
// passed between its workgroups, for kernels whose whole grid is resident
// (resident_launch): an iteration of a Krylov solver then needs no kernel
// boundary.  A launch costs about 5 us on MI355X and each reduction of an
// iteration used to end one; a grid sum takes about 2 us.
#pragma once

#include <cstdlib>
#include <mutex>

#include "common.hpp"

namespace tnlmi {

constexpr int kGridMax = 256;        // workgroups at most: one per CU
constexpr int kGridValues = 32;      // values per sum at most

// How long a workgroup waits for the others before it gives up, in ticks of
// 100 MHz: 2 s, or TNLMI_GRID_WAIT_US microseconds.
inline uint64_t grid_wait()
{
   const char* e = std::getenv( "TNLMI_GRID_WAIT_US" );
   return e ? 100 * std::strtoull( e, nullptr, 10 ) : 200'000'000;
}

// Launches a kernel whose workgroups wait for each other: at most one per compute
// unit, so all are on the chip at the same time once other kernels have ended.
// Two such kernels at a time could each hold units that the other waits for: the
// caller holds resident_turn() from the launch until the kernel has ended.  (No
// cooperative launch: a process with such launches from several threads' streams
// ended in a segmentation fault at its exit.)  False: nothing was launched.
inline bool resident_launch( const void* kernel, int64_t blocks, int threads, void** args, hipStream_t s )
{
   int dev = 0, cus = 0;
   if( hipGetDevice( &dev ) == hipSuccess
       && hipDeviceGetAttribute( &cus, hipDeviceAttributeMultiprocessorCount, dev ) == hipSuccess && blocks <= cus
       && blocks <= kGridMax
       && hipLaunchKernel( kernel, dim3( (unsigned) blocks ), dim3( threads ), args, 0, s ) == hipSuccess )
      return true;
   (void) hipGetLastError();
   return false;
}
// the device's: its streams' kernels share the compute units
inline std::unique_lock< std::mutex > resident_turn()
{
   static std::mutex turns[ 16 ];
   int dev = 0;
   (void) hipGetDevice( &dev );
   return std::unique_lock< std::mutex >( turns[ dev & 15 ] );
}

// One value of one workgroup: two words, each with half of the value and the
// sum's number, so that a reader sees from each word whether it belongs to
// the sum it waits for.  Two buffers in turn: a workgroup that publishes sum k
// has seen every workgroup's part of sum k - 1, so all are done with k - 2.
struct GridSlots
{
   uint64_t word[ 2 ][ kGridValues ][ kGridMax ][ 2 ];
};

// Accesses seen by all workgroups of the running kernel (the XCDs' L2 caches
// are not coherent with each other: these go past them).
template< typename T >
__device__ __forceinline__ T shared_load( const T* p )
{
   return __hip_atomic_load( p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
}
template< typename T >
__device__ __forceinline__ void shared_store( T* p, T v )
{
   __hip_atomic_store( p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
}

// this wave's shared_stores have reached where every workgroup sees them
__device__ __forceinline__ void shared_stores_done()
{
   asm volatile( "s_waitcnt vmcnt(0)" ::: "memory" );
}

// v[j] = the sum over all threads of all workgroups, in a fixed order (the same
// bits in every workgroup).  What a workgroup shared_stores before the sum is
// seen by all after it.  sm: N * T / 64 doubles of LDS.  Returns false when a
// workgroup did not arrive within `wait`.  The others may have seen it arrive and
// end normally when no sum follows: a kernel whose sum was given up says so in a
// word that nothing else writes.
template< int T, int N >
__device__ __forceinline__ bool grid_sum( double ( &v )[ N ], GridSlots* __restrict__ slots, uint32_t number, uint64_t wait,
                                          double* sm )
{
   static_assert( N <= kGridValues && T >= kGridMax, "one thread per workgroup's slot" );
   constexpr int W = T / 64;
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, G = gridDim.x;
   auto block_total = [ & ]( int j ) {
      double r = 0;
#pragma unroll
      for( int i = 0; i < W; i++ )
         r += sm[ j * W + i ];
      return r;
   };
   auto wave_totals = [ & ] {
#pragma unroll
      for( int j = 0; j < N; j++ )
         v[ j ] = group_sum< 64 >( v[ j ] );
      if( lane == 0 )
#pragma unroll
         for( int j = 0; j < N; j++ )
            sm[ j * W + w ] = v[ j ];
   };
   wave_totals();
   shared_stores_done();
   __syncthreads();
   uint64_t( &buf )[ kGridValues ][ kGridMax ][ 2 ] = slots->word[ number & 1 ];
   if( threadIdx.x < N ) {
      const uint64_t bits = (uint64_t) __double_as_longlong( block_total( threadIdx.x ) );
      const uint64_t tag = (uint64_t) number << 32;
      shared_store( &buf[ threadIdx.x ][ blockIdx.x ][ 0 ], tag | ( bits & 0xffffffffu ) );
      shared_store( &buf[ threadIdx.x ][ blockIdx.x ][ 1 ], tag | ( bits >> 32 ) );
   }
   __syncthreads();  // (sm is read above and written below)
   int late = 0;
   if( (int) threadIdx.x < G ) {
      const uint64_t begin = wall_clock64();
      uint64_t lo[ N ], hi[ N ];
      bool there = true, over = false;
      while( true ) {
         there = true;
#pragma unroll
         for( int j = 0; j < N; j++ ) {
            lo[ j ] = shared_load( &buf[ j ][ threadIdx.x ][ 0 ] );
            hi[ j ] = shared_load( &buf[ j ][ threadIdx.x ][ 1 ] );
         }
#pragma unroll
         for( int j = 0; j < N; j++ )
            there = there && (uint32_t) ( lo[ j ] >> 32 ) == number && (uint32_t) ( hi[ j ] >> 32 ) == number;
         if( __ballot( ! there ) == 0 || over )  // (looked once more after the time)
            break;
         over = wave_uniform( (int32_t) ( wall_clock64() - begin >= wait ) );
      }
      late = there ? 0 : 1;
#pragma unroll
      for( int j = 0; j < N; j++ )
         v[ j ] = __longlong_as_double( (long long) ( ( hi[ j ] << 32 ) | ( lo[ j ] & 0xffffffffu ) ) );
   }
   else
#pragma unroll
      for( int j = 0; j < N; j++ )
         v[ j ] = 0;
   wave_totals();
   late = wave_uniform( __syncthreads_or( late ) );
#pragma unroll
   for( int j = 0; j < N; j++ )
      v[ j ] = wave_uniform( block_total( j ) );
   __syncthreads();  // (sm may be written again)
   return ! late;
}

// A barrier: what a workgroup shared_stores before it is seen by all after it.
template< int T >
__device__ __forceinline__ bool grid_barrier( GridSlots* __restrict__ slots, uint32_t number, uint64_t wait, double* sm )
{
   double none[ 1 ] = { 0 };
   return grid_sum< T >( none, slots, number, wait, sm );
}

// grid_sum of `count` values whose wave totals are in sm[ j * T / 64 + wave ]
// already; the results in out[ j ] (LDS).  sm: kGridValues * T / 64 doubles.
// Each wave polls 64 workgroups' slots of one value at a time.
template< int T >
__device__ __forceinline__ bool grid_sum_many( int count, GridSlots* __restrict__ slots, uint32_t number, uint64_t wait,
                                               double* sm, double* out )
{
   constexpr int W = T / 64, kAtOnce = 4;
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, G = gridDim.x;
   shared_stores_done();
   __syncthreads();
   uint64_t( &buf )[ kGridValues ][ kGridMax ][ 2 ] = slots->word[ number & 1 ];
   if( (int) threadIdx.x < count ) {
      double r = 0;
#pragma unroll
      for( int i = 0; i < W; i++ )
         r += sm[ threadIdx.x * W + i ];
      const uint64_t bits = (uint64_t) __double_as_longlong( r );
      const uint64_t tag = (uint64_t) number << 32;
      shared_store( &buf[ threadIdx.x ][ blockIdx.x ][ 0 ], tag | ( bits & 0xffffffffu ) );
      shared_store( &buf[ threadIdx.x ][ blockIdx.x ][ 1 ], tag | ( bits >> 32 ) );
   }
   __syncthreads();  // (sm is read above and written below)
   const int quarters = ( G + 63 ) / 64, jobs = count * quarters;  // job: value job / quarters, slots of quarter job % quarters
   int late = 0;
   for( int job0 = w * kAtOnce; job0 < jobs; job0 += W * kAtOnce ) {
      uint64_t lo[ kAtOnce ], hi[ kAtOnce ];
      const uint64_t begin = wall_clock64();
      bool over = false;
      while( true ) {
         bool there = true;
#pragma unroll
         for( int u = 0; u < kAtOnce; u++ ) {
            const int job = min( job0 + u, jobs - 1 ), slot = min( job % quarters * 64 + lane, G - 1 );
            lo[ u ] = shared_load( &buf[ job / quarters ][ slot ][ 0 ] );
            hi[ u ] = shared_load( &buf[ job / quarters ][ slot ][ 1 ] );
         }
#pragma unroll
         for( int u = 0; u < kAtOnce; u++ )
            there = there && (uint32_t) ( lo[ u ] >> 32 ) == number && (uint32_t) ( hi[ u ] >> 32 ) == number;
         if( __ballot( ! there ) == 0 )
            break;
         if( over ) {
            late = 1;
            break;
         }
         over = wave_uniform( (int32_t) ( wall_clock64() - begin >= wait ) );
      }
#pragma unroll
      for( int u = 0; u < kAtOnce; u++ ) {
         const int job = job0 + u;
         if( job < jobs ) {  // (uniform over the wave)
            const bool mine = job % quarters * 64 + lane < G;
            double v = mine ? __longlong_as_double( (long long) ( ( hi[ u ] << 32 ) | ( lo[ u ] & 0xffffffffu ) ) ) : 0.0;
            v = group_sum< 64 >( v );
            if( lane == 0 )
               sm[ job ] = v;
         }
      }
   }
   late = wave_uniform( __syncthreads_or( late ) );
   if( (int) threadIdx.x < count ) {
      double r = 0;
      for( int q = 0; q < quarters; q++ )
         r += sm[ threadIdx.x * quarters + q ];
      out[ threadIdx.x ] = r;
   }
   __syncthreads();
   return ! late;
}

}  // namespace tnlmi
