// fused_cg.hip -- Jacobi-preconditioned CG with the dot products fused into
// the kernels that produce their operands, and the reliable-update
// mixed-precision CG built from the same kernels.
//
// One CG iteration (CG.hpp:60-105) is three launches:
//   spmv_dot   Ap = A p  and the partial sums of (Ap, p)            (SpMV epilogue)
//   cg_upd     alpha = s1/s2;  x += alpha p;  r -= alpha Ap;  z = r / d (not stored);
//              partial sums of (r, z) [and (r, r)]
//   cg_dir     beta, the residue, TNL's stopping rule (IterativeSolver.hpp:98-121)
//              and the iteration counter;  p = r / d + beta p
// Every block of a kernel reduces the previous kernels' partial sums (one
// per block: 1024 in the FP64 CG, 2048 in the mixed solves' FP32 iterations)
// in the same fixed order, so the scalars are identical in every block and
// from run to run.  The iteration state lives on the device, double-buffered
// by iteration parity (iteration k reads state k & 1, block 0 of its last
// kernel writes state (k + 1) & 1); every kernel returns at once when the
// state says the solver has stopped, so the host enqueues iterations in
// batches and reads the state back once per batch.
//
// Mixed precision (tnlmi_mixed_cg_solve): the same iteration in FP32 on the
// FP32- or BF16-valued matrix, FP32 vectors and accumulation, FP64 dot
// products; x is accumulated in FP64.  Reliable updates (residual
// replacement, Clark et al., "Solving lattice QCD systems of equations using
// mixed precision solvers on GPUs", 2010): when the FP32 residual has dropped
// by `delta` since the last update (or its estimate reaches the tolerance),
// x += correction and r = b - A x are recomputed in FP64 and the search
// direction p is kept, so the Krylov process is not restarted.  The stopping
// test is the FP64 true residual ||b - A x|| / ||b||
// (LinearResidueGetter.hpp:11-23).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <memory>
#include <string>
#include <type_traits>
#include <vector>

#include "blas1.hpp"
#include "grid_sum.hpp"
#include "krylov.hpp"
#include "segments.hpp"
#include "spmv.hpp"
#include "spmv_tile.hpp"

namespace tnlmi {
namespace {

// Blocks of a fused vector kernel = its number of partial sums: 1024 for the
// FP64 CG, 2048 for the FP32 iterations of the mixed solves (their FP32
// vectors move half the bytes per row, and twice the waves keep enough loads
// in flight: reliable BF16 CG on Poisson 256^3 0.281 against 0.320 s; the FP64
// CG measured 2 % slower with 2048, its blocks then summing twice the partials
// first).  kFB: the length of every partial-sum array.
constexpr int kFB = 2048;
template< typename T >
constexpr int blocks_of()
{
   return sizeof( T ) == 8 ? 1024 : 2048;
}
constexpr int kFB32 = blocks_of< float >();  // the mixed solve's kernels
constexpr int kFT = 256;
constexpr int kBatch = 8;  // iterations enqueued between two host reads of the state
static_assert( blocks_of< double >() % kXcds == 0 && blocks_of< float >() % kXcds == 0 && blocks_of< float >() <= kFB,
               "grids split evenly over the XCDs, partial sums fit their arrays" );

struct CgDev
{
   double s1, normb, res, beta;
   double rr, rr_max;  // mixed: (r, r) now and its maximum since the last update
   double s1_prev;     // mixed: (r, z) of the previous iteration (the beta denominator)
   double proj;        // mixed: (r, p) / (r, z) after a residual replacement
   int64_t it;         // TNL's currentIteration
   int32_t active;     // the iteration being run was admitted by nextIteration()
   int32_t s2zero;     // s2 == 0 ended the solve (CG.hpp:66-70)
   int32_t want_update;
   int32_t pad;
};

struct StopRule
{
   int64_t maxit, minit;
   double tol, div;
   int32_t kind = 0;  // residue: 0 TNL's sqrt((r, z)) / ||M^-1 b||, 1 ||r|| / ||b|| (the recurrence residual)
};

__device__ __forceinline__ bool check_next( const StopRule& R, double res, int64_t it )
{
   return ! ( isnan( res ) || it > R.maxit || ( res > R.div && it >= R.minit ) || ( res < R.tol && it >= R.minit ) );
}

// Sum of np partial sums in a fixed order; the same value in every block.
__device__ __forceinline__ double sum_parts( const double* __restrict__ part, double* sm, int np )
{
   double a = 0;
   for( int i = threadIdx.x; i < np; i += kFT )
      a += part[ i ];
   return block_sum< kFT >( a, sm );
}

// N partial-sum arrays at once: their loads in flight together and one pair
// of barriers, each total summed in the same order as sum_parts (so equal to
// it bit for bit).  sm holds N * kFT / 64 doubles.
template< int N >
__device__ __forceinline__ void sum_parts_n( const double* const ( &part )[ N ], double* sm, double ( &out )[ N ],
                                             int np )
{
   double a[ N ];
#pragma unroll
   for( int j = 0; j < N; j++ )
      a[ j ] = 0;
   for( int i = threadIdx.x; i < np; i += kFT )
#pragma unroll
      for( int j = 0; j < N; j++ )
         a[ j ] += part[ j ][ i ];
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
   for( int j = 0; j < N; j++ )
      a[ j ] = group_sum< 64 >( a[ j ] );
   __syncthreads();
   if( lane == 0 )
#pragma unroll
      for( int j = 0; j < N; j++ )
         sm[ j * ( kFT / 64 ) + w ] = a[ j ];
   __syncthreads();
#pragma unroll
   for( int j = 0; j < N; j++ ) {
      double r = 0;
#pragma unroll
      for( int i = 0; i < kFT / 64; i++ )
         r += sm[ j * ( kFT / 64 ) + i ];
      out[ j ] = wave_uniform( r );
   }
}

__device__ __forceinline__ void put_part( double v, double* sm, double* part )
{
   v = block_sum< kFT >( v, sm );
   if( threadIdx.x < 64 )
      part[ blockIdx.x ] = v;
}

// ---- fused SpMV + (Ap, p) partial sums (column-major Ellpack and
// SlicedEllpack; every other format runs its own SpMV kernel, then dot_part)
// Loops stride over the grid kU rows / elements at a time, so that every
// thread has kU independent loads in flight.
constexpr int kU = 4;

// Ellpack / SlicedEllpack, column-major: each thread R adjacent rows, whose
// slots are adjacent in every slot column (vector loads of R column indexes
// and R values), a full grid of row blocks placed XCD-contiguously (the rows
// that share x entries -- a stencil's neighbouring rows and planes -- are
// read by one XCD); one partial sum per block.  R divides the Ellpack row
// alignment (32) and the slice size, so a group never straddles a slice and
// its loads stay inside the padded storage (padding slots hold column -1).
template< typename E, int R >
struct Vec
{
   typedef E type __attribute__( ( ext_vector_type( R ) ) );
};
template< typename V, int R >
struct ValVec
{
   using type = typename Vec< V, R >::type;
   static __device__ __forceinline__ type load( const V* p ) { return __builtin_nontemporal_load( (const type*) p ); }
   template< typename T >
   static __device__ __forceinline__ T get( const type& v, int j )
   {
      return (T) v[ j ];
   }
};
template< int R >
struct ValVec< bf16, R >
{
   using type = typename Vec< uint16_t, R >::type;
   static __device__ __forceinline__ type load( const bf16* p )
   {
      return __builtin_nontemporal_load( (const type*) p );
   }
   template< typename T >
   static __device__ __forceinline__ T get( const type& v, int j )
   {
      return (T) bf16_to_float( v[ j ] );
   }
};

template< int R, typename V, typename T >
__global__ void __launch_bounds__( kFT ) spmv_dot_ell( SegView v, const int32_t* __restrict__ cols,
                                                       const V* __restrict__ vals, const T* __restrict__ p,
                                                       T* __restrict__ Ap, double* __restrict__ part,
                                                       const CgDev* __restrict__ st )
{
   using CV = typename Vec< int32_t, R >::type;
   using VV = ValVec< V, R >;
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   const int64_t blk = xcd_contiguous( blockIdx.x, gridDim.x );
   const int64_t r0 = ( blk * kFT + threadIdx.x ) * R;
   double acc = 0;
   if( r0 < v.n ) {
      int64_t g, stride;
      int32_t w;
      if( v.format == TNLMI_ELLPACK ) {
         g = r0;
         stride = v.ell_aligned;
         w = v.ell_width;
      }
      else {
         const int64_t sl = r0 / v.slice_size;
         g = v.slice_offsets[ sl ] + ( r0 - sl * v.slice_size );
         stride = v.slice_size;
         w = v.slice_seg_sizes[ sl ];
      }
      T y[ R ] = {};
      for( int32_t k = 0; k < w; k++, g += stride ) {
         const CV c = __builtin_nontemporal_load( (const CV*) ( cols + g ) );
         const typename VV::type a = VV::load( vals + g );
#pragma unroll
         for( int j = 0; j < R; j++ )
            if( c[ j ] >= 0 )
               y[ j ] += VV::template get< T >( a, j ) * p[ c[ j ] ];
      }
#pragma unroll
      for( int j = 0; j < R; j++ )
         if( r0 + j < v.n ) {
            Ap[ r0 + j ] = y[ j ];
            acc += (double) y[ j ] * (double) p[ r0 + j ];
         }
   }
   const double bs = block_sum< kFT >( acc, sm );
   if( threadIdx.x < 64 )
      part[ blk ] = bs;
}

// CSR with no row longer than kWholeRowMax (stencil matrices): the tiled CSR
// product in its one-launch form (each wavefront streams its TILE elements,
// every row is summed whole by its owner lane, left to right from 0) with the
// (Ap, p) partial sums in its epilogue: each lane adds v * p[r] for the rows
// it stores, one partial per workgroup.
template< typename V, typename T, int TILE >
__global__ void __launch_bounds__( kFT ) spmv_dot_csr( const int32_t* __restrict__ off,
                                                       const int32_t* __restrict__ tile_rows, int64_t tiles,
                                                       int64_t nnz, int64_t n, const int32_t* __restrict__ cols,
                                                       const V* __restrict__ vals, const T* __restrict__ p,
                                                       T* __restrict__ Ap, double* __restrict__ part,
                                                       const CgDev* __restrict__ st, int32_t tail_max )
{
   static_assert( kFT == 256, "four tile wavefronts per workgroup" );
   __shared__ T lds[ 4 ][ TILE + kWholeRowMax ];
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
   const int64_t blk = xcd_contiguous( blockIdx.x, gridDim.x );
   const int64_t t = blk * 4 + wave;
   double acc = 0;
   if( t < tiles )
      csr_tile< V, T, T, true, TILE >(
         off, n, cols, vals, p, t, tile_rows[ t ], tile_rows[ t + 1 ], nnz, lds[ wave ], lane,
         [ & ]( int64_t r, T v ) {
            Ap[ r ] = v;
            acc += (double) v * (double) p[ r ];
         },
         []( int64_t, T ) {}, tail_max );
   const double bs = block_sum< kFT >( acc, sm );
   if( threadIdx.x < 64 )
      part[ blk ] = bs;
}

// ---- 8-bit column codes: for a matrix whose entries take few distinct
// offsets column - row (a stencil: 7 for the 3D 7-point Laplacian), every
// slot stores a code into a dictionary of at most kCodes offsets instead of
// its 32-bit column (code kPadCode: padding), so the SpMV reads 1 byte of
// index per entry instead of 4.  The columns decoded are exactly the stored
// ones: results are bit-identical to the int32 kernel above.
constexpr int kCodes = 255;
constexpr uint8_t kPadCode = 255;
constexpr int kHash = 4096;  // open-addressing table of the distinct offsets
constexpr uint64_t kEmpty = ~0ull;

template< int R, typename V, typename T >
__global__ void __launch_bounds__( kFT ) spmv_dot_ell_code( SegView v, const uint8_t* __restrict__ codes,
                                                            const int32_t* __restrict__ dict, int32_t ndict,
                                                            const V* __restrict__ vals, const T* __restrict__ p,
                                                            T* __restrict__ Ap, double* __restrict__ part,
                                                            const CgDev* __restrict__ st )
{
   using CB = typename Vec< uint8_t, R >::type;
   using VV = ValVec< V, R >;
   __shared__ double sm[ kFT / 64 ];
   __shared__ int32_t sd[ kCodes ];
   if( ! st->active )
      return;
   for( int i = threadIdx.x; i < ndict; i += kFT )
      sd[ i ] = dict[ i ];
   __syncthreads();
   const int64_t blk = xcd_contiguous( blockIdx.x, gridDim.x );
   const int64_t r0 = ( blk * kFT + threadIdx.x ) * R;
   double acc = 0;
   if( r0 < v.n ) {
      int64_t g, stride;
      int32_t w;
      if( v.format == TNLMI_ELLPACK ) {
         g = r0;
         stride = v.ell_aligned;
         w = v.ell_width;
      }
      else {
         const int64_t sl = r0 / v.slice_size;
         g = v.slice_offsets[ sl ] + ( r0 - sl * v.slice_size );
         stride = v.slice_size;
         w = v.slice_seg_sizes[ sl ];
      }
      // kKU entries at a time: their codes and values, then their reads of p
      // (one contiguous read when the R rows share a code, as in the interior
      // of a stencil: the columns r0 + j + offset are consecutive), then the
      // products, added in entry order as the int32 kernel adds them
      constexpr int kKU = 8;
      T y[ R ] = {};
      for( int32_t k0 = 0; k0 < w; k0 += kKU ) {
         CB c[ kKU ];
         typename VV::type a[ kKU ];
#pragma unroll
         for( int u = 0; u < kKU; u++ ) {
            if( k0 + u < w ) {
               c[ u ] = __builtin_nontemporal_load( (const CB*) ( codes + g + u * stride ) );
               a[ u ] = VV::load( vals + g + u * stride );
            }
            else
#pragma unroll
               for( int j = 0; j < R; j++ )
                  c[ u ][ j ] = kPadCode;
         }
         T pv[ kKU ][ R ];
#pragma unroll
         for( int u = 0; u < kKU; u++ ) {
            const uint32_t c0 = c[ u ][ 0 ];
            bool same = true;
#pragma unroll
            for( int j = 1; j < R; j++ )
               same = same && c[ u ][ j ] == c0;
            if( same && c0 != kPadCode )
               __builtin_memcpy( pv[ u ], p + r0 + sd[ c0 ], sizeof( pv[ u ] ) );
            else
#pragma unroll
               for( int j = 0; j < R; j++ )
                  pv[ u ][ j ] = c[ u ][ j ] != kPadCode ? p[ r0 + j + sd[ c[ u ][ j ] ] ] : (T) 0;
         }
#pragma unroll
         for( int u = 0; u < kKU; u++ )
#pragma unroll
            for( int j = 0; j < R; j++ )
               if( c[ u ][ j ] != kPadCode )
                  y[ j ] += VV::template get< T >( a[ u ], j ) * pv[ u ][ j ];
         g += kKU * stride;
      }
#pragma unroll
      for( int j = 0; j < R; j++ )
         if( r0 + j < v.n ) {
            Ap[ r0 + j ] = y[ j ];
            acc += (double) y[ j ] * (double) p[ r0 + j ];
         }
   }
   const double bs = block_sum< kFT >( acc, sm );
   if( threadIdx.x < 64 )
      part[ blk ] = bs;
}

__device__ __forceinline__ uint32_t offset_hash( uint32_t key )
{
   return ( key * 2654435761u ) >> 20;  // Knuth's multiplicative hash, 12 bits
}

// the slot of row r, entry k, and the row width (Ellpack / SlicedEllpack, column-major)
__device__ __forceinline__ int64_t ell_slot( const SegView& v, int64_t r, int32_t k, int32_t* w )
{
   if( v.format == TNLMI_ELLPACK ) {
      *w = v.ell_width;
      return r + (int64_t) k * v.ell_aligned;
   }
   const int64_t sl = r / v.slice_size;
   *w = v.slice_seg_sizes[ sl ];
   return v.slice_offsets[ sl ] + ( r - sl * v.slice_size ) + (int64_t) k * v.slice_size;
}

// the distinct offsets column - row into the table (a few recent ones kept in
// registers; a plain read before the atomic); more than kCodes, or a full
// probe sequence, sets *overflow
__global__ void __launch_bounds__( kFT ) code_collect( SegView v, const int32_t* __restrict__ cols,
                                                       unsigned long long* table, int32_t* count, int32_t* overflow )
{
   uint32_t recent[ 4 ] = { 0, 0, 0, 0 };
   bool have[ 4 ] = { false, false, false, false };
   int next = 0;
   for( int64_t r = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; r < v.n; r += (int64_t) gridDim.x * blockDim.x ) {
      int32_t w = 0;
      ell_slot( v, r, 0, &w );
      for( int32_t k = 0; k < w; k++ ) {
         const int32_t c = cols[ ell_slot( v, r, k, &w ) ];
         if( c < 0 )
            continue;
         const uint32_t key = (uint32_t) ( c - (int32_t) r );
         bool seen = false;
#pragma unroll
         for( int i = 0; i < 4; i++ )
            seen |= have[ i ] && recent[ i ] == key;
         if( seen )
            continue;
         if( *(volatile int32_t*) overflow )
            return;
         uint32_t h = offset_hash( key );
         bool done = false;
         for( int probe = 0; probe < kHash && ! done; probe++, h = ( h + 1 ) & ( kHash - 1 ) ) {
            const unsigned long long cur = ( (volatile unsigned long long*) table )[ h ];
            if( cur == (unsigned long long) key ) {
               done = true;
               break;
            }
            if( cur != kEmpty )
               continue;
            const unsigned long long prev = atomicCAS( table + h, kEmpty, (unsigned long long) key );
            if( prev == kEmpty ) {
               if( atomicAdd( count, 1 ) >= kCodes )
                  atomicExch( overflow, 1 );
               done = true;
            }
            else if( prev == (unsigned long long) key )
               done = true;
         }
         if( ! done ) {
            atomicExch( overflow, 1 );
            return;
         }
         recent[ next ] = key;
         have[ next ] = true;
         next = ( next + 1 ) & 3;
      }
   }
}

// codes[slot] = code of the slot's offset (slots of padding keep kPadCode)
__global__ void __launch_bounds__( kFT ) code_encode( SegView v, const int32_t* __restrict__ cols,
                                                      const unsigned long long* __restrict__ table,
                                                      const uint8_t* __restrict__ code_of, uint8_t* __restrict__ codes )
{
   for( int64_t r = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; r < v.n; r += (int64_t) gridDim.x * blockDim.x ) {
      int32_t w = 0;
      ell_slot( v, r, 0, &w );
      for( int32_t k = 0; k < w; k++ ) {
         const int64_t g = ell_slot( v, r, k, &w );
         const int32_t c = cols[ g ];
         if( c < 0 )
            continue;
         const uint32_t key = (uint32_t) ( c - (int32_t) r );
         uint32_t h = offset_hash( key );
         for( int probe = 0; probe < kHash; probe++, h = ( h + 1 ) & ( kHash - 1 ) )
            if( table[ h ] == (unsigned long long) key ) {
               codes[ g ] = code_of[ h ];
               break;
            }
      }
   }
}

// The SpMV kernels' nin block partial sums folded, in order, into the
// gridDim.x partial sums the following kernels read.
__global__ void __launch_bounds__( kFT ) fold_parts( const double* __restrict__ in, int64_t nin,
                                                     double* __restrict__ out, const CgDev* __restrict__ st )
{
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   const int64_t chunk = ( nin + gridDim.x - 1 ) / gridDim.x;
   const int64_t b = blockIdx.x * chunk, e = min( nin, b + chunk );
   double a = 0;
   for( int64_t i = b + threadIdx.x; i < e; i += kFT )
      a += in[ i ];
   put_part( a, sm, out );
}

// any other format: the format's own SpMV kernel, then this partial dot
template< typename T >
__global__ void __launch_bounds__( kFT ) dot_part( int64_t n, const T* __restrict__ a, const T* __restrict__ b,
                                                   double* __restrict__ part, const CgDev* __restrict__ st )
{
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   double acc = 0;
   for( int64_t i0 = (int64_t) blockIdx.x * kFT + threadIdx.x; i0 < n; i0 += kU * (int64_t) gridDim.x * kFT )
#pragma unroll
      for( int u = 0; u < kU; u++ ) {
         const int64_t i = i0 + u * (int64_t) gridDim.x * kFT;
         if( i < n )
            acc += (double) a[ i ] * (double) b[ i ];
      }
   put_part( acc, sm, part );
}

// ---- alpha = s1 / (Ap, p);  x += alpha p;  r -= alpha Ap;  partial sums of
// (r, z) and, for the mixed solver, (r, r);  z = r / d
template< typename T, typename X, typename D >
__global__ void __launch_bounds__( kFT ) cg_upd( int64_t n, const double* __restrict__ part1, T* __restrict__ r,
                                                 const T* __restrict__ p, const T* __restrict__ Ap,
                                                 X* __restrict__ x, const D* __restrict__ d,
                                                 double* __restrict__ part2, double* __restrict__ part3,
                                                 const CgDev* __restrict__ st )
{
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   const double s2 = sum_parts( part1, sm, (int) gridDim.x );  // the producers' grid is this grid
   if( s2 == 0.0 )
      return;  // cg_dir ends the solve
   const T alpha = (T) ( st->s1 / s2 );
   double a2 = 0, a3 = 0;
   for( int64_t i0 = (int64_t) blockIdx.x * kFT + threadIdx.x; i0 < n; i0 += kU * (int64_t) gridDim.x * kFT )
#pragma unroll
      for( int u = 0; u < kU; u++ ) {
         const int64_t i = i0 + u * (int64_t) gridDim.x * kFT;
         if( i < n ) {
            const T pi = p[ i ];
            x[ i ] += (X) ( alpha * pi );
            const T ri = r[ i ] - alpha * Ap[ i ];
            r[ i ] = ri;
            const T zi = d ? ri / (T) d[ i ] : ri;
            a2 += (double) ri * (double) zi;
            a3 += (double) ri * (double) ri;
         }
      }
   put_part( a2, sm, part2 );
   if( part3 )
      put_part( a3, sm, part3 );
}

// ---- the end of one iteration: every block computes the scalars from the
// partial sums (the same values in every block), block 0 writes the next
// state, every block updates its share of p = z + beta p.
// FP64 CG: residue sqrt(s1) / normb and TNL's stopping rule
// (IterativeSolver.hpp:98-121; nextIteration() counts every check).
template< typename T, typename D >
__global__ void __launch_bounds__( kFT ) cg_dir( int64_t n, const double* __restrict__ part1,
                                                 const double* __restrict__ part2, const double* __restrict__ part3,
                                                 const T* __restrict__ r, const D* __restrict__ d, T* __restrict__ p,
                                                 const CgDev* __restrict__ cur, CgDev* __restrict__ nxt, StopRule R )
{
   __shared__ double sm[ 3 * ( kFT / 64 ) ];
   const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
   if( ! cur->active ) {
      if( lead )
         *nxt = *cur;
      return;
   }
   double t[ 3 ] = { 0, 0, 0 };
   if( R.kind == 1 ) {
      double t3[ 3 ];
      sum_parts_n< 3 >( { part1, part2, part3 }, sm, t3, (int) gridDim.x );
      t[ 0 ] = t3[ 0 ], t[ 1 ] = t3[ 1 ], t[ 2 ] = t3[ 2 ];
   }
   else {
      double t2[ 2 ];
      sum_parts_n< 2 >( { part1, part2 }, sm, t2, (int) gridDim.x );
      t[ 0 ] = t2[ 0 ], t[ 1 ] = t2[ 1 ];
   }
   const double s2 = t[ 0 ];
   const double s1n = t[ 1 ];
   if( s2 == 0.0 ) {
      if( lead ) {
         *nxt = *cur;
         nxt->res = 0.0;
         nxt->s2zero = 1;
         nxt->active = 0;
      }
      return;
   }
   const double s1 = cur->s1;
   const double beta = s1 == 0.0 ? 0.0 : s1n / s1;
   const double res = sqrt( R.kind == 1 ? t[ 2 ] : s1n ) / cur->normb;
   const bool go = check_next( R, res, cur->it );
   if( lead ) {
      *nxt = *cur;
      nxt->s1 = s1n;
      nxt->beta = beta;
      nxt->res = res;
      nxt->active = go ? 1 : 0;
      nxt->it = cur->it + 1;
   }
   if( ! go )
      return;
   const T tb = (T) beta;
   for( int64_t i0 = (int64_t) blockIdx.x * kFT + threadIdx.x; i0 < n; i0 += kU * (int64_t) gridDim.x * kFT )
#pragma unroll
      for( int u = 0; u < kU; u++ ) {
         const int64_t i = i0 + u * (int64_t) gridDim.x * kFT;
         if( i < n ) {
            const T ri = r[ i ];
            p[ i ] = ( d ? ri / (T) d[ i ] : ri ) + tb * p[ i ];
         }
      }
}

// Mixed: the FP32 iteration's end; asks for a reliable update (and leaves p
// to it) when the residual has dropped by delta since the last update, when
// its estimate reaches the tolerance, or when the iteration budget is spent.
__global__ void __launch_bounds__( kFT ) mx_dir( int64_t n, const double* __restrict__ part1,
                                                 const double* __restrict__ part2, const double* __restrict__ part3,
                                                 const float* __restrict__ r, const float* __restrict__ d,
                                                 float* __restrict__ p, const CgDev* __restrict__ cur,
                                                 CgDev* __restrict__ nxt, double delta2, double tol, int64_t maxit )
{
   __shared__ double sm[ 3 * ( kFT / 64 ) ];
   const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
   if( ! cur->active ) {
      if( lead )
         *nxt = *cur;
      return;
   }
   double t[ 3 ];
   sum_parts_n< 3 >( { part1, part2, part3 }, sm, t, (int) gridDim.x );
   const double s2 = t[ 0 ], s1n = t[ 1 ], rr = t[ 2 ];
   const double s1 = cur->s1;
   const int64_t it = cur->it + 1;
   const double beta = s1 == 0.0 ? 0.0 : s1n / s1;
   const double rr_max = fmax( cur->rr_max, rr );
   const bool want = s2 == 0.0 || rr < delta2 * rr_max || sqrt( rr ) < tol * cur->normb || it >= maxit || isnan( rr );
   if( lead ) {
      *nxt = *cur;
      nxt->it = it;
      nxt->s1_prev = s1;
      if( s2 != 0.0 ) {
         nxt->s1 = s1n;
         nxt->beta = beta;
         nxt->rr = rr;
         nxt->rr_max = rr_max;
      }
      if( want ) {
         nxt->want_update = 1;
         nxt->active = 0;
      }
   }
   if( want )
      return;
   const float tb = (float) beta;
   for( int64_t i0 = (int64_t) blockIdx.x * kFT + threadIdx.x; i0 < n; i0 += kU * (int64_t) gridDim.x * kFT )
#pragma unroll
      for( int u = 0; u < kU; u++ ) {
         const int64_t i = i0 + u * (int64_t) gridDim.x * kFT;
         if( i < n )
            p[ i ] = r[ i ] / d[ i ] + tb * p[ i ];
      }
}

// ---- many iterations in one launch, for matrices of at most kGridRows rows.
// Below about a million rows an iteration's four launches (5 us each, whatever
// the size) take longer than its work.  Here the whole grid stays resident:
// every thread keeps ROWS rows of x, r, p, d (and with KEEP the rows' matrix
// entries) in registers, and an iteration's two reductions are grid sums.  What
// other workgroups read goes through memory: z = r / d after the update, and
// the direction in two buffers in turn.  A row's product gathers z and the old
// direction and forms p = z + beta p_old itself (the same operation its owner
// does), so the new direction needs no exchange of its own.
// A solve to 1e-10, per iteration, against launch by launch: 120 x 97 diffusion
// (11,640 rows) 7.7 against 20.8 us, 500 x 490 12.1 against 24.8 us, 80 x 81 x 79
// 22.8 against 33.8 us, 100 x 101 x 99 (999,900 rows) 35.8 against 47.2 us; with
// FP32 vectors and BF16 values 36.1 against 45.9 us there.  (1,024 threads and 4
// rows each: 512 threads and 8 rows took 41.4 us; dropping the L2 once per sum
// instead of reading past it 42.8 us.)
constexpr int kGridWidth = 8;  // entries per row that KEEP holds

template< typename T, typename X >
struct GridCg
{
   int64_t n, stride;         // rows; of an Ellpack slot column
   int32_t w;                 // Ellpack width
   const int32_t* cols;
   const void* vals;
   T* r;
   T* p[ 2 ];                 // the direction, in turn; in p[ 0 ] when a launch begins or ends
   T* z;
   X* x;
   const void* d;             // Jacobi diagonal (NULL: none)
   CgDev* st;
   GridSlots* slots;
   uint64_t wait;             // for a workgroup in a grid sum
   uint32_t number;           // of the first grid sum
   int32_t most;              // iterations at most
   int32_t* late;             // a grid sum was given up
   StopRule R;
   double delta2, tol;        // mixed
   int64_t maxit;
};

template< typename V, typename T, typename X, typename D, int THREADS, int ROWS, bool KEEP, bool MIXED >
__global__ void __launch_bounds__( THREADS ) grid_cg( GridCg< T, X > a )
{
   __shared__ double sm[ 2 * THREADS / 64 ];
   __shared__ T own[ THREADS * ROWS ];
   const CgDev st0 = *a.st;
   if( ! st0.active )
      return;
   const int32_t base = (int32_t) ( blockIdx.x * ( THREADS * ROWS ) );  // (n <= kGridRows)
   const int64_t r0 = base + threadIdx.x;
   const V* __restrict__ vals = (const V*) a.vals;
   const D* __restrict__ diag = (const D*) a.d;
   T r[ ROWS ], p[ ROWS ], d[ ROWS ], z[ ROWS ];
   X x[ ROWS ];
   int32_t kc[ KEEP ? ROWS : 1 ][ kGridWidth ];
   V kv[ KEEP ? ROWS : 1 ][ kGridWidth ];
#pragma unroll
   for( int j = 0; j < ROWS; j++ ) {
      const int64_t i = r0 + j * THREADS;
      const bool in = i < a.n;
      r[ j ] = in ? a.r[ i ] : (T) 0;
      p[ j ] = in ? a.p[ 0 ][ i ] : (T) 0;
      x[ j ] = in ? a.x[ i ] : (X) 0;
      d[ j ] = in && diag ? (T) diag[ i ] : (T) 1;
      z[ j ] = 0;
      if( KEEP )
#pragma unroll
         for( int k = 0; k < kGridWidth; k++ ) {
            const bool there = in && k < a.w;
            kc[ j ][ k ] = there ? a.cols[ k * a.stride + i ] : -1;
            kv[ j ][ k ] = there ? vals[ k * a.stride + i ] : V{};
         }
   }
   double s1 = st0.s1, s1_prev = st0.s1_prev, beta = st0.beta, res = st0.res, rr = st0.rr, rr_max = st0.rr_max;
   int64_t it = st0.it;
   uint32_t number = a.number;
   int32_t done = 0;
   bool first = true, s2zero = false, want = false, go = true;
   int cur = 0;  // buffer of the direction the gathers read
   while( true ) {
      const T tb = (T) beta;
      const T* pg = a.p[ cur ];
      T* pn = a.p[ cur ^ 1 ];
      // this workgroup's rows of the new direction
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         const int64_t i = r0 + j * THREADS;
         if( ! first )
            p[ j ] = z[ j ] + tb * p[ j ];
         own[ j * THREADS + threadIdx.x ] = p[ j ];
         if( i < a.n )
            shared_store( pn + i, p[ j ] );
      }
      __syncthreads();
      // the new direction at column c
      auto direction = [ & ]( int32_t c ) -> T {
         const uint32_t l = (uint32_t) ( c - base );
         if( l < (uint32_t) ( THREADS * ROWS ) )
            return own[ l ];
         const T po = shared_load( pg + c );
         return first ? po : shared_load( a.z + c ) + tb * po;
      };
      T y[ ROWS ];
      double part[ 1 ] = { 0 };
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         const int64_t i = r0 + j * THREADS;
         y[ j ] = 0;
         if( KEEP ) {
            T g[ kGridWidth ];
#pragma unroll
            for( int k = 0; k < kGridWidth; k++ )
               g[ k ] = kc[ j ][ k ] >= 0 ? direction( kc[ j ][ k ] ) : (T) 0;
#pragma unroll
            for( int k = 0; k < kGridWidth; k++ )
               if( kc[ j ][ k ] >= 0 )
                  y[ j ] += load_val< V, T >( &kv[ j ][ k ], 0 ) * g[ k ];
         }
         else if( i < a.n )
            for( int32_t k0 = 0; k0 < a.w; k0 += kGridWidth ) {
               int32_t c[ kGridWidth ];
               T v[ kGridWidth ], g[ kGridWidth ];
#pragma unroll
               for( int k = 0; k < kGridWidth; k++ ) {
                  const bool there = k0 + k < a.w;
                  c[ k ] = there ? a.cols[ ( k0 + k ) * a.stride + i ] : -1;
                  v[ k ] = there ? load_val< V, T >( vals, ( k0 + k ) * a.stride + i ) : (T) 0;
               }
#pragma unroll
               for( int k = 0; k < kGridWidth; k++ )
                  g[ k ] = c[ k ] >= 0 ? direction( c[ k ] ) : (T) 0;
#pragma unroll
               for( int k = 0; k < kGridWidth; k++ )
                  if( c[ k ] >= 0 )
                     y[ j ] += v[ k ] * g[ k ];
            }
         if( i < a.n )
            part[ 0 ] += (double) y[ j ] * (double) p[ j ];
      }
      first = false;
      cur ^= 1;
      if( ! grid_sum< THREADS >( part, a.slots, number++, a.wait, sm ) ) {
         if( threadIdx.x == 0 )
            *a.late = 1;
         return;
      }
      const double s2 = part[ 0 ];
      // x += alpha p;  r -= alpha Ap;  z = r / d
      double sums[ 2 ] = { 0, 0 };
      if( s2 != 0.0 ) {
         const T alpha = (T) ( s1 / s2 );
#pragma unroll
         for( int j = 0; j < ROWS; j++ ) {
            const int64_t i = r0 + j * THREADS;
            x[ j ] += (X) ( alpha * p[ j ] );
            r[ j ] = r[ j ] - alpha * y[ j ];
            z[ j ] = diag ? r[ j ] / d[ j ] : r[ j ];
            if( i < a.n ) {
               shared_store( a.z + i, z[ j ] );
               sums[ 0 ] += (double) r[ j ] * (double) z[ j ];
               sums[ 1 ] += (double) r[ j ] * (double) r[ j ];
            }
         }
         if( ! grid_sum< THREADS >( sums, a.slots, number++, a.wait, sm ) ) {
            if( threadIdx.x == 0 )
               *a.late = 1;
            return;
         }
      }
      const double s1n = sums[ 0 ];
      done++;
      if( MIXED ) {  // as mx_dir
         rr_max = s2 != 0.0 ? fmax( rr_max, sums[ 1 ] ) : rr_max;
         it++;
         want = s2 == 0.0 || sums[ 1 ] < a.delta2 * rr_max || sqrt( sums[ 1 ] ) < a.tol * st0.normb || it >= a.maxit
                || isnan( sums[ 1 ] );
         s1_prev = s1;
         if( s2 != 0.0 ) {
            beta = s1 == 0.0 ? 0.0 : s1n / s1;
            s1 = s1n;
            rr = sums[ 1 ];
         }
         go = ! want;
      }
      else {  // as cg_dir
         if( s2 == 0.0 ) {
            s2zero = true;
            res = 0.0;
            go = false;
            break;
         }
         beta = s1 == 0.0 ? 0.0 : s1n / s1;
         s1 = s1n;
         res = sqrt( a.R.kind == 1 ? sums[ 1 ] : s1n ) / st0.normb;
         go = check_next( a.R, res, it );
         it++;
      }
      if( ! go || done >= a.most )
         break;
   }
   // the next launch starts from an explicit direction
   if( go )
#pragma unroll
      for( int j = 0; j < ROWS; j++ )
         p[ j ] = z[ j ] + (T) beta * p[ j ];
#pragma unroll
   for( int j = 0; j < ROWS; j++ ) {
      const int64_t i = r0 + j * THREADS;
      if( i < a.n ) {
         a.x[ i ] = x[ j ];
         a.r[ i ] = r[ j ];
         a.p[ 0 ][ i ] = p[ j ];
      }
   }
   if( blockIdx.x == 0 && threadIdx.x == 0 ) {
      CgDev s = st0;
      s.s1 = s1;
      s.s1_prev = s1_prev;
      s.beta = beta;
      s.res = res;
      s.rr = rr;
      s.rr_max = rr_max;
      s.it = it;
      s.s2zero = s2zero ? 1 : 0;
      s.want_update = want ? 1 : 0;
      s.active = go ? 1 : 0;
      *a.st = s;
   }
}

// ---- which matrices a resident launch takes.  What a workgroup reads of another's
// rows goes past the L2, so columns spread over the whole matrix cost more there
// than in the launches, the more the larger the vectors: CG on uniformly random
// columns, resident against launch by launch, per iteration: 100,000 rows of 24
// 35.5 / 43.5 us, 200,000 of 12 39.1 / 39.6, 400,000 of 4 36.4 / 37.4, 524,288 of 3
// 39.7 / 38.3, 1,000,000 of 2 50.7 / 47.9 and of 12 279 / 123 us.  What counts is the lines
// that a wave's lanes ask for (neighbouring rows' neighbouring columns share
// one) beyond the next workgroups' rows: the 27-point grid of 80^3 has 0.76 M and takes
// 48.7 / 61.5 us, of 100^3 1.58 M and 103 / 92 us.  The next workgroups' rows are mostly
// found in the L2 all the same: 1,000,000 rows of 12 columns within 3,000 rows 59.9 /
// 92.3 us, within 30,000 (16 columns) 339 / 131 us.  The line is lines * rows = 4.5e11 in FP64, in the FP32 iteration
// 9e11 (7e11 against the launches on BF16 values, whose columns are codes): rows
// of 4, random, 524,288 26.1 / 31.3, 1,000,000 66.5 / 50.6 us; 27-point 100^3 56.2 / 61.5 us
// in FP32, 72.5 / 57.9 in BF16.  Below 131,073 rows the launches are never faster.
constexpr double kFar64 = 4.5e11, kFar32 = 9e11, kFarBf16 = 7e11;
constexpr int kFarGroups = 64;  // groups of 64 rows looked at

// The lines of LINE entries of a vector that one product over the slots asks
// from rows beyond the next `block` rows' on either side, from kFarGroups of the groups.
template< int LINE >
__global__ void __launch_bounds__( 1024 ) far_lines( int64_t n, int64_t stride, int32_t w, const int32_t* __restrict__ cols,
                                                     int32_t block, double* __restrict__ out )
{
   __shared__ int32_t sm[ 16 ];
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   const int64_t groups = ( n + 63 ) / 64;
   const int32_t every = ( w + 31 ) / 32;  // slots
   const int32_t slots = ( w + every - 1 ) / every;
   int32_t count = 0;
   for( int g = wave; g < kFarGroups; g += 16 ) {
      const int64_t r = groups * g / kFarGroups * 64 + lane;
      for( int32_t k0 = 0; k0 < slots; k0 += 8 ) {
         int32_t c[ 8 ];
#pragma unroll
         for( int u = 0; u < 8; u++ )
            c[ u ] = r < n && k0 + u < slots ? cols[ (int64_t) ( k0 + u ) * every * stride + r ] : -1;
#pragma unroll
         for( int u = 0; u < 8; u++ ) {
            const int32_t line = c[ u ] >= 0 && abs( c[ u ] / block - (int32_t) r / block ) > 1 ? c[ u ] / LINE : -1;
            const int32_t before = __shfl_up( line, 1, 64 );
            count += line >= 0 && ( lane == 0 || line != before ) ? 1 : 0;
         }
      }
   }
   count = group_sum< 64 >( count );
   if( lane == 0 )
      sm[ wave ] = count;
   __syncthreads();
   if( threadIdx.x == 0 ) {
      double t = 0;
      for( int i = 0; i < 16; i++ )
         t += sm[ i ];
      *out = t * ( (double) groups / kFarGroups ) * ( (double) w / slots );
   }
}

constexpr int64_t kGridRows = int64_t( kGridMax ) * 1024 * 4;
constexpr int32_t kGridIterations = 4096;  // per launch

// One launch of grid_cg, in the caller's resident_turn(); false: this case is none
// for it (nothing was launched).
template< typename V, typename T, typename X, typename D, bool MIXED >
bool grid_cg_launch( const GridCg< T, X >& a, hipStream_t s )
{
   auto go = [ & ]( auto kernel, int threads, int rows ) {
      GridCg< T, X > arg = a;
      void* args[] = { &arg };
      return resident_launch( (const void*) kernel, ceil_div( a.n, (int64_t) threads * rows ), threads, args, s );
   };
   const bool keep = a.w <= kGridWidth;
   const int64_t per_thread = ceil_div( a.n, (int64_t) kGridMax * 1024 );
   if( a.n <= (int64_t) kGridMax * 256 )
      return keep ? go( grid_cg< V, T, X, D, 256, 1, true, MIXED >, 256, 1 )
                  : go( grid_cg< V, T, X, D, 256, 1, false, MIXED >, 256, 1 );
   if( a.n <= (int64_t) kGridMax * 512 )
      return keep ? go( grid_cg< V, T, X, D, 512, 1, true, MIXED >, 512, 1 )
                  : go( grid_cg< V, T, X, D, 512, 1, false, MIXED >, 512, 1 );
   if( per_thread <= 1 )
      return keep ? go( grid_cg< V, T, X, D, 1024, 1, true, MIXED >, 1024, 1 )
                  : go( grid_cg< V, T, X, D, 1024, 1, false, MIXED >, 1024, 1 );
   if( per_thread <= 2 )
      return go( grid_cg< V, T, X, D, 1024, 2, false, MIXED >, 1024, 2 );
   if( per_thread <= 4 )
      return go( grid_cg< V, T, X, D, 1024, 4, false, MIXED >, 1024, 4 );
   return false;
}

// ---- row masks: the iteration of large matrices whose entries take few
// distinct (column - row, value) pairs -- a constant-coefficient stencil: 7 for
// the 3D 7-point Laplacian.  The pairs travel as kernel arguments and a row is
// a bit mask over them (1 or 2 bytes instead of 12 per entry), so the product
// costs little more than reading p, and an iteration forms it twice instead of
// writing and reading A p:
//   mk_dot   partial sums of (A p, p)                                   reads p
//   mk_upd   r -= alpha A p, partial sums of (r, z)                     reads p, r; writes r
//   mk_dir   x += alpha p, then cg_dir's end of the iteration           reads r, p, x; writes p, x
// 9 vectors of n (10 and 11 with a diagonal that varies) instead of 13 and
// the matrix.  A row's entries are added in their order with the stored values,
// so products are those of spmv_dot_ell bit for bit.
// Poisson 256^3, per iteration: FP64 68 + 122 + 105 us against 356 + 5 + 162 + 109
// us on the stored matrix (a solve 321 against 687 ms); reliable BF16 27 + 46 + 52
// against 127 + 5 + 72 + 44 us (148 against 283 ms).  The products' 7 reads of p
// per row (L1 hits mostly) bound mk_dot: 65 us where its 151 MB take 30 at copy
// speed.  16 bytes of rows per thread (2 FP64, 4 FP32) are best: FP64 91 us with 1
// row and 76 with 4.
constexpr int kPairs = 16;
constexpr int kPairHash = 256;
// Below half a million rows an iteration takes the same with and without masks (5-point
// SlicedEllpack 300^2 16.0 us either way; 900^2 19.8 against 28.4), and finding the pairs
// costs a short solve more than it saves (0.1 of 0.29 ms).  The mixed solver would
// collect the column codes instead, which takes longer (100 iterations on 300^2 3.9 against
// 5.2 ms).
constexpr int64_t kMaskRows = 1 << 19, kMaskRowsMixed = 1 << 12;

template< typename T >
struct PairDict
{
   int32_t off[ kPairs ];
   T val[ kPairs ];
};

struct PairTable  // the pairs found so far
{
   unsigned long long key[ kPairHash ];  // mix of the pair (kEmpty: free)
   unsigned long long val[ kPairHash ];  // value bits
   int32_t off[ kPairHash ];
   int32_t count, reject;
};

template< typename V >
__device__ __forceinline__ uint64_t value_bits( const V* vals, int64_t g )
{
   uint64_t b = 0;
   __builtin_memcpy( &b, vals + g, sizeof( V ) );
   return b;
}
__device__ __forceinline__ uint64_t pair_mix( int32_t off, uint64_t bits )
{
   uint64_t z = bits * 0x9e3779b97f4a7c15ull + (uint32_t) off;
   z = ( z ^ ( z >> 29 ) ) * 0xbf58476d1ce4e5b9ull;
   z ^= z >> 32;
   return z == kEmpty ? 0 : z;
}

// The pairs of the first `rows` rows into the table.  A matrix of many pairs has to
// be refused at once: with half a million threads probing a full table a refusal took
// 48 ms on 128^3 rows.  So no thread probes past kPairs occupied entries or
// after the refusal, and a first launch over few rows refuses before most threads
// start (0.1 ms; 0.15 ms where only the last rows differ).
template< typename V >
__global__ void __launch_bounds__( kFT ) pairs_collect( SegView v, const int32_t* __restrict__ cols,
                                                        const V* __restrict__ vals, PairTable* table, int64_t rows )
{
   __shared__ unsigned long long seen[ kFT ];  // by the key's low bits: pairs that are in the table
   seen[ threadIdx.x ] = kEmpty;
   __syncthreads();
   constexpr int kEntries = 8;  // loaded together
   for( int64_t r = (int64_t) blockIdx.x * kFT + threadIdx.x; r < rows; r += (int64_t) gridDim.x * kFT ) {
      const int32_t reject = shared_load( &table->reject );
      int32_t w = 0;
      ell_slot( v, r, 0, &w );
      for( int32_t k0 = 0; k0 < w; k0 += kEntries ) {
         int32_t c[ kEntries ];
         uint64_t bits[ kEntries ];
#pragma unroll
         for( int u = 0; u < kEntries; u++ ) {
            const int64_t g = ell_slot( v, r, min( k0 + u, w - 1 ), &w );
            c[ u ] = cols[ g ];
            bits[ u ] = value_bits( vals, g );
         }
         if( reject )
            return;
         uint32_t fresh = 0;  // entries that this workgroup has not seen
#pragma unroll
         for( int u = 0; u < kEntries; u++ ) {
            const unsigned long long key = pair_mix( c[ u ] - (int32_t) r, bits[ u ] );
            if( c[ u ] >= 0
                && __hip_atomic_load( seen + ( key & ( kFT - 1 ) ), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP )
                      != key )
               fresh |= 1u << u;
         }
         if( ! fresh )
            continue;
         for( int u = 0; u < kEntries; u++ ) {  // (rarely)
            if( ! ( fresh >> u & 1 ) )
               continue;
            if( shared_load( &table->reject ) )
               return;
            const int64_t g = ell_slot( v, r, min( k0 + u, w - 1 ), &w );
            const int32_t off = cols[ g ] - (int32_t) r;
            const uint64_t bit = value_bits( vals, g );
            const unsigned long long key = pair_mix( off, bit );
            bool placed = false;
            for( int probe = 0, h = (int) ( key >> 40 ) & ( kPairHash - 1 ); probe <= kPairs && ! placed;
                 probe++, h = ( h + 1 ) & ( kPairHash - 1 ) ) {
               // (a read first: one atomic by every thread at the same pair would queue up)
               unsigned long long prev = shared_load( &table->key[ h ] );
               if( prev == kEmpty )
                  prev = atomicCAS( &table->key[ h ], kEmpty, key );
               if( prev == kEmpty ) {
                  table->val[ h ] = bit;
                  table->off[ h ] = off;
                  if( atomicAdd( &table->count, 1 ) >= kPairs )
                     shared_store( &table->reject, 1 );
               }
               placed = prev == kEmpty || prev == key;
            }
            if( ! placed )
               shared_store( &table->reject, 1 );
            __hip_atomic_store( seen + ( key & ( kFT - 1 ) ), key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
         }
      }
   }
}

struct RawDict  // the pairs by offset, then value bits
{
   int32_t count;
   int32_t off[ kPairs ];
   uint64_t bits[ kPairs ];
};

// mask[r] = bit q for each entry that is pair q; a row whose entries are not
// pairs in increasing order (another order of the sum, a repeated column, a
// pair that shares another's key) rejects the matrix
template< typename V, typename M >
__global__ void __launch_bounds__( kFT ) pairs_encode( SegView v, const int32_t* __restrict__ cols,
                                                       const V* __restrict__ vals, RawDict D, M* __restrict__ mask,
                                                       int64_t rows, int32_t* reject )
{
   for( int64_t r = (int64_t) blockIdx.x * kFT + threadIdx.x; r < rows; r += (int64_t) gridDim.x * kFT ) {
      uint32_t m = 0;
      if( r < v.n ) {
         int32_t w = 0, last = -1;
         ell_slot( v, r, 0, &w );
         for( int32_t k = 0; k < w; k++ ) {
            const int64_t g = ell_slot( v, r, k, &w );
            const int32_t c = cols[ g ];
            if( c < 0 )
               continue;
            const uint64_t bits = value_bits( vals, g );
            int32_t q = -1;
#pragma unroll
            for( int i = 0; i < kPairs; i++ )
               if( i < D.count && D.off[ i ] == c - (int32_t) r && D.bits[ i ] == bits )
                  q = i;
            if( q <= last || ( last >= 0 && D.off[ q ] == D.off[ last ] ) ) {
               *reject = 1;
               break;
            }
            m |= 1u << q;
            last = q;
         }
      }
      mask[ r ] = (M) m;
   }
}

// is d one value throughout (bit for bit)?
__global__ void __launch_bounds__( kFT ) varies( int64_t n, const double* __restrict__ d, int32_t* __restrict__ out )
{
   const uint64_t first = (uint64_t) __double_as_longlong( d[ 0 ] );
   bool other = false;
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT )
      other = other || (uint64_t) __double_as_longlong( d[ i ] ) != first;
   if( other )
      *out = 1;
}

// R rows of A p from row r0 (p has room for every pair's offset at both ends)
template< int R, int NP, typename M, typename T >
__device__ __forceinline__ void mask_rows( const PairDict< T >& D, const M* __restrict__ mask, const T* __restrict__ p,
                                           int64_t r0, T ( &y )[ R ] )
{
   typename Vec< M, R >::type m = *(const typename Vec< M, R >::type*) ( mask + r0 );
   T g[ NP ][ R ];
#pragma unroll
   for( int k = 0; k < NP; k++ )
      __builtin_memcpy( g[ k ], p + ( r0 + D.off[ k ] ), sizeof( g[ k ] ) );
#pragma unroll
   for( int j = 0; j < R; j++ )
      y[ j ] = 0;
#pragma unroll
   for( int k = 0; k < NP; k++ )
#pragma unroll
      for( int j = 0; j < R; j++ ) {
         const T t = y[ j ] + D.val[ k ] * g[ k ][ j ];
         y[ j ] = m[ j ] >> k & 1 ? t : y[ j ];
      }
}

// The tiles of kFT * R rows in the order of the sweep: each XCD has one
// contiguous range, which its workgroups go through side by side (the planes a
// row reads are then in the XCD's L2).
template< int R, typename F >
__device__ __forceinline__ void sweep( int64_t n, F&& f )
{
   const int64_t tiles = ( n + kFT * R - 1 ) / ( kFT * R );
   const int64_t x = blockIdx.x % kXcds, j = blockIdx.x / kXcds, per = gridDim.x / kXcds;
   const int64_t t0 = tiles * x / kXcds, t1 = tiles * ( x + 1 ) / kXcds;
   for( int64_t t = t0 + j; t < t1; t += per )
      f( ( t * kFT + threadIdx.x ) * R );
}

template< int R, int NP, typename M, typename T >
__global__ void __launch_bounds__( kFT ) mk_dot( int64_t n, PairDict< T > D, const M* __restrict__ mask,
                                                 const T* __restrict__ p, double* __restrict__ part1,
                                                 const CgDev* __restrict__ st )
{
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   double acc = 0;
   sweep< R >( n, [ & ]( int64_t r0 ) {
      if( r0 < n ) {  // (a last group's rows past n: no entries)
         T y[ R ], pr[ R ];
         __builtin_memcpy( pr, p + r0, sizeof( pr ) );
         mask_rows< R, NP >( D, mask, p, r0, y );
#pragma unroll
         for( int j = 0; j < R; j++ )
            acc += r0 + j < n ? (double) y[ j ] * (double) pr[ j ] : 0.0;
      }
   } );
   put_part( acc, sm, part1 );
}

// d: the diagonal where it varies (else NULL and d0)
template< int R, int NP, typename M, typename T, typename DT >
__global__ void __launch_bounds__( kFT ) mk_upd( int64_t n, PairDict< T > D, const M* __restrict__ mask,
                                                 const double* __restrict__ part1, T* __restrict__ r,
                                                 const T* __restrict__ p, const DT* __restrict__ d, T d0,
                                                 double* __restrict__ part2, double* __restrict__ part3,
                                                 const CgDev* __restrict__ st )
{
   __shared__ double sm[ kFT / 64 ];
   if( ! st->active )
      return;
   const double s2 = sum_parts( part1, sm, (int) gridDim.x );
   if( s2 == 0.0 )
      return;  // the direction step ends the solve
   const T alpha = (T) ( st->s1 / s2 );
   double a2 = 0, a3 = 0;
   sweep< R >( n, [ & ]( int64_t r0 ) {
      if( r0 < n ) {
         T y[ R ], rr[ R ], dd[ R ];
         // r has room for a last group's rows past n
         __builtin_memcpy( rr, r + r0, sizeof( rr ) );
#pragma unroll
         for( int j = 0; j < R; j++ )
            dd[ j ] = d && r0 + j < n ? (T) d[ r0 + j ] : d0;
         mask_rows< R, NP >( D, mask, p, r0, y );
#pragma unroll
         for( int j = 0; j < R; j++ ) {
            const T ri = rr[ j ] - alpha * y[ j ];
            rr[ j ] = ri;
            const T zi = ri / dd[ j ];
            if( r0 + j < n ) {
               a2 += (double) ri * (double) zi;
               a3 += (double) ri * (double) ri;
            }
         }
         __builtin_memcpy( r + r0, rr, sizeof( rr ) );
      }
   } );
   put_part( a2, sm, part2 );
   if( part3 )
      put_part( a3, sm, part3 );
}

// x += alpha p; the end of the iteration as cg_dir (or, MIXED, mx_dir)
template< int R, bool MIXED, typename T, typename X, typename DT >
__global__ void __launch_bounds__( kFT ) mk_dir( int64_t n, const double* __restrict__ part1,
                                                 const double* __restrict__ part2, const double* __restrict__ part3,
                                                 const T* __restrict__ r, const DT* __restrict__ d, T d0,
                                                 T* __restrict__ p, X* __restrict__ x, const CgDev* __restrict__ cur,
                                                 CgDev* __restrict__ nxt, StopRule S, double delta2 )
{
   __shared__ double sm[ 3 * ( kFT / 64 ) ];
   const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
   if( ! cur->active ) {
      if( lead )
         *nxt = *cur;
      return;
   }
   double t[ 3 ] = { 0, 0, 0 };
   if( MIXED || S.kind == 1 )
      sum_parts_n< 3 >( { part1, part2, part3 }, sm, t, (int) gridDim.x );
   else {
      double t2[ 2 ];
      sum_parts_n< 2 >( { part1, part2 }, sm, t2, (int) gridDim.x );
      t[ 0 ] = t2[ 0 ], t[ 1 ] = t2[ 1 ];
   }
   const double s2 = t[ 0 ], s1n = t[ 1 ], rr = t[ 2 ], s1 = cur->s1;
   const double beta = s1 == 0.0 ? 0.0 : s1n / s1;
   bool go;
   if( MIXED ) {
      const int64_t it = cur->it + 1;
      const double rr_max = fmax( cur->rr_max, rr );
      go = ! ( s2 == 0.0 || rr < delta2 * rr_max || sqrt( rr ) < S.tol * cur->normb || it >= S.maxit || isnan( rr ) );
      if( lead ) {
         *nxt = *cur;
         nxt->it = it;
         nxt->s1_prev = s1;
         if( s2 != 0.0 ) {
            nxt->s1 = s1n;
            nxt->beta = beta;
            nxt->rr = rr;
            nxt->rr_max = rr_max;
         }
         if( ! go ) {
            nxt->want_update = 1;
            nxt->active = 0;
         }
      }
   }
   else {
      const double res = s2 == 0.0 ? 0.0 : sqrt( S.kind == 1 ? rr : s1n ) / cur->normb;
      go = s2 != 0.0 && check_next( S, res, cur->it );
      if( lead ) {
         *nxt = *cur;
         nxt->res = res;
         nxt->active = go ? 1 : 0;
         if( s2 == 0.0 )
            nxt->s2zero = 1;
         else {
            nxt->s1 = s1n;
            nxt->beta = beta;
            nxt->it = cur->it + 1;
         }
      }
   }
   if( s2 == 0.0 )
      return;
   const T alpha = (T) ( s1 / s2 ), tb = (T) beta;
   sweep< R >( n, [ & ]( int64_t r0 ) {
      if( r0 + R <= n ) {
         T rv[ R ], pv[ R ], dd[ R ];
         X xv[ R ];
         __builtin_memcpy( rv, r + r0, sizeof( rv ) );
         __builtin_memcpy( pv, p + r0, sizeof( pv ) );
         __builtin_memcpy( xv, x + r0, sizeof( xv ) );
#pragma unroll
         for( int j = 0; j < R; j++ )
            dd[ j ] = d ? (T) d[ r0 + j ] : d0;
#pragma unroll
         for( int j = 0; j < R; j++ ) {
            xv[ j ] += (X) ( alpha * pv[ j ] );
            pv[ j ] = rv[ j ] / dd[ j ] + tb * pv[ j ];
         }
         __builtin_memcpy( x + r0, xv, sizeof( xv ) );
         if( go )
            __builtin_memcpy( p + r0, pv, sizeof( pv ) );
      }
      else
         for( int64_t i = r0; i < n; i++ ) {
            const T pi = p[ i ];
            x[ i ] += (X) ( alpha * pi );
            if( go )
               p[ i ] = r[ i ] / ( d ? (T) d[ i ] : d0 ) + tb * pi;
         }
   } );
}

// ---- set-up kernels
__global__ void cg_start( CgDev* st, const double* s1, const double* normb, const double* rr, StopRule R )
{
   st->s1 = s1[ 0 ];
   st->normb = normb[ 0 ];
   st->res = sqrt( R.kind == 1 ? rr[ 0 ] : s1[ 0 ] ) / normb[ 0 ];
   st->beta = 0;
   st->s2zero = 0;
   st->want_update = 0;
   st->active = check_next( R, st->res, 0 ) ? 1 : 0;
   st->it = 1;  // nextIteration() counts the admitted (or refused) iteration
}

// r = b - Ap (FP64), partial sums of r.r
__global__ void __launch_bounds__( kFT ) resid_part( int64_t n, const double* __restrict__ b, double* __restrict__ r,
                                                     double* __restrict__ part )
{
   __shared__ double sm[ kFT / 64 ];
   double acc = 0;
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT ) {
      const double ri = b[ i ] - r[ i ];
      r[ i ] = ri;
      acc += ri * ri;
   }
   put_part( acc, sm, part );
}

__global__ void __launch_bounds__( kFT ) sum_into( const double* __restrict__ part, int np, double* out )
{
   __shared__ double sm[ kFT / 64 ];
   const double v = sum_parts( part, sm, np );
   if( threadIdx.x == 0 )
      out[ 0 ] = v;
}

// Mixed restart after a residual replacement: r = (float) r64, xc = 0, and
// the partial sums of (r, z), (r, r) and (r, p), z = r / d.
__global__ void __launch_bounds__( kFT ) mx_restart( int64_t n, const double* __restrict__ r64,
                                                     float* __restrict__ r, const float* __restrict__ d,
                                                     const float* __restrict__ p, float* __restrict__ xc,
                                                     double* __restrict__ part2, double* __restrict__ part3,
                                                     double* __restrict__ part4 )
{
   __shared__ double sm[ kFT / 64 ];
   double a2 = 0, a3 = 0, a4 = 0;
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT ) {
      const float ri = (float) r64[ i ];
      const float zi = ri / d[ i ];
      r[ i ] = ri;
      xc[ i ] = 0.0f;
      a2 += (double) ri * (double) zi;
      a3 += (double) ri * (double) ri;
      a4 += (double) ri * (double) p[ i ];
   }
   put_part( a2, sm, part2 );
   put_part( a3, sm, part3 );
   put_part( a4, sm, part4 );
}

// The scalars after a replacement.  first: p = z.  Otherwise the kept
// direction is made orthogonal to the new residual (p -= ((r, p) / (r, z)) z,
// as exact CG has (r_{k+1}, p_k) = 0) and p = z + beta p with
// beta = (r, z) / (r, z)_previous -- the residual replacement of Clark et al.
__global__ void __launch_bounds__( kFT ) mx_state( CgDev* st, const double* __restrict__ part2,
                                                   const double* __restrict__ part3, const double* __restrict__ part4,
                                                   const double* normb, int64_t it, int first, int np )
{
   __shared__ double sm[ kFT / 64 ];
   const double s1 = sum_parts( part2, sm, np );
   const double rr = sum_parts( part3, sm, np );
   const double rp = sum_parts( part4, sm, np );
   if( threadIdx.x != 0 )
      return;
   if( first ) {
      st->beta = 0.0;
      st->proj = 0.0;
   }
   else {
      st->proj = s1 != 0.0 ? rp / s1 : 0.0;
      st->beta = st->s1_prev != 0.0 ? s1 / st->s1_prev : 0.0;
   }
   st->s1 = s1;
   st->rr = rr;
   st->rr_max = rr;
   st->normb = normb[ 0 ];
   st->want_update = 0;
   st->it = it;
   st->active = 1;
}

// p = z + beta (p - proj z), z = r / d (p = z on the first start)
__global__ void __launch_bounds__( kFT ) mx_redir( int64_t n, const float* __restrict__ r, const float* __restrict__ d,
                                                   float* __restrict__ p, const CgDev* __restrict__ st, int first )
{
   const float beta = (float) st->beta, proj = (float) st->proj;
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT ) {
      const float zi = r[ i ] / d[ i ];
      p[ i ] = first ? zi : zi + beta * ( p[ i ] - proj * zi );
   }
}

// x += xc (FP64 accumulation of the FP32 correction)
__global__ void __launch_bounds__( kFT ) mx_accumulate( int64_t n, const float* __restrict__ xc, double* __restrict__ x )
{
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT )
      x[ i ] += (double) xc[ i ];
}

template< typename D >
__global__ void to_f32( int64_t n, const D* __restrict__ a, float* __restrict__ o )
{
   for( int64_t i = (int64_t) blockIdx.x * kFT + threadIdx.x; i < n; i += (int64_t) gridDim.x * kFT )
      o[ i ] = (float) a[ i ];
}

// ---- which SpMV stage a matrix gets
struct Stage
{
   const tnlmi_matrix* A = nullptr;
   const tnlmi_spmv_plan* plan = nullptr;
   SegView v{};
   int kind = 0;  // 0: the format's own SpMV kernel + dot_part, 1: fused Ellpack/SlicedEllpack column-major,
                  // 2: fused one-launch tiled CSR (no row longer than kWholeRowMax)
   int64_t grid = 0;                      // blocks of the fused SpMV kernel
   int rows_per_thread = 1;               // Ellpack / SlicedEllpack kernel
   std::shared_ptr< DeviceArray< double > > part;  // its per-block partial sums
   // the slots kind 1 reads: the matrix's own, or (a CSR matrix with short
   // rows) the stage's column-major Ellpack copy of them
   const int32_t* cols = nullptr;
   const void* vals = nullptr;
   int64_t storage = 0;
   std::shared_ptr< DeviceArray< int32_t > > ecols;
   std::shared_ptr< DeviceArray< char > > evals;
   // kind 1 with 8-bit column codes (the inner matrix of the mixed solver)
   std::shared_ptr< DeviceArray< uint8_t > > codes;
   std::shared_ptr< DeviceArray< int32_t > > dict;
   int32_t ndict = 0;
   // kind 1 as row masks (pairs > 0)
   std::shared_ptr< DeviceArray< uint8_t > > masks;  // a row: 1 byte (pairs <= 8) or 2
   int32_t pairs = 0, reach = 0;  // distinct pairs; the largest |column - row|
   PairDict< double > dict64{};
   PairDict< float > dict32{};
};

// The row masks of a column-major Ellpack / SlicedEllpack stage, or nothing
// (more than kPairs distinct pairs, or rows with another order of entries).
// Two passes over the matrix: 0.5 + 0.6 ms for 117 M FP64 entries.
// TNLMI_COLUMN_CODES=0 in the environment keeps the matrix as it is.
template< typename V >
void make_masks_v( Stage& S, PairTable* table, hipStream_t s )
{
   PairTable ht;
   TNLMI_HIP( hipMemsetAsync( table, 0xff, offsetof( PairTable, val ), s ) );
   TNLMI_HIP( hipMemsetAsync( &table->count, 0, 2 * sizeof( int32_t ), s ) );
   for( const unsigned grid : { 8u, 2048u } )
      hipLaunchKernelGGL( pairs_collect< V >, dim3( grid ), dim3( kFT ), 0, s, S.v, S.cols, (const V*) S.vals, table,
                          grid == 8 ? std::min< int64_t >( S.v.n, 8 * kFT ) : S.v.n );
   TNLMI_HIP( hipGetLastError() );
   TNLMI_HIP( hipMemcpyAsync( &ht, table, sizeof( ht ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   if( ht.reject || ht.count > kPairs || ht.count == 0 )
      return;
   std::vector< std::pair< int32_t, uint64_t > > pairs;
   for( int h = 0; h < kPairHash; h++ )
      if( ht.key[ h ] != kEmpty )
         pairs.push_back( { ht.off[ h ], ht.val[ h ] } );
   std::sort( pairs.begin(), pairs.end() );
   RawDict D{};
   D.count = (int32_t) pairs.size();
   for( int q = 0; q < D.count; q++ ) {
      D.off[ q ] = pairs[ q ].first;
      D.bits[ q ] = pairs[ q ].second;
      V v;
      memcpy( &v, &pairs[ q ].second, sizeof( V ) );
      double d;
      if constexpr( std::is_same_v< V, bf16 > )
         d = (double) bf16_to_float( v.bits );
      else
         d = (double) v;
      S.dict64.off[ q ] = S.dict32.off[ q ] = D.off[ q ];
      S.dict64.val[ q ] = d;
      S.dict32.val[ q ] = (float) d;
      S.reach = std::max( S.reach, std::abs( D.off[ q ] ) );
   }
   // (whole tiles of mk_dot: the rows past n hold no entry)
   const int64_t rows = ceil_div( S.v.n, kFT * 4 ) * ( kFT * 4 );
   auto masks = std::make_shared< DeviceArray< uint8_t > >();
   masks->allocate( rows * ( D.count <= 8 ? 1 : 2 ) );
   if( D.count <= 8 )
      hipLaunchKernelGGL( ( pairs_encode< V, uint8_t > ), dim3( 4096 ), dim3( kFT ), 0, s, S.v, S.cols,
                          (const V*) S.vals, D, masks->ptr, rows, &table->reject );
   else
      hipLaunchKernelGGL( ( pairs_encode< V, uint16_t > ), dim3( 4096 ), dim3( kFT ), 0, s, S.v, S.cols,
                          (const V*) S.vals, D, (uint16_t*) masks->ptr, rows, &table->reject );
   TNLMI_HIP( hipGetLastError() );
   int32_t reject = 0;
   TNLMI_HIP( hipMemcpyAsync( &reject, &table->reject, sizeof( reject ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   if( reject )
      return;
   S.masks = masks;
   S.pairs = D.count;
   S.ecols.reset();  // (a copy of a CSR matrix's slots is not read any more)
   S.evals.reset();
}

// scratch: a vector of the matrix's rows that the solve does not use yet
template< typename T >
void make_masks( Stage& S, T* scratch, hipStream_t s )
{
   constexpr int64_t least = sizeof( T ) == 8 ? kMaskRows : kMaskRowsMixed;
   static_assert( least * sizeof( T ) >= sizeof( PairTable ) );
   const char* env = std::getenv( "TNLMI_COLUMN_CODES" );
   if( S.kind != 1 || S.v.n < least || ( env && std::string( env ) == "0" ) )
      return;
   PairTable* table = (PairTable*) scratch;
   switch( S.A->value_type ) {
      case TNLMI_F64:
         return make_masks_v< double >( S, table, s );
      case TNLMI_F32:
         return make_masks_v< float >( S, table, s );
      case TNLMI_BF16:
         return make_masks_v< bf16 >( S, table, s );
   }
}

// One iteration by row masks, T: the vectors' type.  p has S.reach + kMaskRoom
// values of room at both ends, r mask_rows_room( n ) values.
constexpr int64_t kMaskRoom = kFT * 4;
inline int64_t mask_rows_room( int64_t n )  // (whole groups of 2 or 4 rows)
{
   return ceil_div( n, 4 ) * 4;
}
template< typename T, typename X, typename DT, bool MIXED >
void mask_iteration( const Stage& S, T* r, T* p, X* x, const DT* d, T d0, double* part1, double* part2, double* part3,
                     const CgDev* cur, CgDev* nxt, const StopRule& R, double delta2, hipStream_t s )
{
   constexpr int kR = sizeof( T ) == 8 ? 2 : 4;  // rows per thread: 16 bytes
   const dim3 grid( kFB ), block( kFT );
   auto go = [ & ]( auto tag, auto np ) {
      using M = decltype( tag );
      constexpr int NP = decltype( np )::value;
      const M* mask = (const M*) S.masks->ptr;
      const PairDict< T >* D;
      if constexpr( sizeof( T ) == 8 )
         D = &S.dict64;
      else
         D = &S.dict32;
      hipLaunchKernelGGL( ( mk_dot< kR, NP, M, T > ), grid, block, 0, s, S.v.n, *D, mask, (const T*) p, part1, cur );
      hipLaunchKernelGGL( ( mk_upd< kR, NP, M, T, DT > ), grid, block, 0, s, S.v.n, *D, mask, (const double*) part1, r,
                          (const T*) p, d, d0, part2, part3, cur );
   };
   if( S.pairs <= 5 )
      go( uint8_t(), std::integral_constant< int, 5 >() );
   else if( S.pairs <= 7 )
      go( uint8_t(), std::integral_constant< int, 7 >() );
   else if( S.pairs <= 8 )
      go( uint8_t(), std::integral_constant< int, 8 >() );
   else
      go( uint16_t(), std::integral_constant< int, 16 >() );
   hipLaunchKernelGGL( ( mk_dir< kR, MIXED, T, X, DT > ), grid, block, 0, s, S.v.n, (const double*) part1,
                       (const double*) part2, (const double*) part3, (const T*) r, d, d0, p, x, cur, nxt, R, delta2 );
}

// the diagonal's one value if it has one, else NAN (n > 0)
double uniform_diagonal( int64_t n, const double* d, hipStream_t s )
{
   DeviceArray< int32_t > other;
   other.allocate( 1 );
   TNLMI_HIP( hipMemsetAsync( other.ptr, 0, sizeof( int32_t ), s ) );
   hipLaunchKernelGGL( varies, dim3( 2048 ), dim3( kFT ), 0, s, n, d, other.ptr );
   int32_t more = 0;
   double first = 0;
   TNLMI_HIP( hipMemcpyAsync( &more, other.ptr, sizeof( more ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipMemcpyAsync( &first, d, sizeof( first ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   return more ? std::nan( "" ) : first;
}

// The column codes of a column-major Ellpack / SlicedEllpack matrix, or
// nothing (more than kCodes distinct offsets).  Set TNLMI_COLUMN_CODES=0 in
// the environment to keep the int32 columns (identical results, more bytes).
void make_codes( Stage& S, hipStream_t s )
{
   const char* env = std::getenv( "TNLMI_COLUMN_CODES" );
   if( env && std::string( env ) == "0" )
      return;
   const int64_t storage = S.storage;
   DeviceArray< unsigned long long > table;
   DeviceArray< int32_t > flags;  // count, overflow
   table.allocate( kHash );
   flags.allocate( 2 );
   TNLMI_HIP( hipMemsetAsync( table.ptr, 0xff, sizeof( unsigned long long ) * kHash, s ) );
   TNLMI_HIP( hipMemsetAsync( flags.ptr, 0, sizeof( int32_t ) * 2, s ) );
   const unsigned grid = (unsigned) std::min< int64_t >( 4096, std::max< int64_t >( 1, ceil_div( S.v.n, kFT ) ) );
   hipLaunchKernelGGL( code_collect, dim3( grid ), dim3( kFT ), 0, s, S.v, S.cols, table.ptr, flags.ptr,
                       flags.ptr + 1 );
   TNLMI_HIP( hipGetLastError() );
   std::vector< unsigned long long > ht( kHash );
   int32_t hf[ 2 ];
   TNLMI_HIP( hipMemcpyAsync( ht.data(), table.ptr, sizeof( unsigned long long ) * kHash, hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipMemcpyAsync( hf, flags.ptr, sizeof( hf ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   if( hf[ 1 ] != 0 || hf[ 0 ] > kCodes )
      return;
   std::vector< int32_t > keys;
   for( const auto k : ht )
      if( k != kEmpty )
         keys.push_back( (int32_t) (uint32_t) k );
   std::sort( keys.begin(), keys.end() );
   std::vector< uint8_t > code_of( kHash, kPadCode );
   for( int h = 0; h < kHash; h++ )
      if( ht[ h ] != kEmpty )
         code_of[ h ] = (uint8_t) ( std::lower_bound( keys.begin(), keys.end(), (int32_t) (uint32_t) ht[ h ] )
                                    - keys.begin() );
   DeviceArray< uint8_t > dcode_of;
   dcode_of.allocate( kHash );
   S.dict = std::make_shared< DeviceArray< int32_t > >();
   S.dict->allocate( std::max< int64_t >( 1, (int64_t) keys.size() ) );
   S.codes = std::make_shared< DeviceArray< uint8_t > >();
   // R bytes are read per row group: room for the last group's overhang
   S.codes->allocate( storage + 16 );
   TNLMI_HIP( hipMemcpyAsync( dcode_of.ptr, code_of.data(), kHash, hipMemcpyHostToDevice, s ) );
   if( ! keys.empty() )
      TNLMI_HIP( hipMemcpyAsync( S.dict->ptr, keys.data(), sizeof( int32_t ) * keys.size(), hipMemcpyHostToDevice,
                                 s ) );
   TNLMI_HIP( hipMemsetAsync( S.codes->ptr, kPadCode, storage + 16, s ) );
   hipLaunchKernelGGL( code_encode, dim3( grid ), dim3( kFT ), 0, s, S.v, S.cols, table.ptr, dcode_of.ptr,
                       S.codes->ptr );
   TNLMI_HIP( hipGetLastError() );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   S.ndict = (int32_t) keys.size();
}

// kind 1 launch shape over S.v (column-major Ellpack / SlicedEllpack)
void ell_shape( Stage& S )
{
   S.kind = 1;
   // 16-byte loads of the column indexes for 4-byte values, of the values for FP64
   S.rows_per_thread = S.A->value_type == TNLMI_F64 ? 2 : 4;
   if( S.v.format == TNLMI_SLICED_ELLPACK && S.v.slice_size % S.rows_per_thread != 0 )
      S.rows_per_thread = 1;
   S.grid = ceil_div( ceil_div( S.v.n, S.rows_per_thread ), kFT );
   S.part = std::make_shared< DeviceArray< double > >();
   S.part->allocate( S.grid );
}

// CSR rows as column-major Ellpack slots: slot j of row r at j * stride + r
// (padding: column -1, value 0); rows [n, stride) are all padding
//
// Bound: both layouts' bytes.  A workgroup takes ROWS rows, whose entries are
// contiguous in CSR, through LDS, so that the loads and the stores are both
// coalesced.  One lane per row without LDS: a wave's loads of a slot lie w
// entries apart, and with long rows their lines leave L1 before the next slot
// wants them.  10^6 rows in FP64, us before -> now: of 27 entries 898 -> 116
// (5.6 TB/s), 16: 431 -> 67, 9: 113 -> 46, 8: 88 -> 40, 5: 32 -> 26, 1: 8 -> 8;
// Poisson 256^3 907 -> 502.  With 64 rows of up to eight entries, too, 1: 17,
// 5: 31, Poisson 256^3 569: a short row's workgroup has more rows.
constexpr int kCopySlots = 2048;  // of a workgroup: 24 KB of LDS in FP64
constexpr int kCopyRows = kCopySlots / kWholeRowMax, kCopyShortRows = 256;  // kCopyShortRows: w <= kCopyShort
constexpr int kCopyShort = kCopySlots / kCopyShortRows;

// one word of padding per 32 keeps rows of 8, 16 and 32 entries off one bank
__host__ __device__ constexpr int copy_slot( int i ) { return i + ( i >> 5 ); }

template< int ROWS, typename V >
__global__ __launch_bounds__( 256 ) void csr_to_ell( int64_t n, int64_t stride, int32_t w,
                                                     const int32_t* __restrict__ off,
                                                     const int32_t* __restrict__ cols, const V* __restrict__ vals,
                                                     int32_t* __restrict__ ec, V* __restrict__ ev )
{
   __shared__ V sv[ copy_slot( kCopySlots ) ];
   __shared__ int32_t sc[ copy_slot( kCopySlots ) ];
   const int64_t r0 = (int64_t) blockIdx.x * ROWS, r = r0 + threadIdx.x % ROWS;
   const int32_t first = off[ r0 < n ? r0 : n ], last = off[ r0 + ROWS < n ? r0 + ROWS : n ];
   const int32_t b = off[ r < n ? r : n ] - first, e = off[ r < n ? r + 1 : n ] - first;
   for( int32_t i = threadIdx.x; i < last - first; i += 256 ) {  // at most ROWS * w <= kCopySlots
      sc[ copy_slot( i ) ] = cols[ first + i ];
      sv[ copy_slot( i ) ] = vals[ first + i ];
   }
   __syncthreads();
   if( r >= stride )
      return;
   for( int32_t j = threadIdx.x / ROWS; j < w; j += 256 / ROWS ) {
      const bool in = b + j < e;
      ec[ j * stride + r ] = in ? sc[ copy_slot( b + j ) ] : -1;
      ev[ j * stride + r ] = in ? sv[ copy_slot( b + j ) ] : V{};
   }
}

template< typename V >
void csr_to_ell_launch( int64_t n, int64_t stride, int32_t w, const tnlmi_matrix& A, int32_t* ec, void* ev,
                        hipStream_t s )
{
   if( w <= kCopyShort )
      hipLaunchKernelGGL( ( csr_to_ell< kCopyShortRows, V > ), dim3( (unsigned) ceil_div( stride, kCopyShortRows ) ),
                          dim3( 256 ), 0, s, n, stride, w, A.segments->offsets.ptr, A.column_indexes,
                          (const V*) A.values, ec, (V*) ev );
   else
      hipLaunchKernelGGL( ( csr_to_ell< kCopyRows, V > ), dim3( (unsigned) ceil_div( stride, kCopyRows ) ),
                          dim3( 256 ), 0, s, n, stride, w, A.segments->offsets.ptr, A.column_indexes,
                          (const V*) A.values, ec, (V*) ev );
}

// A CSR matrix whose rows are all short (at most kWholeRowMax entries) and
// about equally long (the Ellpack copy at most 1/8 larger than the CSR
// arrays): the stage keeps a column-major Ellpack copy of its slots, made
// here on every solve, and runs the fused Ellpack kernels on it.  Every row
// keeps its entries in CSR order, so the products and sums are those of the
// Ellpack kernels on the same matrix stored as Ellpack.  TNLMI_CG_CSR_COPY=0
// in the environment keeps the one-launch CSR kernel instead, and so does a
// device without room for the copy.
// room: memory of csr_copy_slots( A ) slots for it, or NULL (the copy has its own).
int64_t csr_copy_slots( const tnlmi_matrix& A )  // 0: no copy is made
{
   const char* env = std::getenv( "TNLMI_CG_CSR_COPY" );
   const tnlmi_segments& seg = *A.segments;
   if( seg.format != TNLMI_CSR || A.matrix_type == TNLMI_SYMMETRIC || ( env && std::string( env ) == "0" ) )
      return 0;
   const int64_t n = make_view( seg ).n, slots = ceil_div( n, 64 ) * 64 * std::max( 1, seg.max_size );
   return seg.max_size > kWholeRowMax || slots > seg.elements + seg.elements / 8 ? 0 : slots;
}

bool csr_ell_copy( Stage& S, void* room, hipStream_t s )
{
   const tnlmi_matrix& A = *S.A;
   const tnlmi_segments& seg = *A.segments;
   const int64_t n = S.v.n, slots = csr_copy_slots( A );
   if( slots == 0 )
      return false;
   const int32_t w = std::max( 1, seg.max_size );
   const int64_t stride = slots / w;
   const size_t vs = A.value_type == TNLMI_F64 ? 8 : A.value_type == TNLMI_F32 ? 4 : 2;
   void* evals = room;
   int32_t* ecols = (int32_t*) ( (char*) room + slots * vs );
   if( ! room ) {
      S.ecols = std::make_shared< DeviceArray< int32_t > >();
      S.evals = std::make_shared< DeviceArray< char > >();
      try {
         S.ecols->allocate( slots );
         S.evals->allocate( slots * (int64_t) vs );
      }
      catch( const Error& e ) {
         // no room for the copy: the one-launch CSR kernel on the matrix itself
         if( e.status != TNLMI_BAD_ALLOC )
            throw;
         (void) hipGetLastError();
         S.ecols.reset();
         S.evals.reset();
         return false;
      }
      ecols = S.ecols->ptr;
      evals = S.evals->ptr;
   }
   switch( A.value_type ) {
      case TNLMI_F64: csr_to_ell_launch< double >( n, stride, w, A, ecols, evals, s ); break;
      case TNLMI_F32: csr_to_ell_launch< float >( n, stride, w, A, ecols, evals, s ); break;
      default: csr_to_ell_launch< bf16 >( n, stride, w, A, ecols, evals, s ); break;
   }
   TNLMI_HIP( hipGetLastError() );
   SegView v{};
   v.format = TNLMI_ELLPACK;
   v.col_major = 1;
   v.n = n;
   v.ell_width = w;
   v.ell_aligned = (int32_t) stride;
   S.v = v;
   S.cols = ecols;
   S.vals = evals;
   S.storage = slots;
   return true;
}

Stage make_stage( const tnlmi_matrix* A, const tnlmi_spmv_plan* plan, hipStream_t s, void* room = nullptr )
{
   Stage S;
   S.A = A;
   S.plan = plan;
   S.v = make_view( *A->segments );
   S.cols = A->column_indexes;
   S.vals = A->values;
   S.storage = A->segments->storage;
   if( plan )
      return S;
   const int fmt = S.v.format;
   if( ( fmt == TNLMI_ELLPACK || fmt == TNLMI_SLICED_ELLPACK ) && S.v.col_major && A->matrix_type != TNLMI_SYMMETRIC ) {
      ell_shape( S );
      return S;
   }
   const tnlmi_segments& seg = *A->segments;
   if( fmt == TNLMI_CSR && A->matrix_type != TNLMI_SYMMETRIC && csr_ell_copy( S, room, s ) ) {
      ell_shape( S );
      return S;
   }
   if( fmt == TNLMI_CSR && A->matrix_type != TNLMI_SYMMETRIC && seg.max_size <= kWholeRowMax && seg.tiles > 0
       && ( seg.tile_nnz == kTileNnz || seg.tile_nnz == kTileNnzSmall ) ) {
      S.kind = 2;
      S.grid = ceil_div( seg.tiles, 4 );
      S.part = std::make_shared< DeviceArray< double > >();
      S.part->allocate( S.grid );
   }
   return S;
}

template< typename V, typename T >
void stage_launch_v( const Stage& S, const T* p, T* Ap, double* part, const CgDev* st, hipStream_t s )
{
   const V* vals = (const V*) S.vals;
   double* bp = S.part->ptr;
   if( S.kind == 1 && S.codes ) {
      const uint8_t* c = S.codes->ptr;
      const int32_t* d = S.dict->ptr;
      if( S.rows_per_thread == 4 )
         hipLaunchKernelGGL( ( spmv_dot_ell_code< 4, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v, c, d,
                             S.ndict, vals, p, Ap, bp, st );
      else if( S.rows_per_thread == 2 )
         hipLaunchKernelGGL( ( spmv_dot_ell_code< 2, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v, c, d,
                             S.ndict, vals, p, Ap, bp, st );
      else
         hipLaunchKernelGGL( ( spmv_dot_ell_code< 1, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v, c, d,
                             S.ndict, vals, p, Ap, bp, st );
   }
   else if( S.kind == 2 ) {
      const tnlmi_segments& seg = *S.A->segments;
      const int32_t tail_max = std::max( 0, seg.max_size - 1 );
      if( seg.tile_nnz == kTileNnzSmall )
         hipLaunchKernelGGL( ( spmv_dot_csr< V, T, kTileNnzSmall > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s,
                             seg.offsets.ptr, seg.tile_rows.ptr, seg.tiles, seg.elements, S.v.n, S.A->column_indexes,
                             vals, p, Ap, bp, st, tail_max );
      else
         hipLaunchKernelGGL( ( spmv_dot_csr< V, T, kTileNnz > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s,
                             seg.offsets.ptr, seg.tile_rows.ptr, seg.tiles, seg.elements, S.v.n, S.A->column_indexes,
                             vals, p, Ap, bp, st, tail_max );
   }
   else if( S.kind == 1 ) {
      if( S.rows_per_thread == 4 )
         hipLaunchKernelGGL( ( spmv_dot_ell< 4, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v,
                             S.cols, vals, p, Ap, bp, st );
      else if( S.rows_per_thread == 2 )
         hipLaunchKernelGGL( ( spmv_dot_ell< 2, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v,
                             S.cols, vals, p, Ap, bp, st );
      else
         hipLaunchKernelGGL( ( spmv_dot_ell< 1, V, T > ), dim3( (unsigned) S.grid ), dim3( kFT ), 0, s, S.v,
                             S.cols, vals, p, Ap, bp, st );
   }
   hipLaunchKernelGGL( fold_parts, dim3( blocks_of< T >() ), dim3( kFT ), 0, s, bp, S.grid, part, st );
}

// Ap = A p and the partial sums of (Ap, p)
template< typename T >
void stage_launch( const Stage& S, const T* p, T* Ap, double* part, const CgDev* st, hipStream_t s )
{
   constexpr tnlmi_dtype xt = std::is_same_v< T, double > ? TNLMI_F64 : TNLMI_F32;
   if( S.kind == 0 ) {
      if( S.plan )
         plan_execute( *S.plan, xt, p, Ap, xt, 1.0, 0.0, 0, S.v.n, s );
      else {
         const tnlmi_launch cfg{ TNLMI_MAP_AUTO, 1 };
         spmv_dispatch( *S.A, xt, p, Ap, xt, 1.0, 0.0, 0, S.v.n, cfg, s );
      }
      hipLaunchKernelGGL( dot_part< T >, dim3( blocks_of< T >() ), dim3( kFT ), 0, s, S.v.n, Ap, p, part, st );
      return;
   }
   switch( S.A->value_type ) {
      case TNLMI_F64:
         stage_launch_v< double, T >( S, p, Ap, part, st, s );
         return;
      case TNLMI_F32:
         stage_launch_v< float, T >( S, p, Ap, part, st, s );
         return;
      case TNLMI_BF16:
         stage_launch_v< bf16, T >( S, p, Ap, part, st, s );
         return;
   }
   fail( TNLMI_INVALID_ARGUMENT, "fused CG: unsupported value type" );
}

struct Parts
{
   DeviceArray< double > a, b, c;
   Parts()
   {
      a.allocate( kFB );
      b.allocate( kFB );
      c.allocate( kFB );
   }
};

// pinned host copy of the device state
struct HostState
{
   CgDev* h = nullptr;
   HostState() { TNLMI_HIP( hipHostMalloc( (void**) &h, sizeof( CgDev ), hipHostMallocDefault ) ); }
   ~HostState()
   {
      if( h )
         (void) hipHostFree( h );
   }
   const CgDev& read( const CgDev* d, hipStream_t s )
   {
      TNLMI_HIP( hipMemcpyAsync( h, d, sizeof( CgDev ), hipMemcpyDeviceToHost, s ) );
      TNLMI_HIP( hipStreamSynchronize( s ) );
      return *h;
   }
};

}  // namespace

namespace {

// What a solve by grid_cg needs besides the solve's own arrays.
// z goes where the residual was: a launch holds that in registers, and no
// workgroup reads another's z after the last sum, when it is stored again.
template< typename T >
struct GridWork
{
   DeviceArray< GridSlots > slots;
   DeviceArray< int32_t > late;
   uint32_t number = 1;
   explicit GridWork( hipStream_t s )
   {
      slots.allocate( 1 );
      late.allocate( 1 );
      TNLMI_HIP( hipMemsetAsync( slots.ptr, 0, sizeof( GridSlots ), s ) );
      TNLMI_HIP( hipMemsetAsync( late.ptr, 0, sizeof( int32_t ), s ) );
   }
   template< typename X >
   void fill( GridCg< T, X >& a, const Stage& S, T* r, T* p, T* p1 )
   {
      a.n = S.v.n;
      a.stride = S.v.ell_aligned;
      a.w = S.v.ell_width;
      a.cols = S.cols;
      a.vals = S.vals;
      a.r = a.z = r;
      a.p[ 0 ] = p;
      a.p[ 1 ] = p1;
      a.slots = slots.ptr;
      a.wait = grid_wait();
      a.number = number;
      a.most = kGridIterations;
      a.late = late.ptr;
      number += 2 * kGridIterations;
   }
};

// Which matrices a resident launch takes: Ellpack slots (the matrix's own or the
// copy of a CSR matrix with short rows) of at most kGridRows rows, with few
// enough far lines for vectors of LINE entries per 128 bytes (kFar64 and so on).
template< int LINE >
bool grid_takes( const Stage& S, double far, hipStream_t s )
{
   const int64_t n = S.v.n;
   if( S.kind != 1 || S.v.format != TNLMI_ELLPACK || n <= 0 || n > kGridRows )
      return false;
   if( n <= (int64_t) kGridMax * 512 || (double) n * n * S.v.ell_width <= far )
      return true;
   const int32_t block = n <= (int64_t) kGridMax * 1024 ? 1024 : n <= (int64_t) kGridMax * 2048 ? 2048 : 4096;
   double lines = 0;
   hipLaunchKernelGGL( far_lines< LINE >, dim3( 1 ), dim3( 1024 ), 0, s, n, (int64_t) S.v.ell_aligned, S.v.ell_width, S.cols,
                       block, S.part->ptr );
   TNLMI_HIP( hipMemcpyAsync( &lines, S.part->ptr, sizeof( lines ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   return lines * n <= far;
}

}  // namespace

namespace {

// false: a grid sum of grid_cg was given up (x is what it was, or nearer to the solution)
bool fused_cg_run( const Operator& A, const tnlmi_preconditioner* M, const double* b, double* x,
                   tnlmi_solver_state* st, hipStream_t s, int residue_kind, bool column_codes, bool grid )
{
   const int64_t n = A.rows;
   const double* d = precond_diagonal( M );
   DeviceArray< double > r, p, Ap, sc;
   DeviceArray< CgDev > dev;
   r.allocate( mask_rows_room( n ) );
   p.allocate( n );
   Ap.allocate( n );
   sc.allocate( 4 );
   dev.allocate( 2 );
   Parts parts;
   RedWork w;
   HostState hs;
   const StopRule R{ st->max_iterations, st->min_iterations, st->convergence_residue, st->divergence_residue,
                     residue_kind };
   // normb = ||M^{-1} b|| (CG.hpp:24-29); ||b|| for the recurrence residual
   if( d && residue_kind == 0 ) {
      precond_apply( M, n, b, r.ptr, s );
      nrm2( n, r.ptr, sc.ptr + 1, w, s );
   }
   else
      nrm2( n, b, sc.ptr + 1, w, s );
   double normb = 0;
   TNLMI_HIP( hipMemcpyAsync( &normb, sc.ptr + 1, sizeof( double ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   if( normb == 0.0 ) {
      fill( n, 0.0, x, s );
      st->iterations = 0;
      st->residue = 0.0;
      st->converged = 1;
      return true;
   }
   // r = b - A x; p = z = M^{-1} r; s1 = (r, z)
   A.apply( x, r.ptr, s );
   rsub( n, b, r.ptr, s );
   precond_apply( M, n, r.ptr, p.ptr, s );
   dot( n, r.ptr, p.ptr, sc.ptr + 0, w, s );
   if( residue_kind == 1 )
      dot( n, r.ptr, r.ptr, sc.ptr + 2, w, s );
   hipLaunchKernelGGL( cg_start, dim3( 1 ), dim3( 1 ), 0, s, dev.ptr, sc.ptr + 0, sc.ptr + 1, sc.ptr + 2, R );
   TNLMI_HIP( hipGetLastError() );
   const CgDev* h = &hs.read( dev.ptr, s );
   Stage S = make_stage( A.A, A.plan, s );
   const bool resident = grid && S.A->value_type == TNLMI_F64 && grid_takes< 16 >( S, kFar64, s );
   if( ! resident ) {
      if( h->active )
         make_masks( S, Ap.ptr, s );
      if( column_codes && S.kind == 1 && ! S.pairs )
         make_codes( S, s );
   }
   DeviceArray< double > room;
   double* pp = p.ptr;
   double d0 = 1.0;  // (r / 1 is r: no preconditioner)
   const double* dv = d;
   if( S.pairs ) {
      const int64_t at = S.reach + kMaskRoom;
      room.allocate( n + 2 * at );
      pp = room.ptr + at;
      TNLMI_HIP( hipMemcpyAsync( pp, p.ptr, sizeof( double ) * n, hipMemcpyDeviceToDevice, s ) );
      TNLMI_HIP( hipStreamSynchronize( s ) );
      p.reset();
      if( d ) {
         d0 = uniform_diagonal( n, d, s );
         if( ! std::isnan( d0 ) )
            dv = nullptr;
      }
   }
   // the state is double-buffered by iteration parity: iteration k reads
   // dev[k & 1] and its last kernel writes dev[(k + 1) & 1]
   int par = 0;
   if( resident && h->active ) {
      GridWork< double > work( s );
      GridCg< double, double > a{};
      a.x = x;
      a.d = d;
      a.st = dev.ptr;
      a.R = R;
      do {
         const auto turn = resident_turn();
         work.fill( a, S, r.ptr, p.ptr, Ap.ptr );
         if( ! grid_cg_launch< double, double, double, double, false >( a, s ) )
            break;
         int32_t late = 0;
         TNLMI_HIP( hipMemcpyAsync( &late, work.late.ptr, sizeof( late ), hipMemcpyDeviceToHost, s ) );
         h = &hs.read( dev.ptr, s );
         if( late )
            return false;
      } while( h->active );
   }
   while( h->active ) {
      for( int k = 0; k < kBatch; k++, par ^= 1 ) {
         CgDev* cur = dev.ptr + par;
         double* part3 = residue_kind == 1 ? parts.c.ptr : nullptr;
         if( S.pairs ) {
            mask_iteration< double, double, double, false >( S, r.ptr, pp, x, dv, d0, parts.a.ptr, parts.b.ptr, part3,
                                                             cur, dev.ptr + ( par ^ 1 ), R, 0.0, s );
            continue;
         }
         stage_launch< double >( S, p.ptr, Ap.ptr, parts.a.ptr, cur, s );
         hipLaunchKernelGGL( ( cg_upd< double, double, double > ), dim3( blocks_of< double >() ), dim3( kFT ), 0, s, n,
                             parts.a.ptr,
                             r.ptr, p.ptr, Ap.ptr, x, d, parts.b.ptr, part3, cur );
         hipLaunchKernelGGL( ( cg_dir< double, double > ), dim3( blocks_of< double >() ), dim3( kFT ), 0, s, n,
                             parts.a.ptr,
                             parts.b.ptr, part3, r.ptr, d, p.ptr, cur, dev.ptr + ( par ^ 1 ), R );
      }
      TNLMI_HIP( hipGetLastError() );
      h = &hs.read( dev.ptr + par, s );
   }
   Stop S2{ st };
   S2.it = h->it;
   S2.res = h->res;
   st->iterations = h->it;
   st->residue = h->res;
   st->converged = S2.converged();
   return true;
}

}  // namespace

int64_t ell_copy_values( const Operator& A )
{
   return A.plan || A.A->value_type != TNLMI_F64 || A.rows > kGridRows ? 0 : ceil_div( 3 * csr_copy_slots( *A.A ), 2 );
}

bool ell_slots( const Operator& A, double far, double* room, EllSlots& out, hipStream_t s )
{
   if( A.plan || A.A->value_type != TNLMI_F64 || A.rows > kGridRows || ( ! room && ell_copy_values( A ) > 0 ) )
      return false;
   const Stage S = make_stage( A.A, nullptr, s, room );
   if( ! grid_takes< 16 >( S, far, s ) )
      return false;
   out.n = S.v.n;
   out.stride = S.v.ell_aligned;
   out.w = S.v.ell_width;
   out.cols = S.cols;
   out.vals = (const double*) S.vals;
   return true;
}

void fused_cg_solve( const Operator& A, const tnlmi_preconditioner* M, const double* b, double* x,
                     tnlmi_solver_state* st, hipStream_t s, int residue_kind, bool column_codes )
{
   if( ! fused_cg_run( A, M, b, x, st, s, residue_kind, column_codes, true ) )
      fused_cg_run( A, M, b, x, st, s, residue_kind, column_codes, false );
}

}  // namespace tnlmi

using namespace tnlmi;

extern "C" {

tnlmi_status tnlmi_mixed_cg_solve( const tnlmi_matrix* A, const tnlmi_matrix* A_lo, const tnlmi_spmv_plan* plan,
                                   double delta, const double* d_b, double* d_x, tnlmi_solver_state* st,
                                   int64_t* updates, tnlmi_stream stream )
{
   return guarded( [ & ] {
      if( ! A || ! A_lo || ! A->segments || ! A_lo->segments || ! d_b || ! d_x || ! st )
         fail( TNLMI_INVALID_ARGUMENT, "mixed_cg_solve: NULL argument" );
      if( A->value_type != TNLMI_F64 )
         fail( TNLMI_INVALID_ARGUMENT, "mixed_cg_solve: the outer matrix must hold FP64 values" );
      if( A_lo->value_type != TNLMI_F32 && A_lo->value_type != TNLMI_BF16 )
         fail( TNLMI_INVALID_ARGUMENT, "mixed_cg_solve: the inner matrix must hold FP32 or BF16 values" );
      if( A_lo->rows != A->rows || A_lo->columns != A->columns || A->rows != A->columns )
         fail( TNLMI_INVALID_ARGUMENT, "mixed_cg_solve: the matrices must be square and of one size" );
      if( ! ( delta > 0.0 && delta < 1.0 ) )
         fail( TNLMI_INVALID_ARGUMENT, "mixed_cg_solve: delta must lie in (0, 1)" );
      hipStream_t s = as_stream( stream );
      const int64_t n = A->rows;
      const Operator op{ A, plan, n };
      DeviceArray< double > r64, d64, sc;
      DeviceArray< float > r, p, Ap, xc, d32;
      DeviceArray< CgDev > dev;
      for( auto* v : { &r64, &d64 } )
         v->allocate( n );
      r.allocate( mask_rows_room( n ) );
      for( auto* v : { &p, &Ap, &xc, &d32 } )
         v->allocate( n );
      sc.allocate( 4 );
      dev.allocate( 2 );
      TNLMI_HIP( hipMemsetAsync( p.ptr, 0, sizeof( float ) * n, s ) );
      Parts parts;
      RedWork w;
      HostState hs;
      // Jacobi: d = diag(A) (Diagonal.hpp:27-30); d32 = (float) d
      double dia;
      {
         tnlmi_preconditioner* M = nullptr;
         const tnlmi_status rc = tnlmi_preconditioner_create( TNLMI_PRECOND_DIAGONAL, A, stream, &M );
         if( rc != TNLMI_OK )
            fail( rc, tnlmi_last_error() );
         hipLaunchKernelGGL( to_f32< double >, dim3( kFB32 ), dim3( kFT ), 0, s, n, precond_diagonal( M ), d32.ptr );
         dia = n > kGridRows ? uniform_diagonal( n, precond_diagonal( M ), s ) : std::nan( "" );
         TNLMI_HIP( hipStreamSynchronize( s ) );
         tnlmi_preconditioner_destroy( M );
      }
      nrm2( n, d_b, sc.ptr + 0, w, s );
      double normb = 0;
      TNLMI_HIP( hipMemcpyAsync( &normb, sc.ptr, sizeof( double ), hipMemcpyDeviceToHost, s ) );
      TNLMI_HIP( hipStreamSynchronize( s ) );
      int64_t nupd = 0;
      if( normb == 0.0 ) {
         fill( n, 0.0, d_x, s );
         st->iterations = 0;
         st->residue = 0.0;
         st->converged = 1;
         if( updates )
            *updates = 0;
         return;
      }
      Stage S = make_stage( A_lo, nullptr, s );
      const bool resident = grid_takes< 32 >( S, A_lo->value_type == TNLMI_BF16 ? kFarBf16 : kFar32, s );
      if( S.kind == 1 && ! resident ) {
         make_masks( S, Ap.ptr, s );
         if( ! S.pairs )
            make_codes( S, s );
      }
      DeviceArray< float > room;
      float* pp = p.ptr;
      if( S.pairs ) {
         const int64_t at = S.reach + kMaskRoom;
         room.allocate( n + 2 * at );
         TNLMI_HIP( hipMemsetAsync( room.ptr, 0, sizeof( float ) * ( n + 2 * at ), s ) );
         pp = room.ptr + at;
         p.reset();
      }
      const StopRule R{ st->max_iterations, st->min_iterations, st->convergence_residue, st->divergence_residue };
      int64_t it = 0;
      double res = 0;
      bool first = true;
      int par = 0;  // the state is double-buffered by iteration parity
      std::unique_ptr< GridWork< float > > grid;
      if( resident )
         grid = std::make_unique< GridWork< float > >( s );
      while( true ) {
         // reliable update: r = b - A x in FP64 and the true residual
         op.apply( d_x, r64.ptr, s );
         hipLaunchKernelGGL( resid_part, dim3( kFB32 ), dim3( kFT ), 0, s, n, d_b, r64.ptr, parts.c.ptr );
         hipLaunchKernelGGL( sum_into, dim3( 1 ), dim3( kFT ), 0, s, parts.c.ptr, kFB32, sc.ptr + 1 );
         double rr = 0;
         TNLMI_HIP( hipMemcpyAsync( &rr, sc.ptr + 1, sizeof( double ), hipMemcpyDeviceToHost, s ) );
         TNLMI_HIP( hipStreamSynchronize( s ) );
         res = std::sqrt( rr ) / normb;
         nupd++;
         if( std::isnan( res ) || it > R.maxit || ( res > R.div && it >= R.minit ) || ( res < R.tol && it >= R.minit ) )
            break;
         // replace the FP32 residual by the FP64 one and form the next direction
         CgDev* cur = dev.ptr + par;
         hipLaunchKernelGGL( mx_restart, dim3( kFB32 ), dim3( kFT ), 0, s, n, r64.ptr, r.ptr, d32.ptr, pp, xc.ptr,
                             parts.a.ptr, parts.b.ptr, parts.c.ptr );
         hipLaunchKernelGGL( mx_state, dim3( 1 ), dim3( kFT ), 0, s, cur, parts.a.ptr, parts.b.ptr, parts.c.ptr,
                             sc.ptr + 0, it, first ? 1 : 0, kFB32 );
         hipLaunchKernelGGL( mx_redir, dim3( kFB32 ), dim3( kFT ), 0, s, n, r.ptr, d32.ptr, pp, cur,
                             first ? 1 : 0 );
         first = false;
         const CgDev* h = nullptr;
         int32_t late = 0;
         if( grid ) {
            GridCg< float, float > a{};
            a.x = xc.ptr;
            a.d = d32.ptr;
            a.st = cur;
            a.R = R;
            a.delta2 = delta * delta;
            a.tol = R.tol;
            a.maxit = R.maxit;
            do {
               const auto turn = resident_turn();
               grid->fill( a, S, r.ptr, p.ptr, Ap.ptr );
               const bool launched = A_lo->value_type == TNLMI_F32
                                        ? grid_cg_launch< float, float, float, float, true >( a, s )
                                        : grid_cg_launch< bf16, float, float, float, true >( a, s );
               if( ! launched ) {
                  grid.reset();
                  break;
               }
               TNLMI_HIP( hipMemcpyAsync( &late, grid->late.ptr, sizeof( late ), hipMemcpyDeviceToHost, s ) );
               h = &hs.read( cur, s );
               if( late ) {  // xc is that of the launch's start: replace the residual, and launch by launch from there
                  grid.reset();
                  first = true;
                  break;
               }
            } while( h->active );
         }
         while( ! late && ( ! h || ( ! grid && h->active ) ) ) {
            for( int k = 0; k < kBatch; k++, par ^= 1 ) {
               cur = dev.ptr + par;
               if( S.pairs ) {
                  mask_iteration< float, float, float, true >(
                     S, r.ptr, pp, xc.ptr, std::isnan( dia ) ? d32.ptr : nullptr, (float) dia, parts.a.ptr, parts.b.ptr,
                     parts.c.ptr, cur, dev.ptr + ( par ^ 1 ), R, delta * delta, s );
                  continue;
               }
               stage_launch< float >( S, p.ptr, Ap.ptr, parts.a.ptr, cur, s );
               hipLaunchKernelGGL( ( cg_upd< float, float, float > ), dim3( kFB32 ), dim3( kFT ), 0, s, n, parts.a.ptr,
                                   r.ptr, p.ptr, Ap.ptr, xc.ptr, d32.ptr, parts.b.ptr, parts.c.ptr, cur );
               hipLaunchKernelGGL( mx_dir, dim3( kFB32 ), dim3( kFT ), 0, s, n, parts.a.ptr, parts.b.ptr, parts.c.ptr,
                                   r.ptr, d32.ptr, p.ptr, cur, dev.ptr + ( par ^ 1 ), delta * delta, R.tol, R.maxit );
            }
            TNLMI_HIP( hipGetLastError() );
            h = &hs.read( dev.ptr + par, s );
         }
         it = h->it;
         hipLaunchKernelGGL( mx_accumulate, dim3( kFB32 ), dim3( kFT ), 0, s, n, xc.ptr, d_x );
      }
      st->iterations = it;
      st->residue = res;
      st->converged = ! std::isnan( res ) && res <= R.tol && it <= R.maxit ? 1 : 0;
      if( updates )
         *updates = nupd;
   } );
}

}  // extern "C"
