// krylov_resident.hip -- BiCGStab and GMRES with their iterations in one
// resident launch (the whole grid stays on the chip; grid_sum.hpp), for
// matrices of at most 2^20 rows with Ellpack slots and no or the Diagonal
// preconditioner.
//
// Launch by launch, an iteration is 20 (BiCGStab) or 3 per basis vector and pass
// (GMRES, modified Gram-Schmidt) kernels that each last about as long as a
// launch.  Here a thread keeps its rows of the vectors in registers, sums end
// in grid sums of about 2.5 us, and a vector that other workgroups multiply by A
// goes through memory once.
//
// Convection-diffusion, per iteration against launch by launch: GMRES(10) with
// modified Gram-Schmidt twice on 200^2 40 against 199 us, GMRES(20) on 1024^2 154
// against 339 us; GMRES(30) with classical Gram-Schmidt twice on 120^2 27 against
// 84 us, on 1024^2 111 against 173 us (the basis read three times, 390 MB on
// average, is most of it); BiCGStab on 100^2 15 against 98 us, 500^2 30 against
// 98 us, 1024^2 66 against 125 us.  Small systems: 2 grid sums per basis vector of
// modified Gram-Schmidt, 5 per BiCGStab iteration, 2.2 us each.
#include <algorithm>
#include <type_traits>

#include "blas1.hpp"
#include "grid_sum.hpp"
#include "krylov.hpp"

namespace tnlmi {

class Resident
{
public:
   double* pub[ 2 ];  // vectors that every workgroup reads
   DeviceArray< GridSlots > slots;
   DeviceArray< ResidentState > state;
   DeviceArray< int32_t > late;  // a grid sum was given up
   uint32_t number = 1;
};

std::shared_ptr< Resident > resident_work( double* pub0, double* pub1, hipStream_t s )
{
   auto w = std::make_shared< Resident >();
   w->pub[ 0 ] = pub0;
   w->pub[ 1 ] = pub1;
   w->slots.allocate( 1 );
   w->state.allocate( 1 );
   w->late.allocate( 1 );
   TNLMI_HIP( hipMemsetAsync( w->slots.ptr, 0, sizeof( GridSlots ), s ) );
   TNLMI_HIP( hipMemsetAsync( w->late.ptr, 0, sizeof( int32_t ), s ) );
   return w;
}

namespace {

constexpr int kWidth = 8;          // slots loaded together
constexpr int32_t kMost = 2048;    // iterations per launch

struct Common
{
   int64_t n, stride;
   int32_t w;
   const int32_t* cols;
   const double* vals;
   const double* d;
   double* pub[ 2 ];
   GridSlots* slots;
   ResidentState* st;
   int32_t* late;
   uint64_t wait;
   uint32_t number;
   int64_t maxit, minit;
   double tol, div;
};

__device__ __forceinline__ bool goes_on( const Common& c, double res, int64_t it )
{
   return ! ( isnan( res ) || it > c.maxit || ( res > c.div && it >= c.minit ) || ( res < c.tol && it >= c.minit ) );
}

// This thread's ROWS rows (row j: r0 + j * THREADS) of a matrix; with KEEP
// their entries stay in registers.
template< int THREADS, int ROWS, bool KEEP >
struct Rows
{
   const Common& c;
   int32_t base;
   int64_t r0;
   int32_t kc[ KEEP ? ROWS : 1 ][ kWidth ];
   double kv[ KEEP ? ROWS : 1 ][ kWidth ];
   __device__ __forceinline__ explicit Rows( const Common& c_ ) : c( c_ )
   {
      base = (int32_t) ( blockIdx.x * ( THREADS * ROWS ) );
      r0 = base + threadIdx.x;
      if( KEEP )
#pragma unroll
         for( int j = 0; j < ROWS; j++ )
#pragma unroll
            for( int k = 0; k < kWidth; k++ ) {
               const bool there = in( j ) && k < c.w;
               kc[ j ][ k ] = there ? c.cols[ k * c.stride + row( j ) ] : -1;
               kv[ j ][ k ] = there ? c.vals[ k * c.stride + row( j ) ] : 0.0;
            }
   }
   __device__ __forceinline__ int64_t row( int j ) const { return r0 + j * THREADS; }
   __device__ __forceinline__ bool in( int j ) const { return row( j ) < c.n; }
   __device__ __forceinline__ double load( const double* v, int j, double other = 0.0 ) const
   {
      return in( j ) ? v[ row( j ) ] : other;
   }
   __device__ __forceinline__ void store( double* v, int j, double x ) const
   {
      if( in( j ) )
         v[ row( j ) ] = x;
   }
   // this workgroup's rows of a vector to LDS (own) and to pub, for product
   __device__ __forceinline__ void publish( double* pub, double* own, int j, double x ) const
   {
      own[ j * THREADS + threadIdx.x ] = x;
      if( in( j ) )
         shared_store( pub + row( j ), x );
   }
   // y = A (scale v) over this thread's rows; v: own rows in LDS, others in pub
   // (row by row: the rows' loads together would not fit the registers)
   static __device__ __forceinline__ void next_row()
   {
      if( ROWS > 1 )
         __builtin_amdgcn_sched_barrier( 0 );
   }
   __device__ __forceinline__ void product( const double* pub, const double* own, double scale, double ( &y )[ ROWS ] ) const
   {
      auto at = [ & ]( int32_t col ) {
         const uint32_t l = (uint32_t) ( col - base );
         return scale * ( l < (uint32_t) ( THREADS * ROWS ) ? own[ l ] : shared_load( pub + col ) );
      };
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         y[ j ] = 0;
         if( KEEP ) {
            double g[ kWidth ];
#pragma unroll
            for( int k = 0; k < kWidth; k++ )
               g[ k ] = kc[ j ][ k ] >= 0 ? at( kc[ j ][ k ] ) : 0.0;
#pragma unroll
            for( int k = 0; k < kWidth; k++ )
               if( kc[ j ][ k ] >= 0 )
                  y[ j ] += kv[ j ][ k ] * g[ k ];
         }
         else if( in( j ) )
            for( int32_t k0 = 0; k0 < c.w; k0 += kWidth ) {
               int32_t cl[ kWidth ];
               double v[ kWidth ], g[ kWidth ];
#pragma unroll
               for( int k = 0; k < kWidth; k++ ) {
                  const bool there = k0 + k < c.w;
                  cl[ k ] = there ? c.cols[ ( k0 + k ) * c.stride + row( j ) ] : -1;
                  v[ k ] = there ? c.vals[ ( k0 + k ) * c.stride + row( j ) ] : 0.0;
               }
#pragma unroll
               for( int k = 0; k < kWidth; k++ )
                  g[ k ] = cl[ k ] >= 0 ? at( cl[ k ] ) : 0.0;
#pragma unroll
               for( int k = 0; k < kWidth; k++ )
                  if( cl[ k ] >= 0 )
                     y[ j ] += v[ k ] * g[ k ];
            }
         next_row();
      }
   }
};

// ---------------------------------------------------------------- BiCGStab
// scalars of the solver's array (krylov_ns.hip)
enum { kRho, kRhoOld, kAlpha, kOmega, kBeta, kBnorm, kRast, kApR, kAsS, kAsAs, kRhoNew, kRnorm, kFlag };

struct BicgArgs : Common
{
   const double* rast;
   double *r, *p, *Ap, *x, *sc;
   double b_norm, eps2;
};

template< int THREADS, int ROWS, bool KEEP >
__global__ void __launch_bounds__( THREADS ) bicgstab_resident( BicgArgs a )
{
   __shared__ double sm[ 2 * THREADS / 64 ];
   __shared__ double own[ THREADS * ROWS ];
   const Rows< THREADS, ROWS, KEEP > R( a );
   double r[ ROWS ], p[ ROWS ], Ap[ ROWS ], s[ ROWS ];
#pragma unroll
   for( int j = 0; j < ROWS; j++ ) {
      r[ j ] = R.load( a.r, j );
      p[ j ] = R.load( a.p, j );
   }
   double rho = a.sc[ kRho ], rho_old = rho, alpha = 0, omega = 0, beta = 0, res = 0;
   const double rast2 = a.sc[ kRast ];
   int64_t it = a.st->it;
   uint32_t number = a.number;
   int32_t end = kResidentMore;
   for( int32_t done = 0; done < kMost; done++ ) {
#pragma unroll
      for( int j = 0; j < ROWS; j++ )
         R.publish( a.pub[ 0 ], own, j, p[ j ] );
      if( ! grid_barrier< THREADS >( a.slots, number++, a.wait, sm ) ) {
         end = kResidentLate;
         break;
      }
      R.product( a.pub[ 0 ], own, 1.0, Ap );
      double one[ 1 ] = { 0 };
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         if( a.d )
            Ap[ j ] = Ap[ j ] / R.load( a.d, j, 1.0 );
         one[ 0 ] += Ap[ j ] * R.load( a.rast, j );
      }
      if( ! grid_sum< THREADS >( one, a.slots, number++, a.wait, sm ) ) {
         end = kResidentLate;
         break;
      }
      alpha = rho / one[ 0 ];
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         s[ j ] = r[ j ] - alpha * Ap[ j ];
         R.publish( a.pub[ 1 ], own, j, s[ j ] );
      }
      if( ! grid_barrier< THREADS >( a.slots, number++, a.wait, sm ) ) {
         end = kResidentLate;
         break;
      }
      double As[ ROWS ];
      R.product( a.pub[ 1 ], own, 1.0, As );
      double two[ 2 ] = { 0, 0 };
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         if( a.d )
            As[ j ] = As[ j ] / R.load( a.d, j, 1.0 );
         two[ 0 ] += As[ j ] * s[ j ];
         two[ 1 ] += As[ j ] * As[ j ];
      }
      if( ! grid_sum< THREADS >( two, a.slots, number++, a.wait, sm ) ) {
         end = kResidentLate;
         break;
      }
      omega = two[ 0 ] / two[ 1 ];
      two[ 0 ] = two[ 1 ] = 0;
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         R.store( a.x, j, R.load( a.x, j ) + ( alpha * p[ j ] + omega * s[ j ] ) );
         r[ j ] = s[ j ] - omega * As[ j ];
         two[ 0 ] += r[ j ] * R.load( a.rast, j );
         two[ 1 ] += r[ j ] * r[ j ];
      }
      if( ! grid_sum< THREADS >( two, a.slots, number++, a.wait, sm ) ) {
         end = kResidentLate;
         break;
      }
      rho_old = rho;
      rho = two[ 0 ];
      beta = ( rho / rho_old ) * ( alpha / omega );
      if( fabs( rho ) < a.eps2 * rast2 ) {  // the host restarts with r* = r
         end = kResidentRestart;
         break;
      }
      const double bw = beta * omega;
#pragma unroll
      for( int j = 0; j < ROWS; j++ )
         p[ j ] = r[ j ] + beta * p[ j ] - bw * Ap[ j ];
      res = sqrt( two[ 1 ] ) / a.b_norm;
      const bool go = goes_on( a, res, it );
      it++;
      if( ! go ) {
         end = kResidentStopped;
         break;
      }
   }
   if( end == kResidentLate ) {
      if( threadIdx.x == 0 )
         *a.late = 1;
      return;
   }
#pragma unroll
   for( int j = 0; j < ROWS; j++ ) {
      R.store( a.r, j, r[ j ] );
      R.store( a.p, j, p[ j ] );
      R.store( a.Ap, j, Ap[ j ] );
   }
   if( blockIdx.x == 0 && threadIdx.x == 0 ) {
      a.sc[ kRho ] = rho;
      a.sc[ kRhoOld ] = rho_old;
      a.sc[ kAlpha ] = alpha;
      a.sc[ kOmega ] = omega;
      a.sc[ kBeta ] = beta;
      a.st->res = res;
      a.st->it = it;
      a.st->end = end;
   }
}

// ------------------------------------------------------------------- GMRES
struct GmresArgs : Common
{
   const double* b;
   double *r, *V, *x;
   int64_t ld;
   int32_t passes, rmin, rmax, dmin, dmax;
   double normb;
};

constexpr int kM = 31;  // basis vectors at most (the solver refuses more)

struct Small  // a cycle's least-squares problem, the same in every workgroup
{
   double H[ ( kM + 1 ) * kM ];  // column i at i * ( kM + 1 )
   double s[ kM + 1 ], cs[ kM + 1 ], sn[ kM + 1 ], y[ kM + 1 ];
   double h[ kGridValues ];
   double res;
   int32_t zero_pivot;
};

__device__ __forceinline__ void rotate( double& dx, double& dy, double c, double sn )
{
   const double t = c * dx + sn * dy;
   dy = c * dy - sn * dx;
   dx = t;
}

// Givens rotations of column i, its norm known (GMRES.hpp:729-770); one thread
__device__ __forceinline__ void givens( Small& g, int i, double norm, double normb )
{
   double* H = g.H + i * ( kM + 1 );
   H[ i + 1 ] = norm;
   for( int k = 0; k < i; k++ )
      rotate( H[ k ], H[ k + 1 ], g.cs[ k ], g.sn[ k ] );
   if( H[ i + 1 ] != 0.0 ) {
      const double dx = H[ i ], dy = H[ i + 1 ];
      double c, sn;
      if( fabs( dy ) > fabs( dx ) ) {
         const double t = dx / dy;
         sn = 1.0 / sqrt( 1.0 + t * t );
         c = t * sn;
      }
      else {
         const double t = dy / dx;
         c = 1.0 / sqrt( 1.0 + t * t );
         sn = t * c;
      }
      g.cs[ i ] = c;
      g.sn[ i ] = sn;
      rotate( H[ i ], H[ i + 1 ], c, sn );
      rotate( g.s[ i ], g.s[ i + 1 ], c, sn );
   }
   g.res = fabs( g.s[ i + 1 ] ) / normb;
}

// y = H^-1 s on the leading (k + 1) x (k + 1) block; the first wave (a lane per
// row, columns from the last, as the serial substitution)
__device__ __forceinline__ void back_substitute( Small& g, int k )
{
   const int j = threadIdx.x;
   double y = j <= k ? g.s[ j ] : 0.0;
   bool zero = false;
   for( int i = k; i >= 0; i-- ) {
      const double hii = g.H[ i * ( kM + 1 ) + i ];
      zero = zero || hii == 0.0;
      if( j == i )
         y /= hii;
      const double yi = __shfl( y, i, 64 );
      if( j < i )
         y -= g.H[ i * ( kM + 1 ) + j ] * yi;
   }
   if( j <= k )
      g.y[ j ] = y;
   if( j == 0 )
      g.zero_pivot = zero ? 1 : 0;
}

template< int THREADS, int ROWS, bool KEEP, bool CLASSICAL >
__global__ void __launch_bounds__( THREADS ) gmres_resident( GmresArgs a )
{
   constexpr int W = THREADS / 64;
   constexpr int kGroup = kDotGroup;  // basis vectors read together
   constexpr int kHalf = kGridValues / 2;
   __shared__ double sm[ kGridValues * W ];
   __shared__ double own[ THREADS * ROWS ];
   __shared__ Small g;
   const Rows< THREADS, ROWS, KEEP > R( a );
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   ResidentState st = *a.st;
   uint32_t number = a.number;
   int32_t end = kResidentMore, done = 0;
   double w[ ROWS ];
#pragma unroll
   for( int j = 0; j < ROWS; j++ )
      w[ j ] = R.load( a.r, j );
   bool late = false;
   auto barrier = [ & ] { late = late || ! grid_barrier< THREADS >( a.slots, number++, a.wait, sm ); };
   auto sum = [ & ]( double ( &v )[ 1 ] ) {
      late = late || ! grid_sum< THREADS >( v, a.slots, number++, a.wait, sm );
      v[ 0 ] = wave_uniform( v[ 0 ] );  // (also where no sum was taken: what follows from it branches)
   };
   // sums of `count` values, value k's per-thread part in acc[ k - k0 ] for the group at k0
   auto put = [ & ]( double ( &acc )[ kGroup ], int k0, int count ) {
      const double t = wave_sum_group( acc );  // lane l: value l >> 3
      if( ( lane & 7 ) == 0 && k0 + ( lane >> 3 ) < count )
         sm[ ( k0 + ( lane >> 3 ) ) * W + wave ] = t;
   };
   // publish the residual: v_0 = r / beta
#pragma unroll
   for( int j = 0; j < ROWS; j++ )
      R.publish( a.pub[ 0 ], own, j, w[ j ] );
   barrier();
   while( ! late ) {
      int m = st.m;
      if( a.rmax > a.rmin && st.cycles > 0 ) {  // Baker-Jessup-Kolev adaptive restart, GMRES.hpp:121-146
         if( st.beta_ratio > 0.99 )
            m = a.rmax;
         else if( st.beta_ratio >= 0.175 ) {
            const int step = a.dmin + ( a.dmax - a.dmin ) / static_cast< float >( a.rmax - a.rmin ) * ( m - a.rmin );
            m = m - step >= a.rmin ? m - step : a.rmax;
         }
      }
      st.m = m;
      for( int i = threadIdx.x; i < kM + 1; i += THREADS )
         g.s[ i ] = i == 0 ? st.beta : 0.0;
      double norm = st.beta;  // of the published vector
      int o = m;
      __syncthreads();
      for( int i = 0; i < m; i++ ) {
         if( ! goes_on( a, st.res, st.it++ ) ) {
            o = -1;  // (the check after the step before has ended the cycle)
            end = kResidentStopped;
            break;
         }
         const double inv = 1.0 / norm;
         double* vi = a.V + (int64_t) i * a.ld;
#pragma unroll
         for( int j = 0; j < ROWS; j++ )
            R.store( vi, j, inv * w[ j ] );
         {
            double y[ ROWS ];
            R.product( a.pub[ 0 ], own, inv, y );
#pragma unroll
            for( int j = 0; j < ROWS; j++ )
               w[ j ] = a.d ? y[ j ] / R.load( a.d, j, 1.0 ) : y[ j ];
         }
         double* H = g.H + i * ( kM + 1 );
         const int count = i + 1;
         if constexpr( CLASSICAL ) {
            // the dots of the first pass; then per pass the update, which also
            // takes the next pass's dots while a row's entries of the basis are in
            // registers (the basis is read passes + 1 times).  w is in LDS here:
            // the loops over rows stay loops, with all registers for one row
            __syncthreads();
#pragma unroll
            for( int j = 0; j < ROWS; j++ )
               own[ j * THREADS + threadIdx.x ] = w[ j ];
            for( int pass = 0; pass <= a.passes; pass++ ) {
               if( pass > 0 ) {
                  late = late || ! grid_sum_many< THREADS >( count, a.slots, number++, a.wait, sm, g.h );
                  if( (int) threadIdx.x < count )
                     H[ threadIdx.x ] = pass == 1 ? g.h[ threadIdx.x ] : H[ threadIdx.x ] + g.h[ threadIdx.x ];
               }
               double acc[ kGridValues ];
#pragma unroll
               for( int k = 0; k < kGridValues; k++ )
                  acc[ k ] = 0;
#pragma clang loop unroll( disable )
               for( int j = 0; j < ROWS; j++ ) {
                  if( ! R.in( j ) )
                     break;
                  const uint32_t at = (uint32_t) R.row( j ) * 8u;
                  double v[ kHalf ];  // half of the basis's entries of the row at a time
                  auto load = [ & ]( int k0 ) {
#pragma unroll
                     for( int u = 0; u < kHalf; u++ )
                        if( k0 + u / kGroup * kGroup < count )
                           v[ u ] = *(const double*) ( (const char*) ( a.V + (int64_t) min( k0 + u, i ) * a.ld ) + at );
                  };
                  double wj = own[ j * THREADS + threadIdx.x ];
                  if( pass > 0 ) {
                     double t = 0;
                     for( int k0 = 0; k0 < count; k0 += kHalf ) {
                        load( k0 );
#pragma unroll
                        for( int u = 0; u < kHalf; u++ )
                           if( k0 + u < count )
                              t += v[ u ] * g.h[ k0 + u ];
                     }
                     wj = wj - t;
                     own[ j * THREADS + threadIdx.x ] = wj;
                  }
                  if( pass < a.passes ) {
                     // the upper half, if there is one, is still there
                     if( count > kHalf ) {
                        if( pass == 0 )
                           load( kHalf );
#pragma unroll
                        for( int u = 0; u < kHalf; u++ )
                           if( kHalf + u / kGroup * kGroup < count )
                              acc[ kHalf + u ] += wj * v[ u ];
                     }
                     if( pass == 0 || count > kHalf )
                        load( 0 );
#pragma unroll
                     for( int u = 0; u < kHalf; u++ )
                        if( u / kGroup * kGroup < count )
                           acc[ u ] += wj * v[ u ];
                  }
               }
               if( pass < a.passes )
#pragma unroll
                  for( int q = 0; q < kGridValues / kGroup; q++ )
                     if( q * kGroup < count ) {
                        double part[ kGroup ];
#pragma unroll
                        for( int u = 0; u < kGroup; u++ )
                           part[ u ] = acc[ q * kGroup + u ];
                        put( part, q * kGroup, count );
                     }
            }
#pragma unroll
            for( int j = 0; j < ROWS; j++ )
               w[ j ] = own[ j * THREADS + threadIdx.x ];
         }
         else {
            double v[ ROWS ];
#pragma unroll
            for( int j = 0; j < ROWS; j++ )
               v[ j ] = R.load( a.V, j );
            for( int pass = 0; pass < a.passes; pass++ )
               for( int k = 0; k < count; k++ ) {
                  double h[ 1 ] = { 0 }, next[ ROWS ];
                  const double* vn = a.V + (int64_t) ( k + 1 < count ? k + 1 : 0 ) * a.ld;
#pragma unroll
                  for( int j = 0; j < ROWS; j++ ) {
                     h[ 0 ] += w[ j ] * v[ j ];
                     next[ j ] = R.load( vn, j );  // (arrives while the sum does)
                  }
                  sum( h );
                  if( threadIdx.x == 0 )
                     H[ k ] = pass == 0 ? h[ 0 ] : H[ k ] + h[ 0 ];
#pragma unroll
                  for( int j = 0; j < ROWS; j++ ) {
                     w[ j ] = w[ j ] - h[ 0 ] * v[ j ];
                     v[ j ] = next[ j ];
                  }
               }
         }
         // the norm; its sum also passes w on to all workgroups
         double ww[ 1 ] = { 0 };
#pragma unroll
         for( int j = 0; j < ROWS; j++ ) {
            R.publish( a.pub[ 0 ], own, j, w[ j ] );
            ww[ 0 ] += w[ j ] * w[ j ];
         }
         sum( ww );
         if( late )
            break;
         norm = sqrt( ww[ 0 ] );
         if( threadIdx.x == 0 )
            givens( g, i, norm, a.normb );
         __syncthreads();
         st.res = wave_uniform( g.res );
         done++;
         if( ! goes_on( a, st.res, st.it ) ) {
            o = i;
            break;
         }
      }
      if( late || o < 0 )
         break;
      // x += V y
      const int k = o < m ? o : m - 1;
      if( threadIdx.x < 64 )
         back_substitute( g, k );
      __syncthreads();
      if( wave_uniform( g.zero_pivot ) ) {
         end = kResidentZeroPivot;
         break;
      }
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         double acc = 0;
         for( int k0 = 0; k0 <= k; k0 += kGroup ) {
            double v[ kGroup ];
#pragma unroll
            for( int u = 0; u < kGroup; u++ )
               v[ u ] = R.load( a.V + (int64_t) min( k0 + u, k ) * a.ld, j );
#pragma unroll
            for( int u = 0; u < kGroup; u++ )
               if( k0 + u <= k )
                  acc += v[ u ] * g.y[ k0 + u ];
         }
         const double x = R.load( a.x, j ) + acc;
         R.store( a.x, j, x );
         R.publish( a.pub[ 1 ], own, j, x );
         R.next_row();
      }
      if( o < m ) {
         end = kResidentStopped;
         break;
      }
      barrier();
      // r = M^-1 (b - A x)
      double y[ ROWS ], rr[ 1 ] = { 0 };
      R.product( a.pub[ 1 ], own, 1.0, y );
      __syncthreads();  // (own is written below)
#pragma unroll
      for( int j = 0; j < ROWS; j++ ) {
         w[ j ] = R.load( a.b, j ) - y[ j ];
         if( a.d )
            w[ j ] = w[ j ] / R.load( a.d, j, 1.0 );
         R.publish( a.pub[ 0 ], own, j, w[ j ] );
         rr[ 0 ] += w[ j ] * w[ j ];
      }
      sum( rr );
      if( late )
         break;
      const double old = st.beta;
      st.beta = sqrt( rr[ 0 ] );
      st.res = st.beta / a.normb;
      st.cycles++;
      st.beta_ratio = st.beta / old;
      if( ! goes_on( a, st.res, st.it ) ) {
         end = kResidentStopped;
         break;
      }
      if( done + a.rmax > kMost )
         break;
   }
   if( late ) {
      if( threadIdx.x == 0 )
         *a.late = 1;
      return;
   }
#pragma unroll
   for( int j = 0; j < ROWS; j++ )
      R.store( a.r, j, w[ j ] );
   if( blockIdx.x == 0 && threadIdx.x == 0 ) {
      st.end = end;
      *a.st = st;
   }
}

// ------------------------------------------------------------------ launches
void fill_common( Common& c, Resident& w, const EllSlots& A, const double* d, const Stop& S )
{
   c.n = A.n;
   c.stride = A.stride;
   c.w = A.w;
   c.cols = A.cols;
   c.vals = A.vals;
   c.d = d;
   c.pub[ 0 ] = w.pub[ 0 ];
   c.pub[ 1 ] = w.pub[ 1 ];
   c.slots = w.slots.ptr;
   c.st = w.state.ptr;
   c.late = w.late.ptr;
   c.wait = grid_wait();
   c.number = w.number;
   c.maxit = S.st->max_iterations;
   c.minit = S.st->min_iterations;
   c.tol = S.st->convergence_residue;
   c.div = S.st->divergence_residue;
}

template< typename Args >
bool launch( const void* kernel, int threads, int rows, Args& a, hipStream_t s )
{
   void* args[] = { &a };
   return resident_launch( kernel, ceil_div( a.n, (int64_t) threads * rows ), threads, args, s );
}

void put_state( Resident& w, const ResidentState& h, hipStream_t s )
{
   TNLMI_HIP( hipMemcpyAsync( w.state.ptr, &h, sizeof( h ), hipMemcpyHostToDevice, s ) );
}
// (where any workgroup gave up: kResidentLate, whatever state the others left)
ResidentState get_state( Resident& w, hipStream_t s )
{
   ResidentState h;
   int32_t late = 0;
   TNLMI_HIP( hipMemcpyAsync( &h, w.state.ptr, sizeof( h ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipMemcpyAsync( &late, w.late.ptr, sizeof( late ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   if( late )
      h.end = kResidentLate;
   return h;
}

}  // namespace

// Threads and rows per thread.  60 iterations on 450^2, 700^2 and 1000^2 grids with
// 1,024 threads (1, 2 and 4 rows) against 512 (2, 4 and 8): BiCGStab 1.94 / 1.88, 2.56 /
// 2.56, 3.98 / 3.72 ms; GMRES(20) CGSR 3.66 / 2.38, 4.87 / 3.78, 7.26 / 5.54 ms (with 128
// registers the 32 sums of a pass spill 131), GMRES(10) MGSR 3.63 / 3.25, 4.17 / 4.03,
// 5.39 / 5.38 ms.  Past 2^20 rows, launch by launch: BiCGStab 67 -> 123 us an iteration at
// 1025^2, GMRES(20) CGSR 93 -> 158, GMRES(10) MGSR 91 -> 200.
ResidentEnd resident_bicgstab( Resident& w, const ResidentBicgstab& q, Stop& S, hipStream_t s )
{
   BicgArgs a{};
   fill_common( a, w, q.A, q.d, S );
   a.rast = q.rast;
   a.r = q.r;
   a.p = q.p;
   a.Ap = q.Ap;
   a.x = q.x;
   a.sc = q.sc;
   a.b_norm = q.b_norm;
   a.eps2 = q.eps2;
   ResidentState h{};
   h.it = S.it;
   const auto turn = resident_turn();  // (until get_state)
   put_state( w, h, s );
   const bool keep = a.w <= kWidth;
   const int64_t n = a.n;
   bool ok;
   if( n <= (int64_t) kGridMax * 256 )
      ok = keep ? launch( (const void*) bicgstab_resident< 256, 1, true >, 256, 1, a, s )
                : launch( (const void*) bicgstab_resident< 256, 1, false >, 256, 1, a, s );
   else if( n <= (int64_t) kGridMax * 512 )
      ok = launch( (const void*) bicgstab_resident< 512, 1, false >, 512, 1, a, s );
   else if( n <= (int64_t) kGridMax * 1024 )
      ok = launch( (const void*) bicgstab_resident< 1024, 1, false >, 1024, 1, a, s );
   else if( n <= (int64_t) kGridMax * 2048 )
      ok = launch( (const void*) bicgstab_resident< 1024, 2, false >, 1024, 2, a, s );
   else if( n <= (int64_t) kGridMax * 4096 )
      ok = launch( (const void*) bicgstab_resident< 1024, 4, false >, 1024, 4, a, s );
   else
      ok = false;
   if( ! ok )
      return kResidentNot;
   w.number += 5 * kMost;
   h = get_state( w, s );
   if( h.end != kResidentLate ) {
      S.it = h.it;
      S.res = h.res;
   }
   return (ResidentEnd) h.end;
}

ResidentEnd resident_gmres( Resident& w, const ResidentGmres& q, Stop& S, double& beta, double& beta_ratio, int& cycles,
                            int& m, hipStream_t s )
{
   GmresArgs a{};
   fill_common( a, w, q.A, q.d, S );
   a.b = q.b;
   a.r = q.r;
   a.V = q.V;
   a.x = q.x;
   a.ld = q.ld;
   a.passes = q.passes;
   a.rmin = q.rmin;
   a.rmax = q.rmax;
   a.dmin = q.dmin;
   a.dmax = q.dmax;
   a.normb = q.normb;
   ResidentState h{};
   h.res = S.res;
   h.it = S.it;
   h.beta = beta;
   h.beta_ratio = beta_ratio;
   h.cycles = cycles;
   h.m = m;
   const auto turn = resident_turn();  // (until get_state)
   put_state( w, h, s );
   const bool keep = a.w <= kWidth;
   const int64_t n = a.n;
   bool ok;
   auto go = [ & ]( auto classical ) {
      constexpr bool C = decltype( classical )::value;
      if( n <= (int64_t) kGridMax * 256 )
         return keep ? launch( (const void*) gmres_resident< 256, 1, true, C >, 256, 1, a, s )
                     : launch( (const void*) gmres_resident< 256, 1, false, C >, 256, 1, a, s );
      if( n <= (int64_t) kGridMax * 512 )
         return launch( (const void*) gmres_resident< 512, 1, false, C >, 512, 1, a, s );
      if( n <= (int64_t) kGridMax * 1024 )
         return launch( (const void*) gmres_resident< 512, 2, false, C >, 512, 2, a, s );
      if( n <= (int64_t) kGridMax * 2048 )
         return launch( (const void*) gmres_resident< 512, 4, false, C >, 512, 4, a, s );
      if( n <= (int64_t) kGridMax * 4096 )
         return launch( (const void*) gmres_resident< 512, 8, false, C >, 512, 8, a, s );
      return false;
   };
   ok = q.classical ? go( std::true_type() ) : go( std::false_type() );
   if( ! ok )
      return kResidentNot;
   // sums per iteration: one per basis vector and pass, the norm, two more per cycle
   w.number += ( kMost + kM ) * ( 2 * kM + 4 );
   h = get_state( w, s );
   if( h.end != kResidentLate ) {
      S.it = h.it;
      S.res = h.res;
      beta = h.beta;
      beta_ratio = h.beta_ratio;
      cycles = h.cycles;
      m = h.m;
   }
   return (ResidentEnd) h.end;
}

}  // namespace tnlmi
