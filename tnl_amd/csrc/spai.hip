// spai.hip -- the learned sparse approximate inverse: a message-passing
// network over the graph of A (an edge per nonzero, CSR order) whose output
// is M = D^-1 (I + O) on A's own pattern, a left preconditioner for GMRES.
//
// Network (hidden 64, 3 layers), every 64 x 64 dense layer a BF16 GEMM on
// the matrix cores (v_mfma_f32_16x16x16bf16_1k, FP32 accumulation), BF16
// activations:
//   encoder  E = relu(x_e Ae + ae), H = relu(x_i An + an)      (4 inputs, FP32)
//   layer    P = H Wu, Q = H Wv                                 (FP32)
//            E = relu(E We + P[col] + Q[row] + be)              (fused epilogue)
//            G = mean of the row's E
//            H = relu(H Wh + G Wg + bh)                         (two-term GEMM)
//   decoder  o = E wo + bo,  M_ij = (delta_ij + o_ij) / a_ii
// Training: probe loss L = sum_k ||z_k - M A z_k||^2 / (K n) over Rademacher
// z_k, hand-written backward kernels (MFMA GEMMs with transposed weights for
// the input gradients, LDS-staged MFMA X^T dY for the weight gradients with
// per-block partial sums reduced in block order: deterministic), Adam.
//
// No reference counterpart (TNL has no learned preconditioner).  The CPU
// specification is oracle/spai_oracle.py.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>
#include <vector>

#include "segments.hpp"
#include "spmv.hpp"

namespace tnlmi {
namespace {

constexpr int kH = 64;       // hidden width
constexpr int kL = 3;        // message-passing layers
constexpr int kMats = 5;     // We, Wu, Wv, Wh, Wg per layer
constexpr int kWRows = 256;  // rows per block of the weight-gradient kernel

// flat parameter layout (the oracle's param_shapes order)
constexpr int64_t oAe = 0, oae = 256, oAn = 320, oan = 576, oLayer0 = 640;
constexpr int64_t kLayerSize = kMats * kH * kH + 2 * kH;
constexpr int64_t owo = oLayer0 + kL * kLayerSize, obo = owo + kH;
constexpr int64_t kParams = obo + 1;
__host__ __device__ constexpr int64_t oW( int l, int m )
{
   return oLayer0 + l * kLayerSize + (int64_t) m * kH * kH;
}
__host__ __device__ constexpr int64_t obe( int l )
{
   return oLayer0 + l * kLayerSize + kMats * kH * kH;
}
__host__ __device__ constexpr int64_t obh( int l )
{
   return obe( l ) + kH;
}
enum { mWe = 0, mWu = 1, mWv = 2, mWh = 3, mWg = 4 };

typedef float f4 __attribute__( ( ext_vector_type( 4 ) ) );

__device__ __forceinline__ uint16_t bf( float f )
{
   return float_to_bf16( f );
}
__device__ __forceinline__ float fb( uint16_t b )
{
   return bf16_to_float( b );
}

// ------------------------------------------------------------- dense layers
// Y[R x 64] = sum_t X_t[R x 64] B_t[64 x 64], X_t BF16 row-major, B_t given
// as Bn[n][k] = B[k][n] (BF16).  A wavefront has all of B_t in registers (as the
// first operand of v_mfma_f32_16x16x32_bf16, so that a lane ends up with 4
// consecutive columns of one row: 8- and 16-byte epilogue accesses) and takes
// kTiles tiles of 16 rows.  Bound by memory (32 flop per byte): the layer over
// 326 K edges (EPI_EDGE) takes 40 us for 84 MB of edges and 84 + 84 MB of gathered
// P and Q, most of them in L2, against 89 us with 16x16x16 products, weights read
// per 16 rows and 2-byte stores; the backward one (EPI_DEDGE) 41 us against 70 + 66
// us for the product and a separate pass.
// MFMA 16x16x32 operand layout: lane l holds row l % 16, k = 8 (l / 16) + 0..7
// of either operand (any order of k would do: both have the same), and of the
// result rows 4 (l / 16) + 0..3 (columns of Y), column l % 16 (a row of Y).
typedef __bf16 bf8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef uint16_t u4 __attribute__( ( ext_vector_type( 4 ) ) );
struct Term
{
   const uint16_t* X;
   const uint16_t* Bn;
};
enum Epi { EPI_STORE = 0, EPI_EDGE, EPI_NODE, EPI_DNODE, EPI_DMEAN, EPI_DEDGE };
struct EpiArgs
{
   float* yf;            // EPI_STORE, EPI_DMEAN (FP32 out)
   uint16_t* yb;         // the others (BF16 out)
   const float* bias;    // EPI_EDGE / EPI_NODE
   const float* P;       // EPI_EDGE: + P[col[r]] + Q[row[r]];  EPI_DEDGE: + P[row[r]]
   const float* Q;
   const int32_t* col;
   const int32_t* row;
   const uint16_t* mask;  // EPI_DNODE / EPI_DEDGE: 0 where the activation is not positive
   const int32_t* deg;    // EPI_DMEAN: / deg[r]
};

__device__ __forceinline__ f4 relu4( f4 v )
{
   return f4{ fmaxf( v[ 0 ], 0.f ), fmaxf( v[ 1 ], 0.f ), fmaxf( v[ 2 ], 0.f ), fmaxf( v[ 3 ], 0.f ) };
}
__device__ __forceinline__ u4 bf4( f4 v )
{
   return u4{ bf( v[ 0 ] ), bf( v[ 1 ] ), bf( v[ 2 ] ), bf( v[ 3 ] ) };
}
// v where the activation m is positive
__device__ __forceinline__ f4 masked4( u4 m, f4 v )
{
#pragma unroll
   for( int i = 0; i < 4; i++ )
      v[ i ] = fb( m[ i ] ) > 0.f ? v[ i ] : 0.f;
   return v;
}

template< int NT, int EPI, int kTiles >
__global__ void __launch_bounds__( 256 ) gemm64( int64_t R, Term t0, Term t1, Term t2, EpiArgs e )
{
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   const int lr = lane & 15, lq = lane >> 4;
   const Term ts[ 3 ] = { t0, t1, t2 };
   bf8 B[ NT ][ 4 ][ 2 ];
#pragma unroll
   for( int t = 0; t < NT; t++ )
#pragma unroll
      for( int nb = 0; nb < 4; nb++ )
#pragma unroll
         for( int kb = 0; kb < 2; kb++ )
            B[ t ][ nb ][ kb ] = *(const bf8*) ( ts[ t ].Bn + ( nb * 16 + lr ) * kH + kb * 32 + lq * 8 );
   const int64_t base = ( (int64_t) blockIdx.x * 4 + w ) * ( 16 * kTiles );
#pragma unroll
   for( int tile = 0; tile < kTiles; tile++ ) {
      const int64_t r = base + tile * 16 + lr;
      if( base + tile * 16 >= R )  // (uniform)
         return;
      const int64_t rc = r < R ? r : R - 1;  // a last tile's rows past R: read again, not stored
      f4 acc[ 4 ];
#pragma unroll
      for( int nb = 0; nb < 4; nb++ )
         acc[ nb ] = f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
      for( int t = 0; t < NT; t++ )
#pragma unroll
         for( int kb = 0; kb < 2; kb++ ) {
            const bf8 x = *(const bf8*) ( ts[ t ].X + rc * kH + kb * 32 + lq * 8 );
#pragma unroll
            for( int nb = 0; nb < 4; nb++ )
               acc[ nb ] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( B[ t ][ nb ][ kb ], x, acc[ nb ], 0, 0, 0 );
         }
      int32_t j = 0, i = 0;
      float d = 1.f;
      if( EPI == EPI_EDGE )
         j = e.col[ rc ];  // -1: a padding slot, no edge
      if( EPI == EPI_EDGE || EPI == EPI_DEDGE )
         i = e.row[ rc ];
      if( EPI == EPI_DMEAN )
         d = (float) e.deg[ rc ];
#pragma unroll
      for( int nb = 0; nb < 4; nb++ ) {
         const int c = nb * 16 + lq * 4;
         f4 v = acc[ nb ];
         if( EPI == EPI_EDGE ) {
            const f4 p = j >= 0 ? *(const f4*) ( e.P + (int64_t) j * kH + c ) : f4{ 0.f, 0.f, 0.f, 0.f };
            v = v + p + *(const f4*) ( e.Q + (int64_t) i * kH + c ) + *(const f4*) ( e.bias + c );
         }
         else if( EPI == EPI_NODE )
            v = v + *(const f4*) ( e.bias + c );
         else if( EPI == EPI_DMEAN )
            v = f4{ v[ 0 ] / d, v[ 1 ] / d, v[ 2 ] / d, v[ 3 ] / d };
         else if( EPI == EPI_DEDGE )
            v = v + *(const f4*) ( e.P + (int64_t) i * kH + c );
         if( EPI == EPI_EDGE || EPI == EPI_NODE )
            v = relu4( v );
         if( EPI == EPI_DNODE || EPI == EPI_DEDGE )
            v = masked4( *(const u4*) ( e.mask + rc * kH + c ), v );
         if( r < R ) {
            if( EPI == EPI_STORE || EPI == EPI_DMEAN )
               *(f4*) ( e.yf + r * kH + c ) = v;
            else
               *(u4*) ( e.yb + r * kH + c ) = bf4( v );
         }
      }
   }
}

// dW[64 x 64] = X^T dY over R rows and the column sums of dY.  A workgroup takes
// tiles of kWRows rows in turn, sums in registers and leaves one partial: the
// rows are the k of the products, so a tile goes to LDS transposed (two rows'
// values packed per 32-bit write) and the fragments are 16-byte LDS reads.  The
// column sums are a product with ones.  The next tile's loads are in flight
// while a tile is multiplied.  326 K rows 26 us (84 MB) against 35 us, with 512
// partials instead of 1,276.
constexpr int kWStride = kWRows + 8;  // (16-byte reads of 16 features on different banks)
constexpr int kPart = kH * kH + kH;   // a partial: dW, then the column sums
constexpr int kWBlocks = 512;         // partials at most (two workgroups per CU)

__global__ void __launch_bounds__( 256 ) wgrad64( int64_t R, const uint16_t* __restrict__ X,
                                                  const uint16_t* __restrict__ dY, float* __restrict__ part )
{
   typedef uint16_t u8v __attribute__( ( ext_vector_type( 8 ) ) );
   __shared__ __align__( 16 ) uint16_t sx[ kH * kWStride ], sy[ kH * kWStride ];
   // (w known to be uniform: a matrix instruction does not look at the exec mask)
   const int lane = threadIdx.x & 63, w = wave_uniform( (int32_t) ( threadIdx.x >> 6 ) );
   const int lr = lane & 15, lq = lane >> 4;
   const int64_t tiles = ( R + kWRows - 1 ) / kWRows;
   const int fg = threadIdx.x & 7, rp = threadIdx.x >> 3;  // 8 features of row pairs rp + 32 u
   u8v x0[ 4 ], x1[ 4 ], y0[ 4 ], y1[ 4 ];
   auto fetch = [ & ]( int64_t tile ) {
#pragma unroll
      for( int u = 0; u < 4; u++ ) {
         const int64_t r = tile * kWRows + 2 * ( rp + 32 * u );
         const int64_t a = r < R ? r : R - 1, b = r + 1 < R ? r + 1 : R - 1;
         x0[ u ] = *(const u8v*) ( X + a * kH + fg * 8 );
         x1[ u ] = *(const u8v*) ( X + b * kH + fg * 8 );
         y0[ u ] = *(const u8v*) ( dY + a * kH + fg * 8 );
         y1[ u ] = *(const u8v*) ( dY + b * kH + fg * 8 );
         if( r >= R )
            x0[ u ] = y0[ u ] = u8v{};
         if( r + 1 >= R )
            x1[ u ] = y1[ u ] = u8v{};
      }
   };
   f4 acc[ 4 ], sums = f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
   for( int nb = 0; nb < 4; nb++ )
      acc[ nb ] = f4{ 0.f, 0.f, 0.f, 0.f };
   const bf8 ones = { (__bf16) 1.f, (__bf16) 1.f, (__bf16) 1.f, (__bf16) 1.f,
                      (__bf16) 1.f, (__bf16) 1.f, (__bf16) 1.f, (__bf16) 1.f };
   fetch( blockIdx.x );
   for( int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x ) {
      __syncthreads();  // (the tile before is read)
#pragma unroll
      for( int u = 0; u < 4; u++ )
#pragma unroll
         for( int f = 0; f < 8; f++ ) {
            const int at = ( fg * 8 + f ) * kWStride + 2 * ( rp + 32 * u );
            *(uint32_t*) ( sx + at ) = (uint32_t) x0[ u ][ f ] | (uint32_t) x1[ u ][ f ] << 16;
            *(uint32_t*) ( sy + at ) = (uint32_t) y0[ u ][ f ] | (uint32_t) y1[ u ][ f ] << 16;
         }
      __syncthreads();
      if( tile + gridDim.x < tiles )
         fetch( tile + gridDim.x );
#pragma unroll
      for( int ks = 0; ks < kWRows / 32; ks++ ) {
         const bf8 a = *(const bf8*) ( sx + ( w * 16 + lr ) * kWStride + ks * 32 + lq * 8 );
#pragma unroll
         for( int nb = 0; nb < 4; nb++ ) {
            const bf8 b = *(const bf8*) ( sy + ( nb * 16 + lr ) * kWStride + ks * 32 + lq * 8 );
            acc[ nb ] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( a, b, acc[ nb ], 0, 0, 0 );
            if( nb == w )
               sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16( ones, b, sums, 0, 0, 0 );
         }
      }
   }
   float* out = part + (int64_t) blockIdx.x * kPart;
#pragma unroll
   for( int nb = 0; nb < 4; nb++ )
#pragma unroll
      for( int i = 0; i < 4; i++ )
         out[ ( w * 16 + lq * 4 + i ) * kH + nb * 16 + lr ] = acc[ nb ][ i ];
   if( lq == 0 )
      out[ kH * kH + w * 16 + lr ] = sums[ 0 ];
}

// out[e] (e < split) and out2[e - split] = the sum over nblk partials of
// part[b * width + e]: 16 waves take consecutive shares of the partials, then
// their sums in order -- a fixed order.  out2 NULL: those columns are not wanted.
__global__ void __launch_bounds__( 1024 ) reduce_parts( const float* __restrict__ part, int64_t nblk, int width, int split,
                                                        float* __restrict__ out, float* __restrict__ out2 )
{
   __shared__ float sm[ 16 ][ 64 ];
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   const int e = blockIdx.x * 64 + lane;
   const int64_t share = ( nblk + 15 ) / 16, b0 = min( nblk, w * share ), b1 = min( nblk, b0 + share );
   float s = 0.f;
   if( e < width )
      for( int64_t b = b0; b < b1; b += 8 ) {
         float v[ 8 ];
#pragma unroll
         for( int u = 0; u < 8; u++ )
            v[ u ] = b + u < b1 ? part[ ( b + u ) * width + e ] : 0.f;
#pragma unroll
         for( int u = 0; u < 8; u++ )
            s += v[ u ];
      }
   sm[ w ][ lane ] = s;
   __syncthreads();
   if( w != 0 || e >= width )
      return;
   float t = 0.f;
#pragma unroll
   for( int i = 0; i < 16; i++ )
      t += sm[ i ][ lane ];
   if( e < split )
      out[ e ] = t;
   else if( out2 )
      out2[ e - split ] = t;
}

// ------------------------------------------------------------ graph and IO
struct Graph
{
   int64_t n = 0, E = 0;
   DeviceArray< int32_t > erow, cperm, cptr, deg, ids;
   DeviceArray< uint32_t > keys, skeys;
   DeviceArray< char > sort_tmp;
   DeviceArray< double > diag;
   DeviceArray< float > xe, xn;
   DeviceArray< uint8_t > isd;
};

__global__ void g_rows( int64_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ cols,
                        const double* __restrict__ vals, int32_t* __restrict__ erow, int32_t* __restrict__ deg,
                        double* __restrict__ diag, uint8_t* __restrict__ isd )
{
   const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( i >= n )
      return;
   double d = 0.0;
   for( int32_t e = off[ i ]; e < off[ i + 1 ]; e++ ) {
      erow[ e ] = (int32_t) i;
      const bool dg = cols[ e ] == i;
      isd[ e ] = dg ? 1 : 0;
      if( dg )
         d = vals[ e ];
   }
   deg[ i ] = off[ i + 1 ] - off[ i ];
   diag[ i ] = d;
}

__global__ void g_features( int64_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ cols,
                            const double* __restrict__ vals, const double* __restrict__ diag,
                            float* __restrict__ xe, float* __restrict__ xn )
{
   const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( i >= n )
      return;
   const double di = diag[ i ];
   double oabs = 0.0, rs = 0.0;
   for( int32_t e = off[ i ]; e < off[ i + 1 ]; e++ ) {
      const int32_t j = cols[ e ];
      const double a = vals[ e ];
      if( j < 0 ) {  // padding slot: no edge
         for( int k = 0; k < 4; k++ )
            xe[ (int64_t) e * 4 + k ] = 0.f;
         continue;
      }
      xe[ (int64_t) e * 4 + 0 ] = (float) ( a / di );
      xe[ (int64_t) e * 4 + 1 ] = (float) ( a / diag[ j ] );
      xe[ (int64_t) e * 4 + 2 ] = j == i ? 1.f : 0.f;
      xe[ (int64_t) e * 4 + 3 ] = (float) ( fabs( a ) / di );
      if( j != i )
         oabs += fabs( a );
      rs += a;
   }
   xn[ i * 4 + 0 ] = (float) ( oabs / di );
   xn[ i * 4 + 1 ] = (float) ( rs / di );
   xn[ i * 4 + 2 ] = (float) ( off[ i + 1 ] - off[ i ] ) / 5.f;
   xn[ i * 4 + 3 ] = 1.f;
}

__global__ void g_colptr( int64_t E, int64_t n, const uint32_t* __restrict__ skeys, int32_t* __restrict__ cptr )
{
   const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( p > E )
      return;
   const int32_t prev = p == 0 ? -1 : (int32_t) skeys[ p - 1 ] - 1;
   const int32_t cur = p == E ? (int32_t) n : (int32_t) skeys[ p ] - 1;
   for( int32_t c = prev + 1; c <= cur; c++ )
      cptr[ c ] = (int32_t) p;
}

// sort keys column + 1 (0: a padding slot), so that only the bits of n are sorted
__global__ void iota_k( int64_t E, const int32_t* __restrict__ cols, uint32_t* __restrict__ keys,
                        int32_t* __restrict__ v )
{
   const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( p < E ) {
      keys[ p ] = (uint32_t) ( cols[ p ] + 1 );
      v[ p ] = (int32_t) p;
   }
}

// ------------------------------------------------------------ forward parts
// relu(x W + b) for K = 4 inputs (FP32), BF16 out; 4 columns per thread
__global__ void __launch_bounds__( 256 ) encode_k( int64_t R, const float* __restrict__ x, const float* __restrict__ W,
                                                   const float* __restrict__ b, uint16_t* __restrict__ y )
{
   const int64_t q = (int64_t) blockIdx.x * 256 + threadIdx.x, r = q / 16;
   const int c = (int) ( q % 16 ) * 4;
   if( r >= R )
      return;
   const f4 xr = *(const f4*) ( x + r * 4 );
   f4 v = *(const f4*) ( b + c );
#pragma unroll
   for( int k = 0; k < 4; k++ )
      v += xr[ k ] * *(const f4*) ( W + k * kH + c );
   *(u4*) ( y + r * kH + c ) = bf4( relu4( v ) );
}

__device__ __forceinline__ f4 fb4( u4 v )
{
   return f4{ fb( v[ 0 ] ), fb( v[ 1 ] ), fb( v[ 2 ] ), fb( v[ 3 ] ) };
}

// G = BF16 of the mean of the row's edge features; 4 columns per thread
__global__ void __launch_bounds__( 256 ) mean_k( int64_t n, const int32_t* __restrict__ off, const uint16_t* __restrict__ E,
                                                 uint16_t* __restrict__ G )
{
   const int64_t q = (int64_t) blockIdx.x * 256 + threadIdx.x, i = q / 16;
   const int c = (int) ( q % 16 ) * 4;
   if( i >= n )
      return;
   f4 s = f4{ 0.f, 0.f, 0.f, 0.f };
   const int32_t e0 = off[ i ], d = off[ i + 1 ] - e0;
   for( int32_t e = 0; e < d; e++ )
      s += fb4( *(const u4*) ( E + (int64_t) ( e0 + e ) * kH + c ) );
   if( d > 0 )
      s = f4{ s[ 0 ] / (float) d, s[ 1 ] / (float) d, s[ 2 ] / (float) d, s[ 3 ] / (float) d };
   *(u4*) ( G + i * kH + c ) = bf4( s );
}

// o_e = E_e . wo + bo (FP32), M_e = (delta + o) / a_ii (FP64); 16 lanes per edge
__global__ void __launch_bounds__( 256 ) decode_k( int64_t E, const uint16_t* __restrict__ X, const float* __restrict__ wo,
                                                   const float* __restrict__ bo, const int32_t* __restrict__ erow,
                                                   const int32_t* __restrict__ cols, const uint8_t* __restrict__ isd,
                                                   const double* __restrict__ diag, double* __restrict__ M )
{
   const int64_t q = (int64_t) blockIdx.x * 256 + threadIdx.x, e = q / 16;
   const int c = (int) ( q % 16 ) * 4;
   if( e >= E )
      return;  // (uniform over the 16 lanes)
   const f4 v = fb4( *(const u4*) ( X + e * kH + c ) ), w = *(const f4*) ( wo + c );
   const float o = group_sum< 16 >( v[ 0 ] * w[ 0 ] + v[ 1 ] * w[ 1 ] + v[ 2 ] * w[ 2 ] + v[ 3 ] * w[ 3 ] ) + bo[ 0 ];
   if( c == 0 )
      M[ e ] = cols[ e ] < 0 ? 0.0 : ( (double) isd[ e ] + (double) o ) / diag[ erow[ e ] ];
}

// ------------------------------------------------------------ probe loss
__device__ __forceinline__ uint64_t mix64( uint64_t z )
{
   z += 0x9e3779b97f4a7c15ull;
   z = ( z ^ ( z >> 30 ) ) * 0xbf58476d1ce4e5b9ull;
   z = ( z ^ ( z >> 27 ) ) * 0x94d049bb133111ebull;
   return z ^ ( z >> 31 );
}
__global__ void rademacher_k( int64_t cnt, uint64_t seed, double* __restrict__ Z )
{
   const int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( q < cnt )
      Z[ q ] = ( mix64( seed * 0x2545f4914f6cdd1dull + (uint64_t) q ) >> 63 ) ? 1.0 : -1.0;
}

// y = V x over the CSR pattern (one thread per row; blockIdx.y: the probe)
__global__ void csr_mv( int64_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ cols,
                        const double* __restrict__ V, const double* __restrict__ x, double* __restrict__ y )
{
   const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   x += blockIdx.y * n;
   y += blockIdx.y * n;
   if( i >= n )
      return;
   double s = 0.0;
   for( int32_t e = off[ i ]; e < off[ i + 1 ]; e++ )
      if( cols[ e ] >= 0 )
         s += V[ e ] * x[ cols[ e ] ];
   y[ i ] = s;
}

// r = z - w (in place over w), partial sums of r.r per block
__global__ void __launch_bounds__( 256 ) resid_k( int64_t n, const double* __restrict__ z, double* __restrict__ w,
                                                  double* __restrict__ part )
{
   __shared__ double sm[ 4 ];
   const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
   z += blockIdx.y * n;
   w += blockIdx.y * n;
   part += blockIdx.y * gridDim.x;
   double v = 0.0;
   if( i < n ) {
      const double r = z[ i ] - w[ i ];
      w[ i ] = r;
      v = r * r;
   }
   v = block_sum< 256 >( v, sm );
   if( threadIdx.x == 0 )
      part[ blockIdx.x ] = v;
}

__global__ void sum_k( const double* __restrict__ part, int64_t np, double scale, double* __restrict__ out )
{
   __shared__ double sm[ 4 ];
   double v = 0.0;
   for( int64_t i = threadIdx.x; i < np; i += 256 )
      v += part[ i ];
   v = block_sum< 256 >( v, sm );
   if( threadIdx.x == 0 )
      out[ 0 ] = v * scale;
}

// dL/dM_e = -2 / (K n) sum_k r_k[row] y_k[col]
__global__ void dM_k( int64_t E, int64_t n, int K, const int32_t* __restrict__ erow, const int32_t* __restrict__ cols,
                      const double* __restrict__ Rk, const double* __restrict__ Yk, double* __restrict__ dM )
{
   const int64_t e = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( e >= E )
      return;
   double s = 0.0;
   if( cols[ e ] >= 0 )
      for( int k = 0; k < K; k++ )
         s += Rk[ (int64_t) k * n + erow[ e ] ] * Yk[ (int64_t) k * n + cols[ e ] ];
   dM[ e ] = -2.0 * s / ( (double) K * (double) n );
}

// ------------------------------------------------------------ backward parts
// do_e = dM_e / a_ii;  dS = BF16( do x wo * [E > 0] ) of the last layer (its node
// features reach nothing);  per wave partial sums of do_e E_e and do_e
__global__ void __launch_bounds__( 256 ) dec_bwd_k( int64_t E, const double* __restrict__ dM,
                                                    const int32_t* __restrict__ erow, const double* __restrict__ diag,
                                                    const uint16_t* __restrict__ X, const float* __restrict__ wo,
                                                    uint16_t* __restrict__ dS, float* __restrict__ part )
{
   const int lane = threadIdx.x & 63, c = ( lane & 15 ) * 4, sub = lane >> 4;  // 4 columns of every 4th row
   const f4 wc = *(const f4*) ( wo + c );
   f4 s = f4{ 0.f, 0.f, 0.f, 0.f };
   float so = 0.f;
   constexpr int kAt = 4;  // rows loaded together
   const int64_t wave = (int64_t) blockIdx.x * 4 + ( threadIdx.x >> 6 ), waves = (int64_t) gridDim.x * 4;
   for( int64_t r0 = wave * ( 4 * kAt ); r0 < E; r0 += waves * ( 4 * kAt ) ) {
      float d[ kAt ];
      u4 v[ kAt ];
#pragma unroll
      for( int u = 0; u < kAt; u++ ) {
         const int64_t r = r0 + u * 4 + sub, q = r < E ? r : E - 1;
         d[ u ] = r < E ? (float) ( dM[ q ] / diag[ erow[ q ] ] ) : 0.f;
         v[ u ] = *(const u4*) ( X + q * kH + c );
      }
#pragma unroll
      for( int u = 0; u < kAt; u++ ) {
         const int64_t r = r0 + u * 4 + sub;
         s += d[ u ] * fb4( v[ u ] );
         so += d[ u ];
         if( r < E )
            *(u4*) ( dS + r * kH + c ) = bf4( masked4( v[ u ], d[ u ] * wc ) );
      }
   }
   float* out = part + wave * ( kH + 1 );
#pragma unroll
   for( int i = 0; i < 4; i++ ) {
      float t = s[ i ];
      t += __shfl_xor( t, 16, 64 );
      t += __shfl_xor( t, 32, 64 );
      if( sub == 0 )
         out[ c + i ] = t;
   }
   so += __shfl_xor( so, 16, 64 );
   so += __shfl_xor( so, 32, 64 );
   if( lane == 0 )
      out[ kH ] = so;
}

// dQ_i = BF16( sum over row i of dS ),  dP_j = BF16( sum over column j of dS ); 4 columns per thread
__global__ void __launch_bounds__( 256 ) scatter_k( int64_t n, const int32_t* __restrict__ off,
                                                    const int32_t* __restrict__ cptr, const int32_t* __restrict__ cperm,
                                                    const uint16_t* __restrict__ dS, uint16_t* __restrict__ dP,
                                                    uint16_t* __restrict__ dQ )
{
   const int64_t q = (int64_t) blockIdx.x * 256 + threadIdx.x, i = q / 16;
   const int c = (int) ( q % 16 ) * 4;
   if( i >= n )
      return;
   f4 sq = f4{ 0.f, 0.f, 0.f, 0.f }, sp = sq;
   for( int32_t e = off[ i ]; e < off[ i + 1 ]; e++ )
      sq += fb4( *(const u4*) ( dS + (int64_t) e * kH + c ) );
   for( int32_t p = cptr[ i ]; p < cptr[ i + 1 ]; p++ )
      sp += fb4( *(const u4*) ( dS + (int64_t) cperm[ p ] * kH + c ) );
   *(u4*) ( dQ + i * kH + c ) = bf4( sq );
   *(u4*) ( dP + i * kH + c ) = bf4( sp );
}

// encoder gradients: per wave partials of x^T (dX * [Y > 0]) (4 x 64) and of the
// column sums (64)
__global__ void __launch_bounds__( 256 ) enc_bwd_k( int64_t R, const float* __restrict__ x,
                                                    const float* __restrict__ dX, const uint16_t* __restrict__ Y,
                                                    float* __restrict__ part )
{
   const int lane = threadIdx.x & 63, c = ( lane & 15 ) * 4, sub = lane >> 4;  // 4 columns of every 4th row
   f4 s[ 5 ];  // by input, then the column sums
#pragma unroll
   for( int k = 0; k < 5; k++ )
      s[ k ] = f4{ 0.f, 0.f, 0.f, 0.f };
   constexpr int kAt = 4;  // rows loaded together
   const int64_t wave = (int64_t) blockIdx.x * 4 + ( threadIdx.x >> 6 ), waves = (int64_t) gridDim.x * 4;
   for( int64_t r0 = wave * ( 4 * kAt ); r0 < R; r0 += waves * ( 4 * kAt ) ) {
      f4 xr[ kAt ], g[ kAt ];
      u4 y[ kAt ];
#pragma unroll
      for( int u = 0; u < kAt; u++ ) {
         const int64_t r = r0 + u * 4 + sub, q = r < R ? r : R - 1;
         xr[ u ] = *(const f4*) ( x + q * 4 );
         g[ u ] = *(const f4*) ( dX + q * kH + c );
         y[ u ] = *(const u4*) ( Y + q * kH + c );
      }
#pragma unroll
      for( int u = 0; u < kAt; u++ )
         if( r0 + u * 4 + sub < R ) {
            const f4 m = masked4( y[ u ], g[ u ] );
#pragma unroll
            for( int k = 0; k < 4; k++ )
               s[ k ] += xr[ u ][ k ] * m;
            s[ 4 ] += m;
         }
   }
   float* out = part + wave * ( 5 * kH );
#pragma unroll
   for( int k = 0; k < 5; k++ )
#pragma unroll
      for( int i = 0; i < 4; i++ ) {
         float t = s[ k ][ i ];
         t += __shfl_xor( t, 16, 64 );
         t += __shfl_xor( t, 32, 64 );
         if( sub == 0 )
            out[ k * kH + c + i ] = t;
      }
}

// ------------------------------------------------------------ parameters
__global__ void refresh_bf_k( const float* __restrict__ params, uint16_t* __restrict__ W, uint16_t* __restrict__ WT )
{
   const int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( q >= (int64_t) kL * kMats * kH * kH )
      return;
   const int64_t mat = q / ( kH * kH );
   const int l = (int) ( mat / kMats ), m = (int) ( mat % kMats );
   const int k = (int) ( ( q / kH ) % kH ), nn = (int) ( q % kH );
   const uint16_t v = bf( params[ oW( l, m ) + k * kH + nn ] );
   W[ mat * kH * kH + k * kH + nn ] = v;   // [k][n]: Bn for X W^T
   WT[ mat * kH * kH + nn * kH + k ] = v;  // [n][k]: Bn for X W
}

__global__ void adam_k( int64_t cnt, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                        float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2 )
{
   const int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
   if( q >= cnt )
      return;
   const float gq = g[ q ];
   const float mq = b1 * m[ q ] + ( 1.f - b1 ) * gq;
   const float vq = b2 * v[ q ] + ( 1.f - b2 ) * gq * gq;
   m[ q ] = mq;
   v[ q ] = vq;
   p[ q ] -= lr * ( mq / c1 ) / ( sqrtf( vq / c2 ) + eps );
}

inline dim3 g1( int64_t cnt, int b = 256 )
{
   return dim3( (unsigned) std::max< int64_t >( 1, ceil_div( cnt, b ) ) );
}

}  // namespace
}  // namespace tnlmi

using namespace tnlmi;

namespace tnlmi {
namespace {

struct Acts
{
   DeviceArray< uint16_t > E[ kL + 1 ], H[ kL + 1 ], G[ kL + 1 ];
   DeviceArray< float > P, Q;
};

// What a call works in: the graph, the activations and the backward pass's
// arrays.  A network keeps one, as large as the largest matrix it has seen,
// and gives it back when it is destroyed: 45 allocations and frees of up to
// 84 MB took 7 of the 10 ms of a training step on a 256^2 grid.
struct Workspace
{
   Graph g;
   Acts a;
   DeviceArray< double > M, dM, Y, Rk, lpart, Z;
   DeviceArray< float > dE, dH, dG, part;
   DeviceArray< uint16_t > dS, dSn, dT, dTn, dP, dQ;
   DeviceArray< double > lout;
};

}  // namespace
}  // namespace tnlmi

struct tnlmi_spai
{
   DeviceArray< float > params, grads, m, v;
   DeviceArray< uint16_t > W, WT;  // BF16 copies of the 15 64 x 64 matrices
   int64_t step = 0;
   mutable std::mutex busy;  // held by the call that works in `work`
   mutable Workspace work;
};

namespace tnlmi {
namespace {

// A call's workspace: the network's, or one of its own while another thread's
// call works in that.  The stream is waited for before the workspace passes on.
struct Working
{
   std::unique_lock< std::mutex > lock;
   std::unique_ptr< Workspace > own;
   Workspace* w;
   hipStream_t s;
   Working( const tnlmi_spai& S, hipStream_t stream ) : lock( S.busy, std::try_to_lock ), s( stream )
   {
      if( ! lock.owns_lock() )
         own = std::make_unique< Workspace >();
      w = own ? own.get() : &S.work;
   }
   ~Working() { (void) hipStreamSynchronize( s ); }
};

const uint16_t* Wn( const tnlmi_spai& S, int l, int m )  // Bn for X W^T
{
   return S.W.ptr + (int64_t) ( l * kMats + m ) * kH * kH;
}
const uint16_t* WTn( const tnlmi_spai& S, int l, int m )  // Bn for X W
{
   return S.WT.ptr + (int64_t) ( l * kMats + m ) * kH * kH;
}

void refresh( tnlmi_spai& S, hipStream_t s )
{
   hipLaunchKernelGGL( refresh_bf_k, g1( (int64_t) kL * kMats * kH * kH ), dim3( 256 ), 0, s, S.params.ptr, S.W.ptr,
                       S.WT.ptr );
}

void check_csr( const tnlmi_matrix* A )
{
   if( ! A || ! A->segments )
      fail( TNLMI_INVALID_ARGUMENT, "spai: NULL matrix" );
   if( A->segments->format != TNLMI_CSR || A->value_type != TNLMI_F64 )
      fail( TNLMI_INVALID_ARGUMENT, "spai: the matrix must be CSR with FP64 values" );
   if( A->matrix_type == TNLMI_SYMMETRIC )
      fail( TNLMI_NOT_IMPLEMENTED, "spai: a general matrix is needed (the network reads both triangles' entries)" );
   if( A->rows != A->columns || A->rows <= 0 )
      fail( TNLMI_INVALID_ARGUMENT, "spai: the matrix must be square and not empty" );
}

void build_graph( Graph& g, const tnlmi_matrix& A, hipStream_t s )
{
   g.n = A.rows;
   g.E = A.segments->elements;
   const int32_t* off = A.segments->offsets.ptr;
   const int32_t* cols = A.column_indexes;
   const double* vals = (const double*) A.values;
   g.erow.reserve( g.E );
   g.deg.reserve( g.n );
   g.diag.reserve( g.n );
   g.isd.reserve( g.E );
   g.xe.reserve( g.E * 4 );
   g.xn.reserve( g.n * 4 );
   hipLaunchKernelGGL( g_rows, g1( g.n ), dim3( 256 ), 0, s, g.n, off, cols, vals, g.erow.ptr, g.deg.ptr,
                       g.diag.ptr, g.isd.ptr );
   hipLaunchKernelGGL( g_features, g1( g.n ), dim3( 256 ), 0, s, g.n, off, cols, vals, g.diag.ptr, g.xe.ptr,
                       g.xn.ptr );
   // edges grouped by column (stable radix sort by column): the transposed scatter
   g.ids.reserve( g.E );
   g.keys.reserve( g.E );
   g.skeys.reserve( g.E );
   g.cperm.reserve( g.E );
   g.cptr.reserve( g.n + 1 );
   int bits = 1;
   while( ( g.n >> bits ) != 0 )
      bits++;
   hipLaunchKernelGGL( iota_k, g1( g.E ), dim3( 256 ), 0, s, g.E, cols, g.keys.ptr, g.ids.ptr );
   size_t bytes = 0;
   TNLMI_HIP( hipcub::DeviceRadixSort::SortPairs( nullptr, bytes, g.keys.ptr, g.skeys.ptr, g.ids.ptr, g.cperm.ptr,
                                                  (int) g.E, 0, bits, s ) );
   g.sort_tmp.reserve( (int64_t) bytes + 1 );
   TNLMI_HIP( hipcub::DeviceRadixSort::SortPairs( g.sort_tmp.ptr, bytes, g.keys.ptr, g.skeys.ptr, g.ids.ptr,
                                                  g.cperm.ptr, (int) g.E, 0, bits, s ) );
   hipLaunchKernelGGL( g_colptr, g1( g.E + 1 ), dim3( 256 ), 0, s, g.E, g.n, g.skeys.ptr, g.cptr.ptr );
   TNLMI_HIP( hipGetLastError() );
}

template< int NT, int EPI >
void gemm( int64_t R, Term t0, Term t1, Term t2, const EpiArgs& e, hipStream_t s )
{
   // (4 tiles per wave read the weights once per 64 rows; with fewer rows more waves matter more)
   if( R >= 131072 )
      hipLaunchKernelGGL( ( gemm64< NT, EPI, 4 > ), g1( R, 256 ), dim3( 256 ), 0, s, R, t0, t1, t2, e );
   else
      hipLaunchKernelGGL( ( gemm64< NT, EPI, 1 > ), g1( R, 64 ), dim3( 256 ), 0, s, R, t0, t1, t2, e );
}

// forward pass; keep = every layer's activations (training), else only the last
void forward( const tnlmi_spai& S, const Graph& g, const int32_t* off, const int32_t* cols, Acts& a, bool keep,
              double* M, hipStream_t s )
{
   const int64_t n = g.n, E = g.E;
   const float* p = S.params.ptr;
   const int nE = keep ? kL + 1 : 2, nH = keep ? kL + 1 : 2;
   for( int i = 0; i < nE; i++ )
      a.E[ i ].reserve( E * kH );
   for( int i = 0; i < nH; i++ ) {
      a.H[ i ].reserve( n * kH );
      a.G[ i ].reserve( n * kH );
   }
   a.P.reserve( n * kH );
   a.Q.reserve( n * kH );
   hipLaunchKernelGGL( encode_k, g1( E * 16 ), dim3( 256 ), 0, s, E, g.xe.ptr, p + oAe, p + oae, a.E[ 0 ].ptr );
   hipLaunchKernelGGL( encode_k, g1( n * 16 ), dim3( 256 ), 0, s, n, g.xn.ptr, p + oAn, p + oan, a.H[ 0 ].ptr );
   const Term none{ nullptr, nullptr };
   for( int l = 0; l < kL; l++ ) {
      const int ci = keep ? l : ( l & 1 ), ni = keep ? l + 1 : ( ( l + 1 ) & 1 );
      EpiArgs ep{};
      ep.yf = a.P.ptr;
      gemm< 1, EPI_STORE >( n, Term{ a.H[ ci ].ptr, WTn( S, l, mWu ) }, none, none, ep, s );
      ep.yf = a.Q.ptr;
      gemm< 1, EPI_STORE >( n, Term{ a.H[ ci ].ptr, WTn( S, l, mWv ) }, none, none, ep, s );
      EpiArgs ee{};
      ee.yb = a.E[ ni ].ptr;
      ee.bias = p + obe( l );
      ee.P = a.P.ptr;
      ee.Q = a.Q.ptr;
      ee.col = cols;
      ee.row = g.erow.ptr;
      gemm< 1, EPI_EDGE >( E, Term{ a.E[ ci ].ptr, WTn( S, l, mWe ) }, none, none, ee, s );
      if( l == kL - 1 )
         break;  // (the decoder reads the edges alone)
      hipLaunchKernelGGL( mean_k, g1( n * 16 ), dim3( 256 ), 0, s, n, off, a.E[ ni ].ptr, a.G[ ni ].ptr );
      EpiArgs en{};
      en.yb = a.H[ ni ].ptr;
      en.bias = p + obh( l );
      gemm< 2, EPI_NODE >( n, Term{ a.H[ ci ].ptr, WTn( S, l, mWh ) }, Term{ a.G[ ni ].ptr, WTn( S, l, mWg ) }, none,
                           en, s );
   }
   const int last = keep ? kL : ( kL & 1 );
   hipLaunchKernelGGL( decode_k, g1( E * 16 ), dim3( 256 ), 0, s, E, a.E[ last ].ptr, p + owo, p + obo, g.erow.ptr,
                       cols, g.isd.ptr, g.diag.ptr, M );
   TNLMI_HIP( hipGetLastError() );
}

// sums of nblk partials of `width` columns: the first `split` to out, the others to out2
void reduce( const float* part, int64_t nblk, int width, int split, float* out, float* out2, hipStream_t s )
{
   hipLaunchKernelGGL( reduce_parts, dim3( (unsigned) ceil_div( width, 64 ) ), dim3( 1024 ), 0, s, part, nblk, width,
                       split, out, out2 );
}

void wgrad( int64_t R, const uint16_t* X, const uint16_t* dY, float* gW, float* gb, float* part, hipStream_t s )
{
   const int64_t nb = std::min< int64_t >( kWBlocks, ceil_div( R, kWRows ) );
   hipLaunchKernelGGL( wgrad64, dim3( (unsigned) nb ), dim3( 256 ), 0, s, R, X, dY, part );
   reduce( part, nb, kPart, kH * kH, gW, gb, s );
}

// probe loss on the device: returns L (host) and dL/dM per edge in dM
double probe_loss( const tnlmi_matrix& A, Workspace& w, const double* M, const double* Z, int K, double* dM,
                   hipStream_t s )
{
   const Graph& g = w.g;
   const int64_t n = g.n, E = g.E;
   const int32_t* off = A.segments->offsets.ptr;
   const int32_t* cols = A.column_indexes;
   DeviceArray< double >&Y = w.Y, &Rk = w.Rk, &part = w.lpart, &out = w.lout;
   Y.reserve( n * K );
   Rk.reserve( n * K );
   const int64_t nb = ceil_div( n, 256 );
   part.reserve( nb * K );
   out.reserve( 1 );
   const dim3 probes( (unsigned) nb, (unsigned) K );
   hipLaunchKernelGGL( csr_mv, probes, dim3( 256 ), 0, s, n, off, cols, (const double*) A.values, Z, Y.ptr );
   hipLaunchKernelGGL( csr_mv, probes, dim3( 256 ), 0, s, n, off, cols, M, (const double*) Y.ptr, Rk.ptr );
   hipLaunchKernelGGL( resid_k, probes, dim3( 256 ), 0, s, n, Z, Rk.ptr, part.ptr );
   hipLaunchKernelGGL( sum_k, dim3( 1 ), dim3( 256 ), 0, s, part.ptr, nb * K, 1.0 / ( (double) K * (double) n ),
                       out.ptr );
   if( dM )
      hipLaunchKernelGGL( dM_k, g1( E ), dim3( 256 ), 0, s, E, n, K, g.erow.ptr, cols, Rk.ptr, Y.ptr, dM );
   double L = 0;
   TNLMI_HIP( hipMemcpyAsync( &L, out.ptr, sizeof( double ), hipMemcpyDeviceToHost, s ) );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   return L;
}

// gradients of the loss into S.grads
double loss_grad( tnlmi_spai& S, Workspace& w, const tnlmi_matrix& A, const double* Z, int K, double* Mout,
                  hipStream_t s )
{
   Graph& g = w.g;
   build_graph( g, A, s );
   const int64_t n = g.n, E = g.E;
   const int32_t* off = A.segments->offsets.ptr;
   const int32_t* cols = A.column_indexes;
   Acts& a = w.a;
   w.dM.reserve( E );
   if( ! Mout ) {
      w.M.reserve( E );
      Mout = w.M.ptr;
   }
   forward( S, g, off, cols, a, true, Mout, s );
   const double L = probe_loss( A, w, Mout, Z, K, w.dM.ptr, s );
   float* gr = S.grads.ptr;
   const float* p = S.params.ptr;
   DeviceArray< float >&dE = w.dE, &dH = w.dH, &dG = w.dG, &part = w.part;
   DeviceArray< uint16_t >&dS = w.dS, &dSn = w.dSn, &dT = w.dT, &dTn = w.dTn, &dP = w.dP, &dQ = w.dQ;
   dE.reserve( E * kH );
   dH.reserve( n * kH );
   dG.reserve( n * kH );
   for( auto* v : { &dS, &dSn } )
      v->reserve( E * kH );
   for( auto* v : { &dT, &dTn, &dP, &dQ } )
      v->reserve( n * kH );
   constexpr int64_t kSumBlocks = 512;  // workgroups of dec_bwd_k and enc_bwd_k, four partials each
   part.reserve( std::max< int64_t >( (int64_t) kWBlocks * kPart, kSumBlocks * 4 * 5 * kH ) );
   // decoder
   hipLaunchKernelGGL( dec_bwd_k, dim3( (unsigned) kSumBlocks ), dim3( 256 ), 0, s, E, w.dM.ptr, g.erow.ptr, g.diag.ptr,
                       a.E[ kL ].ptr, p + owo, dS.ptr, part.ptr );
   reduce( part.ptr, kSumBlocks * 4, kH + 1, kH + 1, gr + owo, nullptr, s );
   // the last layer's node update reaches nothing: no gradient
   static_assert( mWg == mWh + 1, "Wh and Wg side by side" );
   TNLMI_HIP( hipMemsetAsync( gr + oW( kL - 1, mWh ), 0, sizeof( float ) * 2 * kH * kH, s ) );
   TNLMI_HIP( hipMemsetAsync( gr + obh( kL - 1 ), 0, sizeof( float ) * kH, s ) );
   const Term none{ nullptr, nullptr };
   for( int l = kL - 1; l >= 0; l-- ) {
      const bool top = l == kL - 1;  // dT = 0 there
      // the edge update's weights; its node terms' gradients
      wgrad( E, a.E[ l ].ptr, dS.ptr, gr + oW( l, mWe ), gr + obe( l ), part.ptr, s );
      hipLaunchKernelGGL( scatter_k, g1( n * 16 ), dim3( 256 ), 0, s, n, off, g.cptr.ptr, g.cperm.ptr, dS.ptr, dP.ptr,
                          dQ.ptr );
      wgrad( n, a.H[ l ].ptr, dP.ptr, gr + oW( l, mWu ), nullptr, part.ptr, s );
      wgrad( n, a.H[ l ].ptr, dQ.ptr, gr + oW( l, mWv ), nullptr, part.ptr, s );
      const Term tP{ dP.ptr, Wn( S, l, mWu ) }, tQ{ dQ.ptr, Wn( S, l, mWv ) }, tT{ dT.ptr, Wn( S, l, mWh ) },
         tS{ dS.ptr, Wn( S, l, mWe ) };
      if( l == 0 ) {
         // the encoders' gradients want dH and dE in FP32
         EpiArgs eh{};
         eh.yf = dH.ptr;
         if( top )
            gemm< 2, EPI_STORE >( n, tP, tQ, none, eh, s );
         else
            gemm< 3, EPI_STORE >( n, tT, tP, tQ, eh, s );
         EpiArgs ee{};
         ee.yf = dE.ptr;
         gemm< 1, EPI_STORE >( E, tS, none, none, ee, s );
         break;
      }
      // the node update below: dT = BF16( dH * [H > 0] ), its weights, and what it
      // passes to its row's edges, dG / deg
      EpiArgs eh{};
      eh.yb = dTn.ptr;
      eh.mask = a.H[ l ].ptr;
      if( top )
         gemm< 2, EPI_DNODE >( n, tP, tQ, none, eh, s );
      else
         gemm< 3, EPI_DNODE >( n, tT, tP, tQ, eh, s );
      std::swap( dT, dTn );
      wgrad( n, a.H[ l - 1 ].ptr, dT.ptr, gr + oW( l - 1, mWh ), gr + obh( l - 1 ), part.ptr, s );
      wgrad( n, a.G[ l ].ptr, dT.ptr, gr + oW( l - 1, mWg ), nullptr, part.ptr, s );
      EpiArgs eg{};
      eg.yf = dG.ptr;
      eg.deg = g.deg.ptr;
      gemm< 1, EPI_DMEAN >( n, Term{ dT.ptr, Wn( S, l - 1, mWg ) }, none, none, eg, s );
      // the edge update below: dS = BF16( (dE + dG[row] / deg) * [E > 0] )
      EpiArgs ed{};
      ed.yb = dSn.ptr;
      ed.P = dG.ptr;
      ed.row = g.erow.ptr;
      ed.mask = a.E[ l ].ptr;
      gemm< 1, EPI_DEDGE >( E, tS, none, none, ed, s );
      std::swap( dS, dSn );
   }
   // encoder
   hipLaunchKernelGGL( enc_bwd_k, dim3( (unsigned) kSumBlocks ), dim3( 256 ), 0, s, E, g.xe.ptr, dE.ptr, a.E[ 0 ].ptr,
                       part.ptr );
   reduce( part.ptr, kSumBlocks * 4, 5 * kH, 5 * kH, gr + oAe, nullptr, s );
   hipLaunchKernelGGL( enc_bwd_k, dim3( (unsigned) kSumBlocks ), dim3( 256 ), 0, s, n, g.xn.ptr, dH.ptr, a.H[ 0 ].ptr,
                       part.ptr );
   reduce( part.ptr, kSumBlocks * 4, 5 * kH, 5 * kH, gr + oAn, nullptr, s );
   TNLMI_HIP( hipGetLastError() );
   TNLMI_HIP( hipStreamSynchronize( s ) );
   return L;
}

}  // namespace
}  // namespace tnlmi

extern "C" {

int64_t tnlmi_spai_parameter_count( void )
{
   return kParams;
}

tnlmi_status tnlmi_spai_create( const float* h_params, tnlmi_spai** out )
{
   return guarded( [ & ] {
      if( ! out || ! h_params )
         fail( TNLMI_INVALID_ARGUMENT, "spai_create: NULL argument" );
      *out = nullptr;
      auto* S = new tnlmi_spai;
      try {
         for( auto* a : { &S->params, &S->grads, &S->m, &S->v } )
            a->allocate( kParams );
         S->W.allocate( (int64_t) kL * kMats * kH * kH );
         S->WT.allocate( (int64_t) kL * kMats * kH * kH );
         TNLMI_HIP( hipMemcpy( S->params.ptr, h_params, sizeof( float ) * kParams, hipMemcpyHostToDevice ) );
         TNLMI_HIP( hipMemset( S->grads.ptr, 0, sizeof( float ) * kParams ) );
         TNLMI_HIP( hipMemset( S->m.ptr, 0, sizeof( float ) * kParams ) );
         TNLMI_HIP( hipMemset( S->v.ptr, 0, sizeof( float ) * kParams ) );
         refresh( *S, nullptr );
         TNLMI_HIP( hipDeviceSynchronize() );
      }
      catch( ... ) {
         delete S;
         throw;
      }
      *out = S;
   } );
}

void tnlmi_spai_destroy( tnlmi_spai* S )
{
   delete S;
}

tnlmi_status tnlmi_spai_get_parameters( const tnlmi_spai* S, float* h_params, float* h_grads )
{
   return guarded( [ & ] {
      if( ! S )
         fail( TNLMI_INVALID_ARGUMENT, "spai: NULL handle" );
      if( h_params )
         TNLMI_HIP( hipMemcpy( h_params, S->params.ptr, sizeof( float ) * kParams, hipMemcpyDeviceToHost ) );
      if( h_grads )
         TNLMI_HIP( hipMemcpy( h_grads, S->grads.ptr, sizeof( float ) * kParams, hipMemcpyDeviceToHost ) );
   } );
}

tnlmi_status tnlmi_spai_apply( const tnlmi_spai* S, const tnlmi_matrix* A, double* d_M, tnlmi_stream stream )
{
   return guarded( [ & ] {
      if( ! S || ! d_M )
         fail( TNLMI_INVALID_ARGUMENT, "spai_apply: NULL argument" );
      check_csr( A );
      hipStream_t s = as_stream( stream );
      const Working work( *S, s );
      build_graph( work.w->g, *A, s );
      forward( *S, work.w->g, A->segments->offsets.ptr, A->column_indexes, work.w->a, false, d_M, s );
      TNLMI_HIP( hipStreamSynchronize( s ) );
   } );
}

tnlmi_status tnlmi_spai_loss_grad( tnlmi_spai* S, const tnlmi_matrix* A, const double* d_Z, int32_t K, double* loss,
                                   double* d_M, tnlmi_stream stream )
{
   return guarded( [ & ] {
      if( ! S || ! d_Z || K <= 0 || ! loss )
         fail( TNLMI_INVALID_ARGUMENT, "spai_loss_grad: invalid argument" );
      check_csr( A );
      const Working work( *S, as_stream( stream ) );
      *loss = loss_grad( *S, *work.w, *A, d_Z, K, d_M, as_stream( stream ) );
   } );
}

tnlmi_status tnlmi_spai_train_step( tnlmi_spai* S, const tnlmi_matrix* A, int32_t K, uint64_t probe_seed,
                                    float learning_rate, double* loss, tnlmi_stream stream )
{
   return guarded( [ & ] {
      if( ! S || K <= 0 || ! loss )
         fail( TNLMI_INVALID_ARGUMENT, "spai_train_step: invalid argument" );
      check_csr( A );
      hipStream_t s = as_stream( stream );
      const Working work( *S, s );
      DeviceArray< double >& Z = work.w->Z;
      Z.reserve( (int64_t) K * A->rows );
      hipLaunchKernelGGL( rademacher_k, g1( (int64_t) K * A->rows ), dim3( 256 ), 0, s, (int64_t) K * A->rows,
                          probe_seed, Z.ptr );
      *loss = loss_grad( *S, *work.w, *A, Z.ptr, K, nullptr, s );
      S->step++;
      const float b1 = 0.9f, b2 = 0.999f;
      const float c1 = 1.f - std::pow( b1, (float) S->step ), c2 = 1.f - std::pow( b2, (float) S->step );
      hipLaunchKernelGGL( adam_k, g1( kParams ), dim3( 256 ), 0, s, kParams, S->params.ptr, S->grads.ptr, S->m.ptr,
                          S->v.ptr, learning_rate, b1, b2, 1e-8f, c1, c2 );
      refresh( *S, s );
      TNLMI_HIP( hipGetLastError() );
      TNLMI_HIP( hipStreamSynchronize( s ) );
   } );
}

tnlmi_status tnlmi_bf16_gemm64( int64_t rows, const uint16_t* d_X, const uint16_t* d_W, float* d_Y,
                                tnlmi_stream stream )
{
   return guarded( [ & ] {
      if( rows < 0 || ! d_X || ! d_W || ! d_Y )
         fail( TNLMI_INVALID_ARGUMENT, "bf16_gemm64: invalid argument" );
      hipStream_t s = as_stream( stream );
      // Y = X W with W row-major [k][n]: the kernel reads B as Bn[n][k], the transpose
      DeviceArray< uint16_t > WT;
      WT.allocate( kH * kH );
      std::vector< uint16_t > h( kH * kH ), t( kH * kH );
      TNLMI_HIP( hipMemcpyAsync( h.data(), d_W, sizeof( uint16_t ) * kH * kH, hipMemcpyDeviceToHost, s ) );
      TNLMI_HIP( hipStreamSynchronize( s ) );
      for( int k = 0; k < kH; k++ )
         for( int nn = 0; nn < kH; nn++ )
            t[ nn * kH + k ] = h[ k * kH + nn ];
      TNLMI_HIP( hipMemcpyAsync( WT.ptr, t.data(), sizeof( uint16_t ) * kH * kH, hipMemcpyHostToDevice, s ) );
      EpiArgs e{};
      e.yf = d_Y;
      if( rows > 0 )
         gemm< 1, EPI_STORE >( rows, Term{ d_X, WT.ptr }, Term{ nullptr, nullptr }, Term{ nullptr, nullptr }, e, s );
      TNLMI_HIP( hipGetLastError() );
      TNLMI_HIP( hipStreamSynchronize( s ) );
   } );
}

}  // extern "C"
