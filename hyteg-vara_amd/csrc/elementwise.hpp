// Device code of the elementwise variable-coefficient P1 operator (kernel bodies shared by the single-problem and the batched launches).
#pragma once

#include "face_combine.hpp"

namespace hyg {

// stencil direction (C W E N S NW SE TC TW TS TSE BC BN BE BNW) from vertex k to vertex j of type t
constexpr int kMCDir[6][4][4] = { { { 0, 2, 3, 7 }, { 1, 0, 5, 8 }, { 4, 6, 0, 9 }, { 11, 13, 12, 0 } },
                                  { { 0, 3, 5, 7 }, { 4, 0, 1, 9 }, { 6, 2, 0, 10 }, { 11, 12, 14, 0 } },
                                  { { 0, 5, 7, 8 }, { 6, 0, 10, 9 }, { 11, 14, 0, 1 }, { 13, 12, 2, 0 } },
                                  { { 0, 7, 8, 9 }, { 11, 0, 1, 4 }, { 13, 2, 0, 6 }, { 12, 3, 5, 0 } },
                                  { { 0, 5, 1, 14 }, { 6, 0, 4, 11 }, { 2, 3, 0, 12 }, { 10, 7, 9, 0 } },
                                  { { 0, 2, 10, 7 }, { 1, 0, 9, 8 }, { 14, 12, 0, 5 }, { 11, 13, 6, 0 } } };
// offset of vertex k of type t from the anchor, encoded x + 2y + 4z
constexpr int kMCOff[6][4] = { { 0, 1, 2, 4 }, { 1, 3, 2, 5 }, { 1, 2, 5, 4 }, { 3, 7, 6, 5 }, { 5, 6, 4, 2 }, { 2, 3, 5, 6 } };
// 6 x the quadrature weights (centroid first), so that kb = 1 for k = 1
constexpr double kQW6[5] = { -0.8, 0.45, 0.45, 0.45, 0.45 };

__device__ __forceinline__ double expT( double a ) { return exp( a ); }
__device__ __forceinline__ float  expT( float a ) { return expf( a ); }

// Layout of the coefficient integrals of a cell: the rows of the anchor lattice (N points per edge) one after the other, each
// with the six types in turn, so that a row of a wave is one run of memory. Position of type 0, x = 0 of row (y, z); the
// types follow each other N - y - z values apart.
__device__ __forceinline__ int kbRow( int N, int y, int z ) { return 6 * ( S3i( N ) - S3i( N - z ) + rowStart( N - z, y ) ); }

// ------------------------------------------------------------------ 1. coefficient integrals
// k(x_q) = k0 exp( g ), g = sum_m a_m cos( theta_m + delta_mq ) with the phase theta_m of the anchor and delta_mq of the
// quadrature point's offset from it: for all anchors of a cell a product of the 30 x 2M matrix (a cos delta, -a sin delta)
// with the 2M x anchors matrix (cos theta, sin theta), done on the matrix cores (16 x 16 x 4 tiles of the same precision).
// e^(i theta) = X_m[x] Y_m[y] Z_m[z] from tables of the three lattice axes, so no sine is taken here.
//
// Rows of the product: 32 slots, 8 for each of the four 16-lane groups of a wave (that is where a lane finds its results):
// slots 0..4 of group g are the points of type g; types 4 and 5 are shared by groups 0, 1 and 2, 3 (points 0..2 and 3, 4 in
// slots 5..7), the last slot of groups 1 and 3 is empty. Columns: 16 anchors of a row.
// A block takes rowsPer (32, or 16 where that leaves too few blocks) rows of a plane, each wave every fourth of them; per tile
// of 16 anchors a wave holds X Z (2 values per step in registers) and walks its rows, whose Y is staged in LDS with the
// constant matrix. (Waves on tiles of their own, whose rows are fewer at large x: 1570 us in FP64 at level 7 on 24 cells, against 1130.)
// 32 modes, level 7, 24 cells (8.6 million anchors), FP32: apply 634 us, with a thread per anchor (kKBarPoint) 713. In FP64 the matrix
// instructions (30 ns each per SIMD, 600 us in all) and the exponentials, which use the same units, take longer than that thread's
// multiply-adds: 1231 against 1103. Where either is taken: kbOnMatrixCores.
constexpr int kKBarRows = 32;

typedef double f64x4 __attribute__( ( ext_vector_type( 4 ) ) );
typedef float  f32x4 __attribute__( ( ext_vector_type( 4 ) ) );
__device__ __forceinline__ f64x4 mma16( double a, double b, f64x4 c ) { return __builtin_amdgcn_mfma_f64_16x16x4f64( a, b, c, 0, 0, 0 ); }
__device__ __forceinline__ f32x4 mma16( float a, float b, f32x4 c ) { return __builtin_amdgcn_mfma_f32_16x16x4f32( a, b, c, 0, 0, 0 ); }
// lane group and slot within its tile of row i of a 16 x 16 result: FP64 results lie 4 rows apart, FP32 ones in sequence
__device__ __forceinline__ void mmaRow( int i, int& g, int& r, double* ) { g = i & 3, r = i >> 2; }
__device__ __forceinline__ void mmaRow( int i, int& g, int& r, float* ) { g = i >> 2, r = i & 3; }
// and the other way round
constexpr int mmaRowOf( int g, int r, double* ) { return 4 * r + g; }
constexpr int mmaRowOf( int g, int r, float* ) { return 4 * g + r; }

template < typename T >
struct KbPair
{
   T re, im;
};

template < typename T, int S >
__global__ __launch_bounds__( kBlock, S > 16 ? 1 : ( sizeof( T ) == 8 ? 2 : 3 ) ) void kKBar( int N, int nC, int rowsPer, const KbPair< T >* __restrict__ axis, const T* __restrict__ mat, T k0,
                                                   T* __restrict__ kb )
{
   typedef typename std::conditional< std::is_same< T, double >::value, f64x4, f32x4 >::type V4;
   constexpr int          MP = 2 * S;
   __shared__ T           At[S * 128];
   __shared__ KbPair< T > Yt[kKBarRows * MP];
   // cell fastest, then plane, then row chunk: all cells' blocks of a kind have the same work, so the 8 XCDs, which get blocks
   // in turn, are loaded alike, and the large blocks come first (row chunk fastest: one XCD had all the long rows, 2750 us)
   const int              c  = int( blockIdx.x ) % nC;
   const int              b  = int( blockIdx.x ) / nC;
   const int              z = b % N, y0 = b / N * rowsPer;
   if ( y0 + z >= N ) // (the whole block) no anchors
      return;
   const int          rows = min( rowsPer, N - z - y0 );
   const KbPair< T >* ax   = axis + i64( c ) * 3 * N * MP;
   for ( int i = int( threadIdx.x ); i < S * 128; i += kBlock )
      At[i] = mat[i64( c ) * S * 128 + i];
   for ( int i = int( threadIdx.x ); i < rows * MP; i += kBlock )
      Yt[i] = ax[( N + y0 ) * MP + i];
   __syncthreads();
   const int lane = int( threadIdx.x & 63u ), g = lane >> 4, h = g >> 1;
   const int tMax = g == 0 ? kMCMax[0] : ( g == 3 ? kMCMax[3] : kMCMax[1] ); // of type g (types 1 and 2 alike)
   T*        out  = kb + i64( c ) * 6 * S3i( N );
   const int wave = int( threadIdx.x >> 6 );
   for ( int xt = 0; 16 * xt < N - z - y0 - wave; ++xt )
   {
      const int x = 16 * xt + ( lane & 15 );
      T         a[S], d[S];
#pragma unroll
      for ( int s = 0; s < S; ++s )
      {
         const KbPair< T > X = ax[( 2 * s + h ) * N + min( x, N - 1 )], Z = ax[( 2 * N + z ) * MP + 2 * s + h];
         const T           re = X.re * Z.re - X.im * Z.im, im = X.re * Z.im + X.im * Z.re;
         a[s] = ( g & 1 ) ? im : re; // (X Z Y)'s real or imaginary part = a Y.re + d Y.im
         d[s] = ( g & 1 ) ? re : -im;
      }
      for ( int y = y0 + wave; y < y0 + rows && 16 * xt < N - z - y; y += kBlock / 64 )
      {
         V4                 c0 = { 0, 0, 0, 0 }, c1 = { 0, 0, 0, 0 };
         const KbPair< T >* Yr = Yt + ( y - y0 ) * MP + h;
#pragma unroll
         for ( int s = 0; s < S; ++s )
         {
            const KbPair< T > Y = Yr[2 * s];
            const T           v = a[s] * Y.re + d[s] * Y.im;
            c0                  = mma16( At[128 * s + lane], v, c0 );
            c1                  = mma16( At[128 * s + 64 + lane], v, c1 );
         }
         T v = T( kQW6[0] ) * expT( T( c0[0] ) );
#pragma unroll
         for ( int q = 1; q < 4; ++q )
            v += T( kQW6[q] ) * expT( T( c0[q] ) );
         v += T( kQW6[4] ) * expT( T( c1[0] ) );
         T e = T( ( g & 1 ) ? kQW6[3] : kQW6[0] ) * expT( T( c1[1] ) ) + T( kQW6[1] ) * expT( T( c1[2] ) );
         e += T( ( g & 1 ) ? 0.0 : kQW6[2] ) * expT( T( c1[3] ) );
         e += __shfl_xor( e, 16, 64 );
         const int nx = N - y - z;
         if ( x < nx )
         {
            // 0: the element is not in the cell
            T* o      = out + kbRow( N, y, z ) + x;
            o[g * nx] = x + tMax <= nx ? k0 * v : T( 0 );
            if ( !( g & 1 ) )
               o[( 4 + h ) * nx] = x + kMCMax[4] <= nx ? k0 * e : T( 0 );
         }
      }
   }
}
static_assert( kMCMax[1] == kMCMax[2] && kMCMax[4] == kMCMax[5], "types handled alike by kKBar" );

// The same integrals with a thread per anchor (consecutive anchors of the cell, whatever their rows), the matrix read with scalar
// loads: per mode three table values, two complex products and 60 multiply-adds.
template < typename T >
__global__ __launch_bounds__( kBlock ) void kKBarPoint( int N, int tilesPerCell, int nModes, int MP, const KbPair< T >* __restrict__ axis,
                                                        const T* __restrict__ mat, T k0, T* __restrict__ kb )
{
   typedef const T __attribute__( ( address_space( 4 ) ) ) CT;
   const int c    = int( blockIdx.x ) / tilesPerCell;
   const int s    = ( int( blockIdx.x ) - c * tilesPerCell ) * kBlock + int( threadIdx.x );
   if ( s >= S3i( N ) )
      return;
   int x, y, z;
   tetXYZ( N, s, x, y, z );
   const KbPair< T >* ax = axis + i64( c ) * 3 * N * MP;
   const CT*          mc = (const CT*) ( mat + i64( c ) * MP * 64 );
   T                  g[30];
#pragma unroll
   for ( int k = 0; k < 30; ++k )
      g[k] = T( 0 );
   for ( int m = 0; m < nModes; ++m )
   {
      const KbPair< T > X = ax[m * N + x], Y = ax[( N + y ) * MP + m], Z = ax[( 2 * N + z ) * MP + m];
      const T           re = X.re * Z.re - X.im * Z.im, im = X.re * Z.im + X.im * Z.re;
      const T           cs = re * Y.re - im * Y.im, sn = re * Y.im + im * Y.re;
      const CT*         a = mc + ( m >> 1 ) * 128 + ( m & 1 ) * 32;
#pragma unroll
      for ( int t = 0; t < 6; ++t )
#pragma unroll
         for ( int q = 0; q < 5; ++q )
         {
            // where kKBar holds point q of type t: group and slot
            const int gr = t < 4 ? t : 2 * ( t - 4 ) + ( q < 3 ? 0 : 1 ), j = t < 4 ? q : ( q < 3 ? q + 5 : q + 2 );
            const int o  = 64 * ( j >> 2 ) + mmaRowOf( gr, j & 3, static_cast< T* >( nullptr ) );
            g[5 * t + q] = fma( cs, a[o], fma( sn, a[o + 16], g[5 * t + q] ) );
         }
   }
   const int nx = N - y - z;
   T*        o  = kb + i64( c ) * 6 * S3i( N ) + kbRow( N, y, z ) + x;
#pragma unroll
   for ( int t = 0; t < 6; ++t )
   {
      T v = T( 0 );
#pragma unroll
      for ( int q = 0; q < 5; ++q )
         v += T( kQW6[q] ) * expT( g[5 * t + q] );
      o[t * nx] = x + kMCMax[t] <= nx ? k0 * v : T( 0 ); // 0: the element is not in the cell
   }
}

// The same integrals for a polynomial coefficient k(x) = sum_i poly[i] x^a y^b z^c over the monomials of degree <= deg
// in the order of the reference's MonomialBasis3D (by total degree; within a degree by decreasing a, then b). One
// thread per anchor; the polynomial is evaluated at the physical position of each of the 30 quadrature points.
template < typename T >
__global__ __launch_bounds__( kBlock ) void kKBarPoly( int L, int tilesPerCell, const ElemCell* __restrict__ cells,
                                                       const double* __restrict__ poly, int deg, T* __restrict__ kb )
{
   const int c    = int( blockIdx.x ) / tilesPerCell;
   const int tile = int( blockIdx.x ) - c * tilesPerCell;
   const int N    = 1 << L;
   const int S    = S3i( N );
   const int s    = tile * kBlock + int( threadIdx.x );
   if ( s >= S )
      return;
   int x, y, z;
   tetXYZ( N, s, x, y, z );
   const ElemCell& ec  = cells[c];
   T*              out = kb + i64( c ) * 6 * S + kbRow( N, y, z ) + x;
   const int       nx  = N - y - z;
   for ( int t = 0; t < 6; ++t )
   {
      if ( x + y + z + kMCMax[t] > N ) // the element is not in the cell
      {
         out[t * nx] = T( 0 );
         continue;
      }
      double v = 0.0;
      for ( int q = 0; q < 5; ++q )
      {
         double d[3] = { double( x ), double( y ), double( z ) };
         for ( int u = 0; u < 4; ++u )
         {
            const double lam = q == 0 ? 0.25 : ( u == q - 1 ? 0.5 : 1.0 / 6.0 );
            for ( int k = 0; k < 3; ++k )
               d[k] += lam * kMC[t][u][k];
         }
         double X[3];
         for ( int r = 0; r < 3; ++r )
            X[r] = ec.v0[r] + ec.a[r][0] * d[0] + ec.a[r][1] * d[1] + ec.a[r][2] * d[2];
         double kq = 0.0;
         int    i  = 0;
         for ( int dg = 0; dg <= deg; ++dg )
            for ( int ea = dg; ea >= 0; --ea )
               for ( int eb = dg - ea; eb >= 0; --eb, ++i )
               {
                  double mv = 1.0;
                  for ( int e = 0; e < ea; ++e )
                     mv *= X[0];
                  for ( int e = 0; e < eb; ++e )
                     mv *= X[1];
                  for ( int e = 0; e < dg - ea - eb; ++e )
                     mv *= X[2];
                  kq += poly[i] * mv;
               }
         v += kQW6[q] * kq;
      }
      out[t * nx] = T( v );
   }
}

// ------------------------------------------------------------------ 2. stencil application per cell
// entry i of the element matrix of type t in the value type
typedef const __attribute__( ( address_space( 4 ) ) ) ElemCell ElemCellAt;
__device__ __forceinline__ double elemK( ElemCellAt* ec, int t, int i, double* ) { return ec->mt[t][i]; }
__device__ __forceinline__ float  elemK( ElemCellAt* ec, int t, int i, float* ) { return ec->mtF[t][i]; }

// Stencil weights W[d] (C W E N S NW SE TC TW TS TSE BC BN BE BNW) of lattice point (px, py, pz) of a macro-cell
// from the coefficient integrals kc of its micro-cells (the incident ones that lie in the cell); DIAG: W[0] only.
template < typename T, bool DIAG >
__device__ __forceinline__ void elemWeights( ElemCellAt* ec, const T* __restrict__ kc, int N, int px, int py, int pz, T W[NDIR] )
{
   // anchors p - o for the eight offsets o in {0,1}^3 (encoded x + 2y + 4z)
   int  aIdx[8], aLen[8];
   bool aOk[8];
#pragma unroll
   for ( int o = 0; o < 8; ++o )
   {
      const int ax = px - ( o & 1 ), ay = py - ( ( o >> 1 ) & 1 ), az = pz - ( ( o >> 2 ) & 1 );
      aOk[o]       = ax >= 0 && ay >= 0 && az >= 0;
      aLen[o]      = aOk[o] ? N - ay - az : 0;
      aIdx[o]      = aOk[o] ? kbRow( N, ay, az ) + ax : 0;
   }
#pragma unroll
   for ( int d = 0; d < NDIR; ++d )
      W[d] = T( 0 );
#pragma unroll
   for ( int t = 0; t < 6; ++t )
#pragma unroll
      for ( int k = 0; k < 4; ++k )
      {
         const int o   = kMCOff[t][k];
         const int as  = px + py + pz - ( ( o & 1 ) + ( ( o >> 1 ) & 1 ) + ( ( o >> 2 ) & 1 ) );
         const bool ok = aOk[o] && as + kMCMax[t] <= N;
         const T    kv = ok ? kc[t * aLen[o] + aIdx[o]] : T( 0 );
         if constexpr ( DIAG )
            W[0] += kv * elemK( ec, t, 5 * k, static_cast< T* >( nullptr ) );
         else
#pragma unroll
            for ( int j = 0; j < 4; ++j )
               W[kMCDir[t][k][j]] += kv * elemK( ec, t, 4 * k + j, static_cast< T* >( nullptr ) );
      }
}

// ------------------------------------------------------------------ 3. the operator, z-marching wavefronts
// A "down" micro-cell is the point reflection of the "up" cell of its colour (p -> (1,1,1) - p up to a lattice step), so its
// element matrix holds the same entries: the vertex of type 0, 1 or 2 that vertex v of type 3, 4 or 5 is mapped to.
constexpr int kMCMirror[3][4] = { { 3, 0, 1, 2 }, { 2, 0, 1, 3 }, { 2, 3, 1, 0 } };
constexpr bool mirrorFits()
{
   for ( int t = 0; t < 3; ++t )
      for ( int a = 0; a < 4; ++a )
         for ( int b = 0; b < 4; ++b )
            for ( int k = 0; k < 3; ++k )
               if ( kMC[3 + t][a][k] - kMC[3 + t][b][k] != kMC[t][kMCMirror[t][b]][k] - kMC[t][kMCMirror[t][a]][k] )
                  return false;
   return true;
}
static_assert( mirrorFits(), "down micro-cells are point reflections of up micro-cells" );
constexpr int kMCEdge[4][4] = { { -1, 0, 1, 2 }, { 0, -1, 3, 4 }, { 1, 3, -1, 5 }, { 2, 4, 5, -1 } }; // vertex pair -> edge

// Contributions of the six micro-cells of the cube anchored at one lattice point to its eight corners (x + 2y + 4z):
// y_i += sum_t kb_t K_t[i,j] (u_j - u_i) over the element edges (the rows of K_t sum to zero). Elements that share an edge
// of the cube share its difference: 19 edges, 36 products with kb, against 96 for the element matrices. K: the edge entries
// of the three up types. Only the corners in WANT are formed.
template < typename T, int WANT >
__device__ __forceinline__ void cubeContributions( const T ( &K )[3][6], const T ( &k )[6], const T ( &u )[8], T ( &acc )[8] )
{
   constexpr int EA[6] = { 0, 0, 0, 1, 1, 2 }, EB[6] = { 1, 2, 3, 2, 3, 3 }; // vertex pairs of an element
#pragma unroll
   for ( int i = 0; i < 8; ++i )
#pragma unroll
      for ( int j = i + 1; j < 8; ++j )
      {
         if ( !( ( WANT >> i ) & 1 ) && !( ( WANT >> j ) & 1 ) )
            continue;
         T    c    = T( 0 );
         bool edge = false;
#pragma unroll
         for ( int t = 0; t < 6; ++t )
#pragma unroll
            for ( int e = 0; e < 6; ++e )
            {
               const int a = kMCOff[t][EA[e]], b = kMCOff[t][EB[e]];
               if ( ( a == i && b == j ) || ( a == j && b == i ) )
               {
                  const T w = K[t % 3][t < 3 ? e : kMCEdge[kMCMirror[t % 3][EA[e]]][kMCMirror[t % 3][EB[e]]]];
                  c         = edge ? fma( k[t], w, c ) : k[t] * w;
                  edge      = true;
               }
            }
         if ( !edge )
            continue;
         const T d = u[j] - u[i];
         if ( ( WANT >> i ) & 1 )
            acc[i] = fma( c, d, acc[i] );
         if ( ( WANT >> j ) & 1 )
            acc[j] = fma( -c, d, acc[j] );
      }
}

// one-sided sum of a point on a cell's face (slot 1..4), edge or vertex, for kFaceCombine / kLowCombine
template < typename T >
__device__ __forceinline__ void elemStoreBoundary( int c, int N, int slot, int px, int py, int pz, T val, int flag,
                                                   const CellInfo* __restrict__ cinfo, const CellFaceSlot* __restrict__ cfs,
                                                   const LowerPrim* __restrict__ prims, const LowerEntry* __restrict__ entries,
                                                   T* __restrict__ part, T* __restrict__ lowPart )
{
   const int NP = N + 1;
   if ( slot <= 4 )
   {
      const CellFaceSlot fs = cfs[4 * c + slot - 1];
      if ( fs.bc & flag )
         part[i64( fs.block ) * NP * NP + facePartIndex( slot - 1, N, px, py, pz )] = val;
      return;
   }
   const CellInfo& ci = cinfo[c];
   if ( !( prims[ci.prim[slot]].bc & flag ) )
      return;
   const int e = ci.entry[slot];
   int       i = 0;
   if ( slot <= 10 )
   {
      const int b[4] = { N - px - py - pz, px, py, pz };
      i              = b[entries[e].l1];
   }
   lowPart[i64( e ) * NP + i] = val;
}

// The (type, node, node) entries of the element matrices that make up each stencil direction, in the order of elemWeights.
struct ElemTerms
{
   int first[NDIR + 1] = {}, term[96] = {}; // term: type + 8 node + 32 other node
};
constexpr ElemTerms elemTermTable()
{
   ElemTerms tb;
   int       n = 0;
   for ( int d = 0; d < NDIR; ++d )
   {
      tb.first[d] = n;
      for ( int t = 0; t < 6; ++t )
         for ( int k = 0; k < 4; ++k )
            for ( int j = 0; j < 4; ++j )
               if ( kMCDir[t][k][j] == d )
                  tb.term[n++] = t + 8 * k + 32 * j;
   }
   tb.first[NDIR] = n;
   return tb;
}
static __constant__ ElemTerms kElemTerms = elemTermTable();

// The operator's value (the cell's part of it) at one point as elemWeights and bElemApply form it, a direction of weight 0 not
// looked at: what kElemSweep takes where its sums are not finite. Loops that are not unrolled, for few registers.
template < typename T >
__device__ __forceinline__ T elemValue( ElemCellAt* ec, const T* __restrict__ kc, const T* __restrict__ xc, int N, int px, int py, int pz )
{
   const T x0  = xc[cidx( N + 1, px, py, pz )];
   T       val = T( 0 );
#pragma unroll 1
   for ( int d = 1; d < NDIR; ++d )
   {
      T w = T( 0 );
#pragma unroll 1
      for ( int i = kElemTerms.first[d]; i < kElemTerms.first[d + 1]; ++i )
      {
         const int e = kElemTerms.term[i], t = e & 7, k = ( e >> 3 ) & 3, j = e >> 5, o = kMCOff[t][k];
         const int ax = px - ( o & 1 ), ay = py - ( ( o >> 1 ) & 1 ), az = pz - ( ( o >> 2 ) & 1 );
         if ( ax >= 0 && ay >= 0 && az >= 0 && ax + ay + az + kMCMax[t] <= N )
            w += kc[kbRow( N, ay, az ) + t * ( N - ay - az ) + ax] * elemK( ec, t, 4 * k + j, static_cast< T* >( nullptr ) );
      }
      const bool on = w != T( 0 );
      val += w * ( xc[cidx( N + 1, px + ( on ? dirX( d ) : 0 ), py + ( on ? dirY( d ) : 0 ), pz + ( on ? dirZ( d ) : 0 ) )] - x0 );
   }
   return val;
}

template < typename T >
struct ElemArgs
{
   const ZSeg*         segs;
   int                 nSegs, nC, L;
   i64                 stride;
   const ElemCell*     cells;
   const T*            kb;
   const CellInfo*     cinfo;
   const CellFaceSlot* cfs;
   const LowerPrim*    prims;
   const LowerEntry*   entries;
   T*                  part;
   T*                  lowPart;
   const T*            dinv;
   int                 flag;
   const T*            x;
   const T*            in1;
   T*                  out0;
   T*                  out1;
   T                   a;
};

// the arguments of a sweep in constant memory (the kernel's argument segment, or a batch's task table)
template < typename T >
using ElemArgsAt = const __attribute__( ( address_space( 4 ) ) ) ElemArgs< T >*;

// What a wave loads for one cube layer z: kb of the six types of anchor rows y-1 and y, and point rows y-1 .. y+1 of plane z+1.
template < typename T >
struct ElemLayer
{
   T k[2][6];
   T u[3];
};

// All points of the closed cells. A wave owns a row y and 62 points (x0 .., lanes 1..62) and marches z: layer z (the cubes
// between planes z and z+1 in the anchor rows y-1 and y) gives its contributions to plane z, which completes it, and to plane z+1,
// which are carried; corners at x+1 are moved by one lane shift per row. A point costs 12 loads of kb and 3 of values (120 B in
// FP64 requested, of which neighbouring rows find half in cache) and 14 edges of either cube (28 products with a difference), where
// a thread per point gathers 24 kb and 15 values. Bound by the vector instructions of a step (180 FP32, of which 105 are the edge
// products) at 55% of the lanes at level 7: rows of a tetrahedron end inside the 62-point windows. Two rows per wave share more
// loads and edge differences but halve the waves in flight (FP32 sweep at level 7 on 24 cells 208 against 196 us, both with 24-plane
// segments).
// A sum of differences turns an infinite value into NaN at points whose weight for it is 0 (and at the point itself): a plane with
// a sum that is not finite stores nothing and is done again point by point behind the march (planes: one bit each).
// Lanes outside a row, rows outside a plane and anchors outside the cell load 0 (the descriptor's range check), so they
// add nothing; elements that stick out of the cell have kb = 0.
// The arguments are read where they are used (ap, made opaque for the rare boundary rows): held in scalar registers through
// the march they spilled, 66 of 250 vector instructions per plane.
template < typename T, int MODE >
__device__ __forceinline__ void elemSweep( int bid, ElemArgsAt< T > ap )
{
   const auto&    p    = *ap;
   constexpr bool kIn1 = MODE == MODE_RESIDUAL || MODE == MODE_JACOBI || MODE == MODE_CHEB0 || MODE == MODE_CHEBK;
   constexpr bool kE   = kIn1 || MODE == MODE_APPLY_ADD;
   constexpr bool kD   = MODE == MODE_JACOBI || MODE == MODE_CHEB0 || MODE == MODE_CHEBK;
   constexpr bool kTwo = MODE == MODE_CHEB0 || MODE == MODE_CHEBK;
   constexpr int  B    = int( sizeof( T ) );
   const int      nbx  = ( p.nSegs + 3 ) / 4, nb = nbx * p.nC; // blocks per cell
   const int      lb   = remapXcd( bid, nb );
   if ( lb >= nb )
      return;
   const int c  = lb / nbx;
   const int si = ( lb - c * nbx ) * 4 + __builtin_amdgcn_readfirstlane( int( threadIdx.x ) >> 6 );
   if ( si >= p.nSegs )
      return;
   const ZSeg     sg = p.segs[si];
   const int      N = 1 << p.L, w = N + 1, NP = N + 1, y0 = sg.y, x0 = sg.x0, z0 = sg.z0, z1 = sg.z1;
   const int      lane = int( threadIdx.x & 63u );
   const int      px   = x0 - 1 + lane;
   const int      SN = S3i( N ), SW = S3i( w );
   const i64      cb    = i64( c ) * p.stride;
   const unsigned bytes = unsigned( ( p.stride + kTailSlack ) * B );
   const auto     rx = makeRsrc( p.x + cb, bytes ), r0 = makeRsrc( p.out0 + cb, bytes );
   const auto     re = makeRsrc( kIn1 ? p.in1 + cb : p.out0 + cb, bytes ), r1 = makeRsrc( kTwo ? p.out1 + cb : p.out0 + cb, bytes );
   const auto     rd = makeRsrc( kD ? p.dinv + cb : p.x + cb, bytes );
   const T*       kc = p.kb + i64( c ) * 6 * SN;
   // the x = 0 and diagonal faces (slots 2 and 3)
   const CellFaceSlot f2 = p.cfs[4 * c + 2], f3 = p.cfs[4 * c + 3];
   const auto         rp2 = makeRsrc( p.part + i64( f2.block ) * NP * NP, unsigned( NP * NP * B ) );
   const auto         rp3 = makeRsrc( p.part + i64( f3.block ) * NP * NP, unsigned( NP * NP * B ) );
   ElemCellAt*        ec  = uniformPtr( p.cells + c );
   T                  K[3][6];
   constexpr int      EA[6] = { 0, 0, 0, 1, 1, 2 }, EB[6] = { 1, 2, 3, 2, 3, 3 };
#pragma unroll
   for ( int t = 0; t < 3; ++t )
#pragma unroll
      for ( int e = 0; e < 6; ++e )
         K[t][e] = elemK( ec, t, 4 * EA[e] + EB[e], static_cast< T* >( nullptr ) );

   // point row y of plane z: byte offset of x = 0, and the number of its points (0 outside the cell)
   auto rowU = [&]( int y, int z, int& n ) {
      n = y >= 0 && z >= 0 ? max( 0, N - y - z + 1 ) : 0;
      return n > 0 ? ( SW - S3i( w - z ) + rowStart( w - z, y ) ) * B : 0;
   };
   auto loadU = [&]( int y, int z ) {
      int       n;
      const int o = rowU( y, z, n );
      return bufLoad< T >( rx, unsigned( px ) < unsigned( n ) ? unsigned( px * B ) : kDropOffset, o );
   };
   // layer z: kb of the anchor rows and the point rows of plane z+1
   auto loadLayer = [&]( ElemLayer< T >& Q, int z ) {
      const int  W  = N - z; // anchors of row 0
      const auto rk = makeRsrc( kc + 6 * ( SN - S3i( W ) ), W > 0 ? unsigned( 6 * T2i( W ) * B ) : 0u );
#pragma unroll
      for ( int r = 0; r < 2; ++r )
      {
         const int      y = y0 - 1 + r, n = y >= 0 ? max( 0, W - y ) : 0;
         const int      o  = n > 0 ? 6 * rowStart( W, y ) * B : 0;
         const unsigned vo = unsigned( px ) < unsigned( n ) ? unsigned( px * B ) : kDropOffset;
#pragma unroll
         for ( int t = 0; t < 6; ++t )
            Q.k[r][t] = bufLoad< T >( rk, vo, o + t * n * B );
      }
#pragma unroll
      for ( int r = 0; r < 3; ++r )
         Q.u[r] = loadU( y0 - 1 + r, z + 1 );
   };
   T lo[3], loX[3]; // plane z: the rows and their values at x+1
   T cn = T( 0 ), cs = T( 0 ); // contributions of layer z-1 to plane z: at the anchor's x, and at x+1 (to be shifted)
   // contributions of layer z: `first` forms only those to plane z+1
   auto layer = [&]( const ElemLayer< T >& Q, const T ( &hiX )[3], bool first, T& n, T& s ) {
      n  = cn;
      s  = cs;
      cn = cs = T( 0 );
#pragma unroll
      for ( int r = 0; r < 2; ++r )
      {
         const T u[8] = { lo[r], loX[r], lo[r + 1], loX[r + 1], Q.u[r], hiX[r], Q.u[r + 1], hiX[r + 1] };
         T       q[8];
#pragma unroll
         for ( int k = 0; k < 8; ++k )
            q[k] = T( 0 );
         // the row's points are the upper y corners of anchor row y-1 and the lower ones of row y
         if ( r == 0 )
         {
            if ( first )
               cubeContributions< T, 0xc0 >( K, Q.k[r], u, q );
            else
               cubeContributions< T, 0xcc >( K, Q.k[r], u, q );
            n += q[2];
            s += q[3];
            cn += q[6];
            cs += q[7];
         }
         else
         {
            if ( first )
               cubeContributions< T, 0x30 >( K, Q.k[r], u, q );
            else
               cubeContributions< T, 0x33 >( K, Q.k[r], u, q );
            n += q[0];
            s += q[1];
            cn += q[4];
            cs += q[5];
         }
      }
   };
   const bool     on2 = x0 == 0 && ( f2.bc & p.flag ) != 0, on3 = ( f3.bc & p.flag ) != 0;
   const bool     mine = lane >= 1 && lane <= 62;
   const int      pIn  = mine && px > 0 && ( p.flag & 1 ) ? px : ( 1 << 28 ); // interior when it lies before the row end
   const unsigned vx   = unsigned( px * B ), v2 = mine && px == 0 ? 0u : kDropOffset;
   const T        a    = p.a;
   int            z    = z0;
   // points of the planes z = 0 and y = 0 and the edge x = 0 on the diagonal face
   auto boundary = [&]( int y, T val ) {
      ElemArgsAt< T > q = ap;
      asm volatile( "" : "+s"( q ) );
      elemStoreBoundary( c, N, classifySlot( N, px, y, z ), px, y, z, val, q->flag, q->cinfo, q->cfs, q->prims, q->entries, q->part,
                         q->lowPart );
   };
   unsigned again = 0; // planes that are done again
   T        vEdge = T( 0 ); // value of the row's point on the edge between local vertices 2 and 3 (x = 0 on the diagonal face)
   // one plane: `cur` holds layer z, `nxt` receives layer z+1; EDGE: the row or the plane lies on a face of the cell
   auto step = [&]( auto EDGE, ElemLayer< T >& cur, ElemLayer< T >& nxt ) {
      int       cnt;
      const int o = rowU( y0, z, cnt );
      // lanes past the row end read what follows in the array (or 0 past its slack); their results are dropped
      const T ein = kE ? bufLoad< T >( re, vx, o ) : T( 0 ), edi = kD ? bufLoad< T >( rd, vx, o ) : T( 0 );
      if ( z + 1 < z1 )
         loadLayer( nxt, z + 1 );
      T hiX[3], n, s;
#pragma unroll
      for ( int r = 0; r < 3; ++r )
         hiX[r] = laneMove< kDppWaveShl1 >( cur.u[r] );
      layer( cur, hiX, false, n, s );
      const T   Ax = n + laneMove< kDppWaveShr1 >( s );
      const int xe = N - y0 - z; // row end
      if ( xe >= x0 ) // (wave-uniform) something of the row in the window
      {
         if ( __builtin_expect( __ballot( !isfinite( Ax ) ) != 0, 0 ) )
            again |= 1u << ( z - z0 );
         else if ( EDGE.value && ( y0 == 0 || z == 0 ) )
         {
            if ( mine && px <= xe )
               boundary( y0, Ax );
         }
         else
         {
            T q0 = T( 0 ), q1 = T( 0 );
            epilogue< T, MODE >( Ax, lo[1], ein, ein, edi, a, q0, q1 );
            const unsigned so = pIn < xe ? vx : kDropOffset;
            bufStore( q0, r0, so, o );
            if constexpr ( kTwo )
               bufStore( q1, r1, so, o );
            if ( xe > 0 )
            {
               // face points: x = 0 and the row end
               if ( on2 )
                  bufStore( Ax, rp2, v2, facePartIndex( 2, N, 0, y0, z ) * B );
               if ( on3 && xe <= x0 + 61 )
                  bufStore( Ax, rp3, mine && px == xe ? 0u : kDropOffset, facePartIndex( 3, N, xe, y0, z ) * B );
            }
            else
               vEdge = Ax;
         }
      }
#pragma unroll
      for ( int r = 0; r < 3; ++r )
      {
         lo[r]  = cur.u[r];
         loX[r] = hiX[r];
      }
      ++z;
   };
   ElemLayer< T > A, Bq;
   if ( z0 > 0 )
   {
      T hiX[3], n, s;
#pragma unroll
      for ( int r = 0; r < 3; ++r )
         lo[r] = loadU( y0 - 1 + r, z0 - 1 );
      loadLayer( Bq, z0 - 1 );
      loadLayer( A, z0 );
#pragma unroll
      for ( int r = 0; r < 3; ++r )
      {
         loX[r] = laneMove< kDppWaveShl1 >( lo[r] );
         hiX[r] = laneMove< kDppWaveShl1 >( Bq.u[r] );
      }
      layer( Bq, hiX, true, n, s );
#pragma unroll
      for ( int r = 0; r < 3; ++r )
      {
         lo[r]  = Bq.u[r];
         loX[r] = hiX[r];
      }
   }
   else
   {
#pragma unroll
      for ( int r = 0; r < 3; ++r )
         lo[r] = loadU( y0 - 1 + r, 0 );
      loadLayer( A, 0 );
#pragma unroll
      for ( int r = 0; r < 3; ++r )
         loX[r] = laneMove< kDppWaveShl1 >( lo[r] );
   }
   // The general stores of the row y = 0 and the plane z = 0 stay out of the main loop, whose scalar registers they would
   // spill.
   if ( y0 == 0 || z0 == 0 )
      do
      {
         step( std::true_type(), A, Bq );
         A = Bq;
      } while ( y0 == 0 && z < z1 );
   while ( z < z1 )
   {
      step( std::false_type(), A, Bq );
      if ( z >= z1 )
         break;
      step( std::false_type(), Bq, A );
   }
   if ( x0 == 0 && lane == 1 )
   {
      z = N - y0;
      if ( y0 > 0 && z > 0 && z >= z0 && z < z1 )
         boundary( y0, vEdge );
   }
   if ( again != 0 )
   {
      ElemArgsAt< T > q = ap;
      asm volatile( "" : "+s"( q ) );
      for ( ; again != 0; again &= again - 1 )
      {
         z = z0 + __builtin_ctz( again );
         if ( lane < 1 || lane > 62 || px > N - y0 - z )
            continue;
         const i64 cq  = i64( c ) * q->stride;
         const T   val = elemValue( uniformPtr( q->cells + c ), q->kb + i64( c ) * 6 * S3i( N ), q->x + cq, N, px, y0, z );
         if ( classifySlot( N, px, y0, z ) != 0 )
            boundary( y0, val );
         else if ( q->flag & 1 )
         {
            const i64 o  = cq + cidx( N + 1, px, y0, z );
            const T   e  = kIn1 ? q->in1[o] : ( MODE == MODE_APPLY_ADD ? q->out0[o] : T( 0 ) );
            T         q0 = T( 0 ), q1 = T( 0 );
            epilogue< T, MODE >( val, q->x[o], e, e, kD ? q->dinv[o] : T( 0 ), q->a, q0, q1 );
            q->out0[o] = q0;
            if constexpr ( kTwo )
               q->out1[o] = q1;
         }
      }
   }
}

// wavefronts per SIMD
template < typename T >
constexpr int kElemOccupancy = sizeof( T ) == 4 ? 6 : 3;

template < typename T, int MODE >
__global__ __launch_bounds__( kBlock, kElemOccupancy< T > ) void kElemSweep( ElemArgs< T > p )
{
   // p is the whole argument segment
   elemSweep< T, MODE >( int( blockIdx.x ), (ElemArgsAt< T >) __builtin_amdgcn_kernarg_segment_ptr() );
}

// arguments of the sweep of one level, and its blocks
template < typename T >
ElemArgs< T > elemArgs( const MeshCtx& m, const LevelGeom& g, const hyg_op_s::Level& ol, int L, const StencilCall& c )
{
   constexpr bool dbl = std::is_same< T, double >::value;
   ElemArgs< T >  e;
   e.segs    = g.eSegs;
   e.nSegs   = g.nESegs;
   e.nC      = m.mesh->nC();
   e.L       = L;
   e.stride  = g.stride;
   e.cells   = ol.elem;
   e.kb      = dbl ? (const T*) ol.kb : (const T*) ol.kbF;
   e.cinfo   = m.cellInfo;
   e.cfs     = m.cellFaces;
   e.prims   = m.prims;
   e.entries = m.entries;
   e.part    = dbl ? (T*) ol.facePart : (T*) ol.facePartF;
   e.lowPart = dbl ? (T*) ol.lowPart : (T*) ol.lowPartF;
   e.dinv    = dbl ? (const T*) ol.dinv : (const T*) ol.dinvF;
   e.flag    = c.flag;
   e.x       = (const T*) c.x;
   e.in1     = (const T*) c.in1;
   e.out0    = (T*) c.out0;
   e.out1    = (T*) c.out1;
   e.a       = T( c.a );
   return e;
}
template < typename T >
int elemBlocks( const ElemArgs< T >& e )
{
   return xcdGrid( ( ( e.nSegs + 3 ) / 4 ) * e.nC );
}

// blocks per cell with a thread per point
__host__ __device__ constexpr int elemTiles( int L ) { return ( S3i( ( 1 << L ) + 1 ) + kBlock - 1 ) / kBlock; }

// March (kElemSweep) or a thread per point (kElemApply)? The march reads each integral and value about once but fills 62-point
// windows with rows of at most N + 1 points and walks its planes one after the other; threads gather 24 integrals and 15 values each,
// most of them from cache, and pack their lanes whatever the length of the rows. Sweep with kept integrals, threads / march, us:
// level 8, 24 cells FP64 1838 / 1393, FP32 1443 / 759, 6 cells 424 / 361, 365 / 195; level 7, 162 cells 1642 / 1507, 1294 / 819, 24
// cells 250 / 251, 193 / 122, 6 cells 51 / 64, 49 / 43, 3 cells 32.4 / 38.5, 28.1 / 27.7, 1 cell 14.6 / 17.2, 12.2 / 13.9; level 6, 162
// cells 234 / 332, 164 / 156, 24 cells 37 / 57, 32 / 39 (eight such problems in a batch 281 / 421, 221 / 226); level 5, 24 cells in a
// batch of six 34 / 86, 30 / 54; level 4, 960 cells 42 / 172, 40 / 99; level 4, 3 cells 10.0 / 13.7, 10.2 / 13.1. In a batch a problem
// takes the route that it takes alone, so that its results are the same.
inline bool elemMarches( int L, int nC, int dtype )
{
   if ( dtype == 4 )
      return L >= 8 || ( L == 7 && nC >= 3 ) || ( L == 6 && nC >= 100 );
   return L >= 8 || ( L == 7 && nC >= 64 );
}

// One thread per point of the closed macro-cell. DIAG: the diagonal entry instead of
// the product. BND: the points on the cell's faces, edges and vertices only, listed in bnd[0 .. nBnd) by their index in the
// cell array (the surrogate operator does the interior points itself). STW: the point's stencil weights are read from wst
// ([cell][direction][point], the blended operator) instead of assembled from the coefficient integrals.
template < typename T, int MODE, bool DIAG, bool BND = false, bool STW = false >
__device__ __forceinline__ void bElemApply( int bid, int L, int tilesPerCell, i64 stride, const ElemCell* __restrict__ cells,
                                                        const T* __restrict__ kb, const CellInfo* __restrict__ cinfo,
                                                        const CellFaceSlot* __restrict__ cfs, const LowerPrim* __restrict__ prims,
                                                        const LowerEntry* __restrict__ entries, T* __restrict__ part,
                                                        T* __restrict__ lowPart, const T* __restrict__ dinv, int flag,
                                                        const T* __restrict__ x, const T* __restrict__ in1,
                                                        T* __restrict__ out0, T* __restrict__ out1, T a,
                                                        const int* __restrict__ bnd = nullptr, int nBnd = 0,
                                                        const T* __restrict__ wst = nullptr )
{
   const int c    = bid / tilesPerCell;
   const int tile = bid - c * tilesPerCell;
   const int N = 1 << L, w = N + 1;
   int       s = tile * kBlock + int( threadIdx.x );
   if constexpr ( BND )
   {
      if ( s >= nBnd )
         return;
      s = bnd[s];
   }
   else if ( s >= S3i( w ) )
      return;
   int px, py, pz;
   tetXYZ( w, s, px, py, pz );
   const int slot = classifySlot( N, px, py, pz );
   if ( slot == 0 && !( flag & 1 ) )
      return;
   T W[NDIR];
   if constexpr ( STW )
   {
      const T* wc = wst + i64( c ) * NDIR * S3i( w ) + s;
#pragma unroll
      for ( int d = 0; d < NDIR; ++d )
         W[d] = ( DIAG && d > 0 ) ? T( 0 ) : wc[i64( d ) * S3i( w )];
   }
   else
      elemWeights< T, DIAG >( uniformPtr( cells + c ), kb + i64( c ) * 6 * S3i( N ), N, px, py, pz, W );
   const i64 q = i64( c ) * stride + cidx( w, px, py, pz );
   T         val;
   if constexpr ( DIAG )
      val = W[0];
   else
   {
      const int Wz = w - pz;
      const int tc = T2i( Wz ) - py, bc = T2i( Wz + 1 ) - py, nn = Wz - py;
      const int off[NDIR] = { 0, -1, 1, nn, -( nn + 1 ), nn - 1, -nn, tc, tc - 1, tc - nn, tc - nn + 1, -bc, -bc + nn + 1, -bc + 1, -bc + nn };
      val = T( 0 );
      if constexpr ( STW )
      {
#pragma unroll
         for ( int d = 0; d < NDIR; ++d )
            val += W[d] * x[q + ( W[d] != T( 0 ) ? off[d] : 0 )];
      }
      else
      {
         // The rows of the element matrices sum to zero: differences to the point, which lose less in FP32 than the weights'
         // sum (error of a V-cycle of twelve problems against FP64 1.2e-7 instead of 3.0e-7) and need no centre weight. A direction of
         // weight 0 is not looked at.
         const T x0 = x[q];
#pragma unroll
         for ( int d = 1; d < NDIR; ++d )
            val += W[d] * ( x[q + ( W[d] != T( 0 ) ? off[d] : 0 )] - x0 );
      }
   }
   if ( slot == 0 )
   {
      if constexpr ( DIAG )
         out0[q] = val;
      else
      {
         T i1 = T( 0 ), r0, r1;
         if constexpr ( MODE == MODE_RESIDUAL || MODE == MODE_JACOBI || MODE == MODE_CHEB0 || MODE == MODE_CHEBK )
            i1 = in1[q];
         if constexpr ( MODE == MODE_APPLY_ADD )
            i1 = out0[q];
         epilogue< T, MODE >( val, x[q], i1, i1, dinv[q], a, r0, r1 );
         out0[q] = r0;
         if constexpr ( MODE == MODE_CHEB0 || MODE == MODE_CHEBK )
            out1[q] = r1;
      }
   }
   else
      elemStoreBoundary( c, N, slot, px, py, pz, val, flag, cinfo, cfs, prims, entries, part, lowPart );
}

template < typename T, int MODE, bool DIAG, bool BND = false, bool STW = false >
__global__ __launch_bounds__( kBlock ) void kElemApply( int L, int tilesPerCell, i64 stride, const ElemCell* __restrict__ cells,
                                                        const T* __restrict__ kb, const CellInfo* __restrict__ cinfo,
                                                        const CellFaceSlot* __restrict__ cfs, const LowerPrim* __restrict__ prims,
                                                        const LowerEntry* __restrict__ entries, T* __restrict__ part,
                                                        T* __restrict__ lowPart, const T* __restrict__ dinv, int flag,
                                                        const T* __restrict__ x, const T* __restrict__ in1,
                                                        T* __restrict__ out0, T* __restrict__ out1, T a,
                                                        const int* __restrict__ bnd = nullptr, int nBnd = 0,
                                                        const T* __restrict__ wst = nullptr, int nb = 0 )
{
   // nb > 0: the grid is padded to a multiple of 8 and each XCD takes a contiguous range of cells (the hardware deals
   // workgroups out round-robin over the XCDs), so a cell's coefficients and source stay in one XCD's L2
   const int b = nb > 0 ? remapXcd( int( blockIdx.x ), nb ) : int( blockIdx.x );
   if ( nb > 0 && b >= nb )
      return;
   bElemApply< T, MODE, DIAG, BND, STW >( b, L, tilesPerCell, stride, cells, kb, cinfo, cfs, prims, entries, part, lowPart, dinv, flag, x,
                                          in1, out0, out1, a, bnd, nBnd, wst );
}

} // namespace hyg
