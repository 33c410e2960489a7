// Shared by the P2 kernels of p2.hip and the on-the-fly variable-coefficient kernels (p2kq.hpp): class
// sub-lattices of a cell's points, the tile tables that map blocks to them, and the assembly of a point's stencil
// from the coefficient values at the quadrature points of its micro-cells.
#pragma once
#include "face_combine.hpp"

#include <utility>

namespace hyg {

__host__ __device__ constexpr int triCount( int n )
{
   return n > 0 ? n * ( n + 1 ) / 2 : 0;
}

// number of points of one (ku, kv) sub-lattice inside a cell face (face coordinates u = 2 i + 2 - ku, v = 2 j + 2 - kv)
__host__ __device__ constexpr int p2FaceSubCount( int N, int ku, int kv )
{
   return N - 5 + ku + kv < 0 ? 0 : triCount( ( N - 5 + ku + kv ) / 2 + 1 );
}
struct P2FaceTiles
{
   int start[5]; // first tile of each (ku, kv) = (s & 1, s >> 1) sub-lattice within a face; start[4] = per face
};

// parity class of the points of face F whose face coordinates have parities (KU, KV)
__host__ __device__ constexpr int p2FaceClass( int F, int KU, int KV )
{
   return ( F == 2 ? 0 : KU ) | ( ( F == 0 ? KV : ( F == 2 ? KU : ( F == 3 ? ( KU + KV ) & 1 : 0 ) ) ) << 1 ) | ( ( F == 0 ? 0 : KV ) << 2 );
}

// interior points of a lattice with N intervals of parity class cls: p = 2 q + cls, q' = q - (1 - cls), |q'| <= M
__host__ __device__ constexpr int p2InteriorExtent( int N, int cls )
{
   const int k = ( cls & 1 ) + ( ( cls >> 1 ) & 1 ) + ( ( cls >> 2 ) & 1 );
   return ( N - 1 - k ) / 2 - ( 3 - k );
}
// all points of parity class cls of a cell lattice with N intervals: p = 2 q + cls, |q| <= M; M = -1 when the class
// has no point (N = 2, cls = 7: (1, 1, 1) lies outside the cell; integer division would round -1/2 up to 0)
__host__ __device__ constexpr int p2ClassExtent( int N, int cls )
{
   const int r = N - ( cls & 1 ) - ( ( cls >> 1 ) & 1 ) - ( ( cls >> 2 ) & 1 );
   return r < 0 ? -1 : r / 2;
}
struct P2ClassTiles
{
   int start[65]; // first tile of each class within a cell; start[nClasses] = tiles per cell
};

// tiles of all points of each class of a cell
inline P2ClassTiles p2ClassTiles( int N )
{
   P2ClassTiles ct;
   ct.start[0] = 0;
   for ( int k = 0; k < 8; ++k )
      ct.start[k + 1] = ct.start[k] + ceilDiv( S3i( p2ClassExtent( N, k ) + 1 ), kBlock );
   return ct;
}

// up to three functions handled by one stored-stencil pass (the components of a vector function)
template < typename T >
struct P2Comps
{
   const T* x[3];
   const T* in1[3];
   T*       out0[3];
   T*       out1[3];
};

// Stored stencils (setup) and the on-the-fly apply: the stencil of a point is the sum, over the micro-cells that have
// it as node l (on the cell's side of face F for a face point), of row l of its element matrix, keyed by the offset to
// the other node.
constexpr int p2OffsetIndex( const P2StencilOffsets& o, int dx, int dy, int dz )
{
   for ( int e = 0; e < o.n; ++e )
      if ( o.d[e][0] == dx && o.d[e][1] == dy && o.d[e][2] == dz )
         return e;
   return -1;
}
constexpr int kP2MaxPairs = 24; // micro-cells of a point: 24 at vertex nodes, fewer in the edge-midpoint classes

// Element matrix of -div(k grad) from the moments of k. The gradient of a quadratic is linear on the element, so
//   A_lj = sum_{a,b} kappa_ab (grad phi_l at vertex a) . (grad phi_j at vertex b),  kappa_ab = sum_q w_q k_q lambda_a lambda_b,
// and with G_ab = |det J| grad lambda_a . grad lambda_b (the same for all micro-cells of a type in a cell) a row costs about
// 45 multiply-adds, against 110 for the sum over the 11 quadrature points, and reads 10 numbers per micro-cell and 10
// uniform ones instead of 11 and 110. At vertex b the gradient of vertex node a is (4 delta_ab - 1) grad lambda_a, that of
// edge node (a, b) is 4 grad lambda_b at vertex a and 4 grad lambda_a at vertex b.
constexpr int kP2Moments = 10;
__host__ __device__ constexpr int p2Mom( int a, int b ) // kappa_ab, a and b in any order
{
   const int i = a < b ? a : b, j = a < b ? b : a;
   return i * 4 - i * ( i + 1 ) / 2 + j;
}
// local number of the edge node between vertices a and b
__host__ __device__ constexpr int p2EdgeNode( int a, int b )
{
   for ( int e = 0; e < 6; ++e )
      if ( ( kP2EdgeNodes[e][0] == a && kP2EdgeNodes[e][1] == b ) || ( kP2EdgeNodes[e][0] == b && kP2EdgeNodes[e][1] == a ) )
         return 4 + e;
   return -1;
}
// row L of the element matrix: m the moments, g[p2Mom( a, b )] = G_ab
template < int L, typename T, typename GP >
__device__ __forceinline__ void p2Row( const T ( &m )[kP2Moments], GP g, T ( &r )[10] )
{
   T R[4];
#pragma unroll
   for ( int a = 0; a < 4; ++a )
      R[a] = ( m[p2Mom( a, 0 )] + m[p2Mom( a, 1 )] ) + ( m[p2Mom( a, 2 )] + m[p2Mom( a, 3 )] );
   if constexpr ( L < 4 )
   {
      const T K = ( R[0] + R[1] ) + ( R[2] + R[3] ), b0 = fma( T( -4 ), R[L], K );
      T       s[4]; // sum_b kappa_bc (4 delta_bL - 1)
#pragma unroll
      for ( int c = 0; c < 4; ++c )
      {
         s[c] = T( 4 ) * fma( T( 4 ), m[p2Mom( L, c )], -R[c] );
         r[c] = T( g[p2Mom( L, c )] ) * fma( T( 16 ), m[p2Mom( L, c )], fma( T( -4 ), R[c], b0 ) );
      }
#pragma unroll
      for ( int e = 0; e < 6; ++e )
      {
         const int c = kP2EdgeNodes[e][0], d = kP2EdgeNodes[e][1];
         r[4 + e]    = fma( T( g[p2Mom( L, c )] ), s[d], T( g[p2Mom( L, d )] ) * s[c] );
      }
   }
   else
   {
      constexpr int a = kP2EdgeNodes[L - 4][0], b = kP2EdgeNodes[L - 4][1];
      const T       Ra = T( 4 ) * R[a], Rb = T( 4 ) * R[b];
      T             ma[4], mb[4];
#pragma unroll
      for ( int c = 0; c < 4; ++c )
      {
         ma[c] = T( 16 ) * m[p2Mom( a, c )];
         mb[c] = T( 16 ) * m[p2Mom( b, c )];
         r[c]  = fma( T( g[p2Mom( c, b )] ), ma[c] - Ra, T( g[p2Mom( c, a )] ) * ( mb[c] - Rb ) );
      }
#pragma unroll
      for ( int e = 0; e < 6; ++e )
      {
         const int c = kP2EdgeNodes[e][0], d = kP2EdgeNodes[e][1];
         r[4 + e]    = fma( ma[c], T( g[p2Mom( b, d )] ),
                            fma( ma[d], T( g[p2Mom( b, c )] ), fma( mb[c], T( g[p2Mom( a, d )] ), mb[d] * T( g[p2Mom( a, c )] ) ) ) );
      }
   }
}
// the same with the node known at run time, uniform over the wave
template < typename T, typename GP >
__device__ __forceinline__ void p2RowOf( int l, const T ( &m )[kP2Moments], GP g, T ( &r )[10] )
{
   switch ( l )
   {
   case 0: p2Row< 0 >( m, g, r ); break;
   case 1: p2Row< 1 >( m, g, r ); break;
   case 2: p2Row< 2 >( m, g, r ); break;
   case 3: p2Row< 3 >( m, g, r ); break;
   case 4: p2Row< 4 >( m, g, r ); break;
   case 5: p2Row< 5 >( m, g, r ); break;
   case 6: p2Row< 6 >( m, g, r ); break;
   case 7: p2Row< 7 >( m, g, r ); break;
   case 8: p2Row< 8 >( m, g, r ); break;
   default: p2Row< 9 >( m, g, r ); break;
   }
}

// The micro-cells of a point of class cls: type, node, the node's offset from 2 * anchor and, per row j, the slot of node j in
// the point's stencil (p2StencilOffsets).
struct P2KQEntry
{
   int t = 0, l = 0, mcmax = 0, nd[3] = {}, slot[10] = {};
};
struct P2KQEntries
{
   int       n = 0;
   P2KQEntry e[kP2MaxPairs];
};
struct P2KQEntryTables
{
   P2KQEntries c[8];
};
constexpr P2KQEntryTables p2KQEntryTables()
{
   P2KQEntryTables tb;
   for ( int cls = 0; cls < 8; ++cls )
   {
      P2KQEntries&           L  = tb.c[cls];
      const P2StencilOffsets so = p2StencilOffsets( cls );
      for ( int t = 0; t < 6; ++t )
         for ( int l = 0; l < 10; ++l )
         {
            if ( p2NodeClass( t, l ) != cls )
               continue;
            P2KQEntry& e = L.e[L.n++];
            e.t          = t;
            e.mcmax      = p2CellMaxSum( t );
            e.l          = l;
            for ( int k = 0; k < 3; ++k )
               e.nd[k] = p2NodeOffset( t, l, k );
            for ( int jj = 0; jj < 10; ++jj )
               e.slot[jj] = p2OffsetIndex( so, p2NodeOffset( t, jj, 0 ) - e.nd[0], p2NodeOffset( t, jj, 1 ) - e.nd[1], p2NodeOffset( t, jj, 2 ) - e.nd[2] );
         }
   }
   return tb;
}
constexpr P2KQEntryTables           kP2Entries = p2KQEntryTables();
static __constant__ P2KQEntryTables kP2KQTab   = p2KQEntryTables();

// What a point of class CLS at (px, py, pz) of a cell gets from the stencil kernels of the variable coefficient: all points that
// are not on a cell edge. Interior points get the mode's epilogue, face points leave their one-sided sum in `part`.
// false: nothing; pi: position in the partial sums of a face point (slot > 0)
__device__ __forceinline__ bool p2PointWanted( int c, int N, int px, int py, int pz, const CellFaceSlot* __restrict__ cfs, int flag, int& slot,
                                               i64& pi )
{
   slot = classifySlot( N, px, py, pz );
   pi   = 0;
   if ( slot > 4 || ( slot == 0 && !( flag & 1 ) ) ) // cell edges and vertices: kP2KEdge
      return false;
   if ( slot == 0 )
      return true;
   const CellFaceSlot fs = cfs[4 * c + slot - 1];
   pi = i64( fs.block ) * ( N + 1 ) * ( N + 1 ) + facePartIndex( slot - 1, N, px, py, pz );
   return ( fs.bc & flag ) != 0;
}
// Which stencil nodes of a point lie in the cell (of a face point; an interior point has all): the offset's components against
// the distances to the four faces.
struct P2Inside
{
   bool lo[3][2], sum[2]; // x, y, z >= 1, 2; N - x - y - z >= 1, 2
   __device__ __forceinline__ P2Inside( int N, int px, int py, int pz )
   {
      const int b0 = N - px - py - pz;
      for ( int k = 0; k < 2; ++k )
      {
         lo[0][k] = px > k;
         lo[1][k] = py > k;
         lo[2][k] = pz > k;
         sum[k]   = b0 > k;
      }
   }
   // dx, dy, dz known at compile time
   __device__ __forceinline__ bool has( int dx, int dy, int dz ) const
   {
      const int d = dx + dy + dz;
      bool      in = true;
      if ( dx < 0 )
         in = in && lo[0][-dx - 1];
      if ( dy < 0 )
         in = in && lo[1][-dy - 1];
      if ( dz < 0 )
         in = in && lo[2][-dz - 1];
      if ( d > 0 )
         in = in && sum[d - 1];
      return in;
   }
};
// starts of the rows py + dy of the planes pz + dz (|dy|, |dz| <= 2) of a cell array, at px
__device__ __forceinline__ void p2RowStarts( int N, int px, int py, int pz, int ( &rb )[5][5] )
{
   const int w = N + 1;
#pragma unroll
   for ( int dz = -2; dz <= 2; ++dz )
   {
      const int Wz = w - ( pz + dz );
      const int pb = S3i( w ) - S3i( Wz );
#pragma unroll
      for ( int dy = -2; dy <= 2; ++dy )
         rb[dz + 2][dy + 2] = pb + rowStart( Wz, py + dy ) + px;
   }
}

// cell-interior and cell-face points of the variable-coefficient operator assembled on the fly (p2kq.hpp; defined for
// double and float in p2kq_f64.hip and p2kq_f32.hip)
template < typename T >
void launchP2KQPoints( int L, int nC, i64 stride, const T* el, const T* kq, i64 kqStride, const T* dinv, const P2Comps< T >& cp, int nc,
                       int mode, T a, const CellFaceSlot* cfs, int flag, T* part, i64 partStride, hipStream_t s );

} // namespace hyg
