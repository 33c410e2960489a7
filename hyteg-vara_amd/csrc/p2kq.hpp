// On-the-fly variable-coefficient P2 kernels (P2ElementwiseOperator< p2_div_k_grad_affine_q4 >,
// P2ElementwiseOperator.cpp:100-310): cell-interior and cell-face points. Compiled once per value type
// (p2kq_f64.hip, p2kq_f32.hip).
#pragma once
#include "p2_common.hpp"

namespace hyg {

// ------------------------------------------------------------------ variable coefficient, assembled on the fly
// The stencil of a point is assembled in registers from the rows of its micro-cells (p2Row; the slots of the ten nodes are
// known at compile time) and then applied to up to three components, so a vector function's components share it. A
// micro-cell's moments are 10 loads of consecutive values by consecutive threads, each value of the 65 (vertex class), 27 or
// 19 points of the stencil is loaded once. A micro-cell at a time: the branch around it (a face point takes those inside the
// cell) keeps the loads of one from being hoisted above another's (branch-free, with zero moments outside the cell, the
// compiler kept the loads of all 24 micro-cells of a vertex point in flight and spilled 400 registers).
// Three components on the shell (960 cells, P2 level 4, 3 x 5.2 million points, FP64): the two launches 960 us, against 1868
// us with rows of 11-point sums read from LDS (110 multiply-adds and 55 LDS reads per row, a load per node and micro-cell).
// Per point 75 loads of moments and 29 per component of values remain; the vertex class (1/8 of the points, 24 micro-cells each)
// takes 420 us of it at two waves per SIMD.
template < typename T, int CLS, int K >
__device__ __forceinline__ void p2AddRow( int c, int Nc, int SA, int px, int py, int pz, const T* __restrict__ kq, i64 kqStride,
                                          const T* __restrict__ g, T ( &W )[p2StencilOffsets( CLS ).n] )
{
   typedef const T __attribute__( ( address_space( 4 ) ) ) CT;
   constexpr P2KQEntry e  = kP2Entries.c[CLS].e[K];
   const int           ax = ( px - e.nd[0] ) >> 1, ay = ( py - e.nd[1] ) >> 1, az = ( pz - e.nd[2] ) >> 1;
   if ( ax >= 0 && ay >= 0 && az >= 0 && ax + ay + az + e.mcmax <= Nc )
   {
      const T*       kv = kq + i64( c * 6 + e.t ) * SA;
      const unsigned o  = unsigned( cidx( Nc + 1, ax, ay, az ) );
      T              m[kP2Moments], r[10];
#pragma unroll
      for ( int q = 0; q < kP2Moments; ++q )
         m[q] = ( kv + i64( q ) * kqStride )[o];
      p2Row< e.l >( m, (CT*) ( g + ( c * 6 + e.t ) * kP2Moments ), r );
#pragma unroll
      for ( int j = 0; j < 10; ++j )
         W[e.slot[j]] += r[j];
   }
}
template < typename T, int CLS, int... K >
__device__ __forceinline__ void p2Assemble( int c, int Nc, int px, int py, int pz, const T* __restrict__ kq, i64 kqStride,
                                            const T* __restrict__ g, T ( &W )[p2StencilOffsets( CLS ).n], std::integer_sequence< int, K... > )
{
   const int SA = S3i( Nc + 1 );
   ( p2AddRow< T, CLS, K >( c, Nc, SA, px, py, pz, kq, kqStride, g, W ), ... );
}
template < typename T >
__device__ __forceinline__ void p2EmitInterior( int mode, int nc, const T ( &val )[3], i64 q, const P2Comps< T >& cp,
                                                const T* __restrict__ dinv, T a )
{
#pragma unroll
   for ( int k = 0; k < 3; ++k )
   {
      if ( k >= nc )
         break;
      T r0 = T( 0 ), r1 = T( 0 );
      switch ( mode )
      {
      case MODE_APPLY: epilogue< T, MODE_APPLY >( val[k], T( 0 ), T( 0 ), T( 0 ), T( 1 ), a, r0, r1 ); break;
      case MODE_APPLY_ADD:
      {
         const T o = cp.out0[k][q];
         epilogue< T, MODE_APPLY_ADD >( val[k], T( 0 ), o, o, T( 1 ), a, r0, r1 );
         break;
      }
      case MODE_RESIDUAL:
      {
         const T i1 = cp.in1[k][q];
         epilogue< T, MODE_RESIDUAL >( val[k], T( 0 ), i1, i1, T( 1 ), a, r0, r1 );
         break;
      }
      case MODE_JACOBI:
      {
         const T i1 = cp.in1[k][q];
         epilogue< T, MODE_JACOBI >( val[k], cp.x[k][q], i1, i1, dinv[q], a, r0, r1 );
         break;
      }
      case MODE_CHEB0:
      {
         const T i1 = cp.in1[k][q];
         epilogue< T, MODE_CHEB0 >( val[k], cp.x[k][q], i1, i1, dinv[q], a, r0, r1 );
         break;
      }
      default:
      {
         const T i1 = cp.in1[k][q];
         epilogue< T, MODE_CHEBK >( val[k], cp.x[k][q], i1, i1, dinv[q], a, r0, r1 );
         break;
      }
      }
      cp.out0[k][q] = r0;
      if ( mode == MODE_CHEB0 || mode == MODE_CHEBK )
         cp.out1[k][q] = r1;
   }
}
// All points of class CLS of a cell that are not on a cell edge: the class sub-lattice {2 q + kappa : 2 |q| + |kappa| <= N}
// (p2ClassExtent), so the points on the x = 0 and diagonal faces sit in the waves of their rows' interior points and
// are read and written with them. Interior points get the mode's epilogue, face points store their one-sided sums.
template < typename T, int CLS >
__device__ __forceinline__ void p2KQIntPt( int c, int s, int N, i64 stride, const T* __restrict__ el, const T* __restrict__ kq,
                                           i64 kqStride, const T* __restrict__ dinv, const P2Comps< T >& cp, int nc, int mode, T a,
                                           const CellFaceSlot* __restrict__ cfs, int flag, T* __restrict__ part, i64 partStride )
{
   constexpr int              kx = CLS & 1, ky = ( CLS >> 1 ) & 1, kz = ( CLS >> 2 ) & 1;
   constexpr P2StencilOffsets off = p2StencilOffsets( CLS );
   const int                  M   = p2ClassExtent( N, CLS );
   if ( s >= S3i( M + 1 ) )
      return;
   int qx, qy, qz;
   tetXYZ( M + 1, s, qx, qy, qz );
   const int px = 2 * qx + kx, py = 2 * qy + ky, pz = 2 * qz + kz;
   int       slot;
   i64       pi;
   if ( !p2PointWanted( c, N, px, py, pz, cfs, flag, slot, pi ) )
      return;
   T W[off.n];
#pragma unroll
   for ( int e = 0; e < off.n; ++e )
      W[e] = T( 0 );
   p2Assemble< T, CLS >( c, N >> 1, px, py, pz, kq, kqStride, el, W, std::make_integer_sequence< int, kP2Entries.c[CLS].n >() );
   int rb[5][5];
   p2RowStarts( N, px, py, pz, rb );
   const i64 cb     = i64( c ) * stride;
   const int q      = rb[2][2];
   const P2Inside in( N, px, py, pz );
   T          val[3] = { T( 0 ), T( 0 ), T( 0 ) };
#pragma unroll
   for ( int e = 0; e < off.n; ++e )
   {
      // a node outside the cell has no weight
      const int o = in.has( off.d[e][0], off.d[e][1], off.d[e][2] ) ? rb[off.d[e][2] + 2][off.d[e][1] + 2] + off.d[e][0] : zeroValue( N );
      // explicit fused multiply-adds: every component (and the single-component pass) rounds alike
      val[0] = fma( W[e], ( cp.x[0] + cb )[unsigned( o )], val[0] );
      if ( nc > 1 )
      {
         val[1] = fma( W[e], ( cp.x[1] + cb )[unsigned( o )], val[1] );
         val[2] = fma( W[e], ( cp.x[2] + cb )[unsigned( o )], val[2] );
      }
   }
   if ( slot == 0 )
      p2EmitInterior< T >( mode, nc, val, cb + q, cp, dinv, a );
   else
   {
#pragma unroll
      for ( int k = 0; k < 3; ++k )
      {
         if ( k >= nc )
            break;
         part[i64( k ) * partStride + pi] = val[k];
      }
   }
}
template < typename T, int CLS >
__device__ __forceinline__ void p2KQIntDispatch( int cls, int c, int s, int N, i64 stride, const T* el, const T* kq, i64 kqStride,
                                                 const T* dinv, const P2Comps< T >& cp, int nc, int mode, T a, const CellFaceSlot* cfs,
                                                 int flag, T* part, i64 partStride )
{
   if ( cls == CLS )
      p2KQIntPt< T, CLS >( c, s, N, stride, el, kq, kqStride, dinv, cp, nc, mode, a, cfs, flag, part, partStride );
   else if constexpr ( CLS < 7 )
      p2KQIntDispatch< T, CLS + 1 >( cls, c, s, N, stride, el, kq, kqStride, dinv, cp, nc, mode, a, cfs, flag, part, partStride );
}
// VERTEX: the points of class 0, whose 65-point stencil needs twice the registers of the other classes; else classes 1..7
template < typename T, bool VERTEX >
__global__ __launch_bounds__( kBlock, VERTEX ? 2 : 4 ) void kP2KQInt( int L, i64 stride, P2ClassTiles ct, const T* __restrict__ el,
                                                      const T* __restrict__ kq, i64 kqStride, const T* __restrict__ dinv,
                                                      P2Comps< T > cp, int nc, int mode, T a, const CellFaceSlot* __restrict__ cfs,
                                                      int flag, T* __restrict__ part, i64 partStride, int nC )
{
   const int t0 = VERTEX ? 0 : ct.start[1], per = ( VERTEX ? ct.start[1] : ct.start[8] ) - t0;
   // each XCD takes a contiguous range of cells (the hardware deals workgroups out round-robin over the 8 XCDs), so
   // a cell's coefficient values and source stay in one XCD's L2 while its class blocks run
   const int b = remapXcd( int( blockIdx.x ), nC * per );
   if ( b >= nC * per ) // the whole block (grid padded to a multiple of 8)
      return;
   const int c = b / per;
   const int t = t0 + b - c * per;
   if constexpr ( VERTEX )
      p2KQIntPt< T, 0 >( c, t * kBlock + int( threadIdx.x ), 1 << L, stride, el, kq, kqStride, dinv, cp, nc, mode, a, cfs, flag, part,
                         partStride );
   else
   {
      int cls = 1;
      while ( cls < 7 && t >= ct.start[cls + 1] )
         ++cls;
      p2KQIntDispatch< T, 1 >( cls, c, ( t - ct.start[cls] ) * kBlock + int( threadIdx.x ), 1 << L, stride, el, kq, kqStride, dinv, cp, nc,
                               mode, a, cfs, flag, part, partStride );
   }
}
template < typename T >
void launchP2KQPoints( int L, int nC, i64 stride, const T* el, const T* kq, i64 kqStride, const T* dinv, const P2Comps< T >& cp, int nc,
                       int mode, T a, const CellFaceSlot* cfs, int flag, T* part, i64 partStride, hipStream_t s )
{
   const P2ClassTiles ct = p2ClassTiles( 1 << L );
   if ( ct.start[1] > 0 )
      hipLaunchKernelGGL( ( kP2KQInt< T, true > ), dim3( xcdGrid( nC * ct.start[1] ) ), dim3( kBlock ), 0, s, L, stride, ct, el, kq, kqStride,
                          dinv, cp, nc, mode, a, cfs, flag, part, partStride, nC );
   if ( ct.start[8] > ct.start[1] )
      hipLaunchKernelGGL( ( kP2KQInt< T, false > ), dim3( xcdGrid( nC * ( ct.start[8] - ct.start[1] ) ) ), dim3( kBlock ), 0, s, L, stride, ct,
                          el, kq, kqStride, dinv, cp, nc, mode, a, cfs, flag, part, partStride, nC );
}

} // namespace hyg
