// gfx950 kernels of the variable-coefficient P1 operator -div(k grad u), assembled element by element
// on the fly (the reference's P1ElementwiseOperator<p1_div_k_grad_affine_q3>,
// elementwiseoperators/P1ElementwiseOperator.cpp:64-301, forms/form_hyteg_generated/p1/
// p1_div_k_grad_affine_q3.cpp:179-381).
//
// On an affine micro-tetrahedron the gradients are constant, so the element matrix is
// kb_e * K_t: K_t is the element matrix of k = 1 for the micro-cell type t of the macro-cell (held in
// ElemCell::mt) and kb_e = 6 sum_q w_q k(x_q) is the 5-point degree-3 quadrature of k over the
// element divided by its volume (w = -2/15 at the centroid, 3/40 at the four points with barycentric
// coordinates (1/2, 1/6, 1/6, 1/6)). Each apply
//   1. evaluates kb_e for every micro-cell: the log-coefficient at the 30 quadrature points of the six cell types of a
//      lattice point is a matrix product of the modes' phase factors there with a constant matrix of their amplitudes
//      and offsets (kKBarTables, once per level at operator creation), with a thread per anchor (kKBarPoint) or on the
//      matrix cores (kKBar);
//   2. forms the product at every point of the closed cells, with a thread per point (kElemApply) or, on long rows, marching
//      over the cubes of the anchor lattice plane by plane (kElemSweep); interior points get the epilogue, points on
//      faces, edges and vertices store the cell's one-sided sum;
//   3. adds the one-sided sums of face, edge and vertex points over their cells and writes every
//      replica (kFaceCombine, kLowCombine).
// The inverse diagonal (per point, since it depends on k) is built the same way at operator setup.

#include "elementwise.hpp"

namespace hyg {

// ------------------------------------------------------------------ coefficient tables
// Tables of one level, built once. axis[c 3 N MP + b N MP + ..]: e^(i phase) of mode m at n lattice steps along axis b
// (axis 0: with the phase at the cell's vertex 0), at m N + n for axis 0 (lanes take consecutive n) and n MP + m for axes 1 and 2
// (lanes take the same n, modes follow each other); MP modes with zeros behind the nModes given; mat: the matrix of kKBar in
// the order in which its lanes hold it (step, tile, lane). Phases are reduced in turns before the sine is taken.
template < typename T >
__device__ void kbMatrix( const ElemCell& ec, const double* __restrict__ modes, int nModes, int i, T* __restrict__ mat )
{
   const int s = i >> 7, tile = ( i >> 6 ) & 1, lane = i & 63, k = 4 * s + ( lane >> 4 ), m = k >> 1;
   int       g, r;
   mmaRow( lane & 15, g, r, static_cast< T* >( nullptr ) );
   const int j = 4 * tile + r; // slot of the group
   const int t = j < 5 ? g : 4 + ( g >> 1 ), q = j < 5 ? j : ( ( g & 1 ) ? j - 2 : j - 5 );
   double    v = 0.0;
   if ( m < nModes && q < 5 )
   {
      double d[3] = { 0.0, 0.0, 0.0 }; // lattice offset of quadrature point q of type t from the anchor
      for ( int u = 0; u < 4; ++u )
      {
         const double lam = q == 0 ? 0.25 : ( u == q - 1 ? 0.5 : 1.0 / 6.0 );
         for ( int b = 0; b < 3; ++b )
            d[b] += lam * kMC[t][u][b];
      }
      double turns = 0.0;
      for ( int b = 0; b < 3; ++b )
         turns += d[b] * ( modes[5 * m] * ec.a[0][b] + modes[5 * m + 1] * ec.a[1][b] + modes[5 * m + 2] * ec.a[2][b] );
      double sn, cs;
      sincos( 2.0 * M_PI * turns, &sn, &cs );
      v = modes[5 * m + 4] * ( ( k & 1 ) ? -sn : cs );
   }
   mat[i] = T( v );
}
__global__ __launch_bounds__( kBlock ) void kKBarTables( const ElemCell* __restrict__ cells, const double* __restrict__ modes, int nModes,
                                                         int MP, int N, KbPair< double >* __restrict__ axis,
                                                         KbPair< float >* __restrict__ axisF, double* __restrict__ mat,
                                                         float* __restrict__ matF )
{
   const int       c  = int( blockIdx.x );
   const ElemCell& ec = cells[c];
   const int       i0 = int( blockIdx.y ) * kBlock + int( threadIdx.x ), step = int( gridDim.y ) * kBlock;
   for ( int i = i0; i < 3 * N * MP; i += step )
   {
      const int b = i / ( MP * N ), r = i - b * MP * N, m = b == 0 ? r / N : r % MP, n = b == 0 ? r % N : r / MP;
      double    cs = 0.0, sn = 0.0;
      if ( m < nModes )
      {
         const double kx = modes[5 * m], ky = modes[5 * m + 1], kz = modes[5 * m + 2];
         double       t  = n * ( kx * ec.a[0][b] + ky * ec.a[1][b] + kz * ec.a[2][b] );
         if ( b == 0 )
            t += kx * ec.v0[0] + ky * ec.v0[1] + kz * ec.v0[2];
         sincos( 2.0 * M_PI * ( t - rint( t ) ) + ( b == 0 ? modes[5 * m + 3] : 0.0 ), &sn, &cs );
      }
      const i64 o = i64( c ) * 3 * N * MP + i;
      axis[o]     = { cs, sn };
      axisF[o]    = { float( cs ), float( sn ) };
   }
   for ( int i = i0; i < MP * 64; i += step )
   {
      kbMatrix( ec, modes, nModes, i, mat + i64( c ) * MP * 64 );
      kbMatrix( ec, modes, nModes, i, matF + i64( c ) * MP * 64 );
   }
}

// ------------------------------------------------------------------ launch
// Coefficient integrals by matrix products (kKBar) or a thread per anchor (kKBarPoint)? The products are paid for 8, 32 or 64 modes
// and for tiles of 16 anchors of a row, a thread for the modes there are, one after the other. Apply with n modes, thread / products,
// us. Long rows, level 7 on 24 cells: FP32 n = 24 592 / 632, 28 652 / 634, 32 713 / 634, 64 1206 / 1579 (6 cells 168 / 189, 183 / 189,
// 199 / 189); FP64 32 1103 / 1232, 16 788 / 1225. Shorter rows: level 6 on 24 cells FP32 32 125 / 131, level 5 on 240 cells FP64 32
// 226 / 338, level 4 on 960 cells 174 / 312. Few anchors, where a thread's chain of modes is the whole time, FP64: level 3 on 24 cells
// n = 4 17.7 / 17.0, 12 20.5 / 20.0, 24 24.7 / 19.9, 64 39.1 / 25.9; level 4 on 24 cells 24 26.0 / 26.7, 32 28.9 / 26.8; level 4 on 48
// cells 32 29.5 / 31.5; level 3 on 162 cells 32 29.1 / 33.6; level 2 on 162 cells 24 26.1 / 23.1, 33 29.6 / 39.7.
static bool kbOnMatrixCores( int n, int L, int nC, int dtype )
{
   if ( L >= 7 )
      return dtype == 4 && n > 26 && n <= 32;
   const i64 rows = ( i64( nC ) << L ) * ( ( 1 << L ) + 1 ) / 2; // of anchors
   if ( L == 4 )
      return rows <= 3300 && n > 24 && n <= 32;
   return L <= 3 && n >= 3 && ( n <= 8 || n > 12 || L <= 2 ) && rows <= ( n <= 32 ? 1800 : 900 );
}

template < typename T >
static void launchKBar( const hyg_op_s& op, int L, int nC, T* kb, hipStream_t s )
{
   constexpr bool         dbl = std::is_same< T, double >::value;
   const hyg_op_s::Level& ol  = op.levels[L];
   const int              N   = 1 << L;
   if ( op.kPolyDeg >= 0 )
   {
      const int tK = ceilDiv( S3i( N ), kBlock );
      hipLaunchKernelGGL( ( kKBarPoly< T > ), dim3( nC * tK ), dim3( kBlock ), 0, s, L, tK, ol.elem, op.kPoly, op.kPolyDeg, kb );
      return;
   }
   const auto* axis = static_cast< const KbPair< T >* >( dbl ? ol.kbAxis : ol.kbAxisF );
   const T*    mat  = dbl ? (const T*) ol.kbMat : (const T*) ol.kbMatF;
   if ( !kbOnMatrixCores( op.nModes, L, nC, dbl ? 8 : 4 ) )
   {
      const int tK = ceilDiv( S3i( N ), kBlock );
      hipLaunchKernelGGL( ( kKBarPoint< T > ), dim3( nC * tK ), dim3( kBlock ), 0, s, N, tK, op.nModes, kbModes( op.nModes ), axis, mat,
                          T( op.k0 ), kb );
      return;
   }
   const int rows   = nC * N * ceilDiv( N, kKBarRows ) >= 2048 ? kKBarRows : 16; // 2048: four blocks per CU and half of them empty
   const int chunks = ceilDiv( N, rows );
   auto      kf     = kKBar< T, 32 >;
   switch ( kbModes( op.nModes ) )
   {
   case 8: kf = kKBar< T, 4 >; break;
   case 32: kf = kKBar< T, 16 >; break;
   default: break;
   }
   hipLaunchKernelGGL( kf, dim3( nC * N * chunks ), dim3( kBlock ), 0, s, N, nC, rows, axis, mat, T( op.k0 ), kb );
}

// per-level tables of the Fourier coefficient, once at operator setup
void launchKBarTables( const MeshCtx& m, const hyg_op_s& op, int L, hipStream_t s )
{
   const hyg_op_s::Level& ol = op.levels[L];
   if ( op.kPolyDeg >= 0 || !ol.kbAxis )
      return;
   const int N = 1 << L, MP = kbModes( op.nModes );
   hipLaunchKernelGGL( kKBarTables, dim3( m.mesh->nC(), std::min( 16, ceilDiv( 3 * N * MP, kBlock ) ) ), dim3( kBlock ), 0, s, ol.elem,
                       op.modes, op.nModes, MP, N, static_cast< KbPair< double >* >( ol.kbAxis ),
                       static_cast< KbPair< float >* >( ol.kbAxisF ), ol.kbMat, ol.kbMatF );
}

// coefficient integrals of every level in both value types, kept for the applies that follow
void launchElementwiseStore( const MeshCtx& m, hyg_op_s& op, hipStream_t s )
{
   for ( int L = op.minL; L <= op.maxL; ++L )
   {
      launchKBar< double >( op, L, m.mesh->nC(), op.levels[L].kb, s );
      launchKBar< float >( op, L, m.mesh->nC(), op.levels[L].kbF, s );
   }
   op.stored = true;
}

template < typename T, int MODE, bool DIAG >
static void elemT( const MeshCtx& m, LevelGeom& g, const hyg_op_s& op, int L, const StencilCall& c, hipStream_t s )
{
   constexpr bool             dbl = std::is_same< T, double >::value;
   const hyg_op_s::Level&     ol  = op.levels[L];
   const int                  nC  = m.mesh->nC();
   const int                  N   = 1 << L, w = N + 1;
   T*                         kb  = dbl ? (T*) ol.kb : (T*) ol.kbF;
   T*                         part = dbl ? (T*) ol.facePart : (T*) ol.facePartF;
   T*                         low  = dbl ? (T*) ol.lowPart : (T*) ol.lowPartF;
   const T*                   dv   = DIAG ? nullptr : ( dbl ? (const T*) ol.dinv : (const T*) ol.dinvF );
   const T*                   x    = (const T*) c.x;
   const T*                   in1  = (const T*) c.in1;
   T*                         out0 = (T*) c.out0;
   T*                         out1 = (T*) c.out1;
   // 1. coefficient integrals of all micro-cells (kept from hyg_op_store_local_matrices when stored)
   if ( !op.stored )
      launchKBar< T >( op, L, nC, kb, s );
   // 2. per-cell stencils (interior results, one-sided sums of face, edge and vertex points); the surrogate operator
   //    does its interior points with the polynomial stencils
   const int tA = ceilDiv( S3i( w ), kBlock );
   if ( !DIAG && surrogateActive( op, L ) )
   {
      const int tB = ceilDiv( ol.surNBnd, kBlock );
      hipLaunchKernelGGL( ( kElemApply< T, MODE, DIAG, true > ), dim3( nC * tB ), dim3( kBlock ), 0, s, L, tB, g.stride, ol.elem, kb,
                          m.cellInfo, m.cellFaces, m.prims, m.entries, part, low, dv, c.flag, x, in1, out0, out1, T( c.a ), ol.surBnd,
                          ol.surNBnd );
      launchSurrogateInterior( m, g, op, L, std::is_same< T, double >::value ? 8 : 4, c, s );
   }
   else if ( op.blend )
      hipLaunchKernelGGL( ( kElemApply< T, MODE, DIAG, false, true > ), dim3( xcdGrid( nC * tA ) ), dim3( kBlock ), 0, s, L, tA, g.stride,
                          ol.elem, kb, m.cellInfo, m.cellFaces, m.prims, m.entries, part, low, dv, c.flag, x, in1, out0, out1, T( c.a ),
                          nullptr, 0, dbl ? (const T*) ol.bw : (const T*) ol.bwF, nC * tA );
   else if ( DIAG || !elemMarches( L, nC, dbl ? 8 : 4 ) )
      hipLaunchKernelGGL( ( kElemApply< T, MODE, DIAG > ), dim3( xcdGrid( nC * tA ) ), dim3( kBlock ), 0, s, L, tA, g.stride, ol.elem, kb,
                          m.cellInfo, m.cellFaces, m.prims, m.entries, part, low, dv, c.flag, x, in1, out0, out1, T( c.a ), nullptr, 0,
                          nullptr, nC * tA );
   else
   {
      const ElemArgs< T > e = elemArgs< T >( m, g, ol, L, c );
      hipLaunchKernelGGL( ( kElemSweep< T, MODE > ), dim3( elemBlocks( e ) ), dim3( kBlock ), 0, s, e );
   }
   // 3. face, edge and vertex values
   const int nLow = g.firstFaceChunk, nFace = g.nChunks - g.firstFaceChunk;
   if ( nFace > 0 )
      hipLaunchKernelGGL( ( kFaceCombine< T, MODE > ), dim3( xcdGrid( ceilDiv( nFace, kBlock / 64 ) ) ), dim3( kBlock ), 0, s,
                          g.chunks + g.firstFaceChunk, nFace, m.entries, m.mesh->nV() + m.mesh->nE(), part, (const T*) nullptr,
                          dv, L, g.stride, c.flag, x, in1, out0, out1, T( c.a ) );
   if ( nLow > 0 )
      hipLaunchKernelGGL( ( kLowCombine< T, MODE > ), dim3( ceilDiv( nLow, kBlock / 64 ) ), dim3( kBlock ), 0, s, g.chunks, nLow,
                          m.entries, low, dv, L, g.stride, c.flag, x, in1, out0, out1, T( c.a ) );
}

template < typename T >
static void elemMode( const MeshCtx& m, LevelGeom& g, const hyg_op_s& op, int L, const StencilCall& c, hipStream_t s )
{
   switch ( c.mode )
   {
   case MODE_APPLY:
      elemT< T, MODE_APPLY, false >( m, g, op, L, c, s );
      break;
   case MODE_APPLY_ADD:
      elemT< T, MODE_APPLY_ADD, false >( m, g, op, L, c, s );
      break;
   case MODE_RESIDUAL:
      elemT< T, MODE_RESIDUAL, false >( m, g, op, L, c, s );
      break;
   case MODE_JACOBI:
      elemT< T, MODE_JACOBI, false >( m, g, op, L, c, s );
      break;
   case MODE_CHEB0:
      elemT< T, MODE_CHEB0, false >( m, g, op, L, c, s );
      break;
   default:
      elemT< T, MODE_CHEBK, false >( m, g, op, L, c, s );
      break;
   }
}

void launchElementwise( const MeshCtx& m, LevelGeom& g, const hyg_op_s& op, int L, int dtype, const StencilCall& c, hipStream_t s )
{
   if ( dtype == 8 )
      elemMode< double >( m, g, op, L, c, s );
   else
      elemMode< float >( m, g, op, L, c, s );
}

void launchElementwiseInverseDiagonal( const MeshCtx& m, LevelGeom& g, const hyg_op_s& op, int L, hipStream_t s )
{
   // the coefficient tables of the level (called once per level when the operator is created)
   launchKBarTables( m, op, L, s );
   const hyg_op_s::Level& ol = op.levels[L];
   const i64              n  = i64( m.mesh->nC() ) * g.stride + kTailSlack;
   (void) hipMemsetAsync( ol.dinv, 0, size_t( n ) * sizeof( double ), s );
   StencilCall c;
   c.mode = MODE_APPLY;
   c.flag = 15;
   c.out0 = ol.dinv;
   elemT< double, MODE_APPLY, true >( m, g, op, L, c, s );
   hipLaunchKernelGGL( ( kInvertAll< double > ), dim3( 1024 ), dim3( kBlock ), 0, s, n, ol.dinv );
   if ( surrogateActive( op, L ) )
      launchSurrogateInverseDiagonal( m, g, op, L, s );
   launchConvert( n, 4, ol.dinvF, 8, ol.dinv, s );
}

} // namespace hyg
