// Shared by the cell-tiled kernels (one spline order per translation unit,
// CA_ORDER set on the compile line): bricks of mesh cells, their part tables
// and particle runs, node windows, the launch.
//
// Bricks of mesh cells are cut into parts of bounded particle count (a part
// table built on the device before the launch), and each workgroup walks
// parts from an XCD-local range of that table, so dense clusters are spread
// over every CU and empty bricks cost nothing.  A brick's particles are its
// cell runs along the last dimension (contiguous in the cell-sorted order),
// walked through a flattened index so consecutive lanes read consecutive
// particles.
#pragma once
#include "ca_device.hpp"

#include <utility>

#ifndef CA_ORDER
#error "CA_ORDER must be defined"
#endif

#define CA_CAT2( a, b ) a##b
#define CA_CAT( a, b ) CA_CAT2( a, b )
#define CA_SUFFIX CA_CAT( o, CA_ORDER )

namespace cabana_amd
{
namespace
{

constexpr int ORDER = CA_ORDER;
constexpr int K = ORDER + 1;
constexpr int BLOCK = 256;
// Stencil base node of a particle in cell c (ghosted node index):
// c + halo + BASE_SHIFT + {0, 1 if ORDER == 2}.
constexpr int BASE_SHIFT = ( ORDER == 1 ) ? 0 : -1;
template <int... FORMS>
struct FormList
{
    static constexpr int N = sizeof...( FORMS );
    static constexpr int v[N] = { FORMS... };
};

constexpr int ng_of( int form )
{
    return ( form == FORM_SV || form == FORM_VD ) ? 1 : 3;
}
constexpr int np_of( int form )
{
    return ( form == FORM_SV || form == FORM_SG )
               ? 1
               : ( ( form == FORM_VV || form == FORM_VD ) ? 3 : 9 );
}
__device__ __forceinline__ size_t align16( size_t b )
{
    return ( b + 15 ) & ~(size_t)15;
}

struct TileGeom
{
    int brick;
    int part;
    int c0[3];
    int c1[3];
};

// The parts of this workgroup.  Runs of up to 32 consecutive parts of the
// table (at least eight runs for each XCD) are dealt to the XCDs in turn
// (workgroups are dealt round-robin to them), so neighbouring bricks share an
// L2 and crowded regions, whose parts are the full ones, spread over all XCDs:
// with one contiguous eighth of the table for each, the FP64 adjoint gather of
// 101 x 64 x 77 cells x 10 took 0.87 ms, with runs 0.64 ms.  The workgroups of
// one XCD stride through its runs.  Every workgroup leaves the loop at the end
// of the table.
struct PartLoop
{
    int total;
    int shift;
    int xcd;
    int first;
    int stride;
    __device__ explicit PartLoop( const TileArgs& ta )
    {
        total = *ta.num_parts;
        shift = min( 5, 31 - __clz( max( total >> 6, 1 ) ) );
        xcd = blockIdx.x & 7;
        first = blockIdx.x >> 3;
        stride = gridDim.x >> 3;
    }
    __device__ bool more( int loc ) const { return ( loc >> shift ) << ( shift + 3 ) < total; }
    // Table entry of the loop's position, -1 past the end of the table.
    __device__ int part( int loc ) const
    {
        const int w = ( ( ( loc >> shift ) * 8 + xcd ) << shift ) + ( loc & ( ( 1 << shift ) - 1 ) );
        return w < total ? w : -1;
    }
};

__device__ __forceinline__ void part_geometry_of( const TileArgs& ta, const MeshDev& m,
                                                  int2 pr, TileGeom& g )
{
    g.brick = pr.x;
    g.part = pr.y;
    const int ti = g.brick / ( ta.ntile[1] * ta.ntile[2] );
    const int tj = ( g.brick / ta.ntile[2] ) % ta.ntile[1];
    const int tk = g.brick % ta.ntile[2];
    g.c0[0] = ti * ta.tile[0];
    g.c0[1] = tj * ta.tile[1];
    g.c0[2] = tk * ta.tile[2];
#pragma unroll
    for ( int d = 0; d < 3; ++d )
        g.c1[d] = min( g.c0[d] + ta.tile[d], m.num_cell[d] );
}

__device__ __forceinline__ void part_geometry( const TileArgs& ta, const MeshDev& m,
                                               int w, TileGeom& g )
{
    part_geometry_of( ta, m, ta.parts[w], g );
}

// Fills the run table of the brick (one run per (i, j) cell row) and returns
// the number of particles.  run_pre has nruns + 1 entries.
__device__ __forceinline__ int setup_runs( const TileArgs& ta,
                                           const MeshDev& m,
                                           const TileGeom& g,
                                           int64_t* run_start, int* run_pre )
{
    const int nj = g.c1[1] - g.c0[1];
    const int nruns = ( g.c1[0] - g.c0[0] ) * nj;
    for ( int r = threadIdx.x; r < nruns; r += BLOCK )
    {
        const int ci = g.c0[0] + r / nj, cj = g.c0[1] + r % nj;
        const int64_t cfirst =
            ( (int64_t)ci * m.num_cell[1] + cj ) * m.num_cell[2] + g.c0[2];
        const int64_t clast = cfirst + ( g.c1[2] - g.c0[2] ) - 1;
        const int64_t st = ta.cell_offsets[cfirst];
        run_start[r] = st;
        run_pre[r + 1] = (int)( ta.cell_offsets[clast] + ta.cell_counts[clast] - st );
    }
    __syncthreads();
    if ( threadIdx.x == 0 )
    {
        run_pre[0] = 0;
        for ( int r = 0; r < nruns; ++r )
            run_pre[r + 1] += run_pre[r];
    }
    __syncthreads();
    return run_pre[nruns];
}

// Run containing flattened brick position v (binary search).
__device__ __forceinline__ int find_run( const int* run_pre, int nruns, int v )
{
    int lo = 0, hi = nruns - 1;
    while ( lo < hi )
    {
        const int mid = ( lo + hi + 1 ) >> 1;
        if ( run_pre[mid] <= v )
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// floor(a / b) for 0 <= a < 2^22 and b >= 1 from a rounded reciprocal rb of
// b: (a + 1/2) / b lies at least 1/(2b) from an integer, and the two
// roundings move it by at most (a + 1/2) / b * 2^-23 < 1/(2b).
__device__ __forceinline__ int div_small( int a, float rb )
{
    return (int)( ( (float)a + 0.5f ) * rb );
}

// Maps a flat window index to (node, dof) with the grid's unit-stride
// dimension fastest, so window loads/stores coalesce.  rW holds the
// reciprocals of the window extents (window indices stay below 2^22).
template <int NG>
__device__ __forceinline__ void window_coords( const TileArgs& ta, int f, const int W[3],
                                               const float rW[3], int q[3], int& d )
{
    const int pa = ta.flush_perm[0], pb = ta.flush_perm[1],
              pc = ta.flush_perm[2];
    const int node = f / NG;
    d = f - node * NG;
    const int r = div_small( node, rW[pc] );
    q[pc] = node - r * W[pc];
    q[pa] = div_small( r, rW[pb] );
    q[pb] = r - q[pa] * W[pb];
}

template <class KernelPtr, class Args>
hipError_t launch_tile_kernel( KernelPtr k, const Args& a, const TileArgs& t,
                               size_t lds, hipStream_t s, int block = BLOCK )
{
    if ( lds > 64 * 1024 )
    {
        hipError_t e = hipFuncSetAttribute(
            reinterpret_cast<const void*>( k ),
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds );
        if ( e != hipSuccess )
            return e;
    }
    hipLaunchKernelGGL( k, dim3( (unsigned)t.grid ), dim3( block ), lds, s, a, t );
    return hipGetLastError();
}

} // namespace
} // namespace cabana_amd
