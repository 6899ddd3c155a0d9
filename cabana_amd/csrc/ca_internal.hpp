// Internal types shared by the C-ABI layer and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/cabana_amd.h"

namespace cabana_amd
{

// Mesh constants as the kernels see them.  low/rdx follow evaluateSpline
// (Cabana_Grid_Splines.hpp:1283-1342): low = coordinate of ghosted node 0,
// dx = coordinate(node 1) - coordinate(node 0), rdx = 1 / dx.
struct MeshDev
{
    double low[3];
    double rdx[3];
    int32_t num_node[3]; // ghosted node extent
    int32_t num_cell[3];
    int32_t halo;        // halo cell width of the local grid
    int32_t periodic[3];
    int32_t stag[3];     // 1 where the arrays' entity sits at cell centres
};

// Particle field addressing (Cabana_Slice.hpp:119-190).  For a power-of-two
// vector length the block and lane come from shift/mask; when one block holds
// every particle, shift = 62 so the block index is always 0.
// Particle field (Cabana slice addressing, Cabana_Slice.hpp:119-190):
// element (p, c) at data[(p / vl) * stride + p % vl + vl * c].  The vector
// length is a power of two (as every Cabana AoSoA's) or covers all particles,
// so the index is a shift and a mask; every element index of the field fits
// in 32 bits.  Both are checked on the host; device addressing is 32-bit
// integer math plus one 64-bit pointer add, with no branches.
struct PFieldDev
{
    char* data;
    uint32_t vl;
    uint32_t stride;
    int32_t shift;
    int32_t ncomp;
    uint32_t mask;

    __device__ __forceinline__ uint32_t base( int64_t p64 ) const
    {
        const uint32_t p = (uint32_t)p64;
        return ( p >> shift ) * stride + ( p & mask );
    }
    // base( p ) of a field with vector_length 1.
    __device__ __forceinline__ uint32_t row( int64_t p ) const { return (uint32_t)p * stride; }
    template <class T>
    __device__ __forceinline__ T* ptr( uint32_t b, int c ) const
    {
        return reinterpret_cast<T*>( data + (uint64_t)( b + vl * (uint32_t)c ) * sizeof( T ) );
    }
    // Components [0, N) of particle p.  CONTIG (vector_length 1, checked
    // by the caller's host code) moves them as 16/8-byte vectors (4-byte
    // aligned access), one instruction per 16 bytes instead of one per
    // component; otherwise (AoSoA) each component is its own access,
    // coalesced across lanes.
    template <class T, int N, bool CONTIG = false>
    __device__ __forceinline__ void load( int64_t p, T* v ) const;
    template <class T, int N, bool CONTIG = false>
    __device__ __forceinline__ void store( int64_t p, const T* v ) const;
};

namespace detail
{
template <class T, int W>
struct VecOf;
template <>
struct VecOf<float, 4>
{
    typedef float type __attribute__( ( ext_vector_type( 4 ), aligned( 4 ) ) );
};
template <>
struct VecOf<float, 2>
{
    typedef float type __attribute__( ( ext_vector_type( 2 ), aligned( 4 ) ) );
};
template <>
struct VecOf<double, 2>
{
    typedef double type __attribute__( ( ext_vector_type( 2 ), aligned( 8 ) ) );
};

template <class T, int N>
__device__ __forceinline__ void vec_copy_in( const T* src, T* dst )
{
    constexpr int W = 16 / (int)sizeof( T );
    int i = 0;
#pragma unroll
    for ( ; i + W <= N; i += W )
    {
        const typename VecOf<T, W>::type x = *reinterpret_cast<const typename VecOf<T, W>::type*>( src + i );
#pragma unroll
        for ( int e = 0; e < W; ++e )
            dst[i + e] = x[e];
    }
    if constexpr ( W == 4 && N % 4 >= 2 )
    {
        const typename VecOf<T, 2>::type x = *reinterpret_cast<const typename VecOf<T, 2>::type*>( src + i );
        dst[i] = x[0];
        dst[i + 1] = x[1];
        i += 2;
    }
#pragma unroll
    for ( ; i < N; ++i )
        dst[i] = src[i];
}

template <class T, int N>
__device__ __forceinline__ void vec_copy_out( const T* src, T* dst )
{
    constexpr int W = 16 / (int)sizeof( T );
    int i = 0;
#pragma unroll
    for ( ; i + W <= N; i += W )
    {
        typename VecOf<T, W>::type x;
#pragma unroll
        for ( int e = 0; e < W; ++e )
            x[e] = src[i + e];
        *reinterpret_cast<typename VecOf<T, W>::type*>( dst + i ) = x;
    }
    if constexpr ( W == 4 && N % 4 >= 2 )
    {
        typename VecOf<T, 2>::type x;
        x[0] = src[i];
        x[1] = src[i + 1];
        *reinterpret_cast<typename VecOf<T, 2>::type*>( dst + i ) = x;
        i += 2;
    }
#pragma unroll
    for ( ; i < N; ++i )
        dst[i] = src[i];
}
} // namespace detail

template <class T, int N, bool CONTIG>
__device__ __forceinline__ void PFieldDev::load( int64_t p, T* v ) const
{
    if constexpr ( CONTIG )
    {
        detail::vec_copy_in<T, N>( ptr<const T>( row( p ), 0 ), v );
    }
    else
    {
        const uint32_t b = base( p );
#pragma unroll
        for ( int c = 0; c < N; ++c )
            v[c] = *ptr<const T>( b, c );
    }
}

template <class T, int N, bool CONTIG>
__device__ __forceinline__ void PFieldDev::store( int64_t p, const T* v ) const
{
    if constexpr ( CONTIG )
    {
        detail::vec_copy_out<T, N>( v, ptr<T>( row( p ), 0 ) );
    }
    else
    {
        const uint32_t b = base( p );
#pragma unroll
        for ( int c = 0; c < N; ++c )
            *ptr<T>( b, c ) = v[c];
    }
}

// Grid array: element strides are 32-bit and every element's byte offset fits
// in 32 bits (checked on the host), so device addressing is a uniform 64-bit
// base plus a 32-bit offset.
struct GFieldDev
{
    char* data;
    int32_t s[4];
    int32_t ext[4];
};

template <class T>
__device__ __forceinline__ T* gptr( const GFieldDev& g, int elem )
{
    return reinterpret_cast<T*>(
        g.data + (uint32_t)( (uint32_t)elem * (uint32_t)sizeof( T ) ) );
}

// Bilinear forms B(P, G; W, dW) between a particle vector P and a node vector
// G.  P2G scatters dB/dG, G2P gathers dB/dP and the position adjoint
// differentiates B through the weights.
enum Form : int32_t
{
    FORM_SV = 0,  // P[1]  G[1]: P0 G0 W
    FORM_VV = 1,  // P[3]  G[3]: sum_d Pd Gd W
    FORM_SG = 2,  // P[1]  G[3]: sum_d P0 Gd dW_d
    FORM_VD = 3,  // P[3]  G[1]: sum_d Pd G0 dW_d
    FORM_TD = 4,  // P[9]  G[3]: sum P[3a+b] G[a] dW_b
    FORM_TDT = 5, // P[9]  G[3]: sum P[3a+b] G[b] dW_a
    FORM_COUNT = 6
};

// Forward operator -> form.  P2G: ScalarValue->SV, VectorValue->VV,
// ScalarGradient->SG, VectorDivergence->VD, TensorDivergence->TD.
// G2P: ScalarValue->SV, VectorValue->VV, ScalarGradient->VD,
// VectorGradient->TDT, VectorDivergence->SG.
inline int p2g_form( int op )
{
    static const int f[5] = { FORM_SV, FORM_VV, FORM_SG, FORM_VD, FORM_TD };
    return f[op];
}
inline int g2p_form( int op )
{
    static const int f[5] = { FORM_SV, FORM_VV, FORM_VD, FORM_TDT, FORM_SG };
    return f[op];
}
inline int form_pcomp( int form )
{
    static const int n[6] = { 1, 3, 1, 3, 9, 9 };
    return n[form];
}
inline int form_gdof( int form )
{
    static const int n[6] = { 1, 3, 3, 1, 3, 3 };
    return n[form];
}

constexpr int MAX_TERMS = 3;       // terms fused into one scatter pass
constexpr int MAX_GATHER_TERMS = 5; // terms fused into one gather pass
constexpr int MAX_CALL_TERMS = 16; // terms accepted by one API call

// One term of a scatter pass (P2G forward, or G2P adjoint):
//   grid += mult * dB/dG (P = pin)
//   xbar += mult * dB/dx (P = pin, G = gx)     [only when the pass has xbar]
struct ScatterTermDev
{
    PFieldDev pin;
    GFieldDev grid;
    GFieldDev gx;
    double mult;
    int32_t form;
};

// One term of a gather pass (G2P forward, or P2G adjoint):
//   pout += mult * dB/dP (G = grid)
//   xbar += mult * dB/dx (P = px, G = grid)     [only when the pass has xbar]
struct GatherTermDev
{
    PFieldDev pout;
    PFieldDev px;
    GFieldDev grid;
    double mult;
    int32_t form;
};

struct ScatterArgs
{
    MeshDev mesh;
    PFieldDev points;
    PFieldDev xbar;
    int64_t begin;
    int64_t end;
    int32_t nterms;
    int32_t has_xbar;
    int32_t contig; // every particle field of the pass has vector_length 1
    ScatterTermDev t[MAX_TERMS];
    unsigned long long* skipped;
};

struct GatherArgs
{
    MeshDev mesh;
    PFieldDev points;
    PFieldDev xbar;
    int64_t begin;
    int64_t end;
    int32_t nterms;
    int32_t has_xbar;
    int32_t contig; // every particle field of the pass has vector_length 1
    GatherTermDev t[MAX_GATHER_TERMS];
    unsigned long long* skipped;
};

// Every term of a call in one pass over the particles, for any set of
// operators: the spline is evaluated once per particle, then the G2P terms
// run in call order (each adds into its particle field) and after them the
// P2G terms (each reads its particle field, which a G2P term of the same
// particle may just have updated, and adds into its grid with atomics).
// One term of such a pass: its particle field (output of a G2P term, input
// of a P2G term), grid, multiplier and form.
struct MultiTermDev
{
    PFieldDev f;
    GFieldDev grid;
    double mult;
    int32_t form;
};
struct MultiTermArgs
{
    MeshDev mesh;
    PFieldDev points;
    int64_t begin;
    int64_t end;
    int32_t n_g2p;
    int32_t n_p2g;
    MultiTermDev g[MAX_CALL_TERMS];
    MultiTermDev s[MAX_CALL_TERMS];
    unsigned long long* skipped;
};
// Kernel arguments are limited to 4 KiB.
static_assert( sizeof( MultiTermArgs ) <= 4000, "MultiTermArgs exceeds the kernel argument space" );
inline MultiTermDev multi_term( const GatherTermDev& t ) { return { t.pout, t.grid, t.mult, t.form }; }
inline MultiTermDev multi_term( const ScatterTermDev& t ) { return { t.pin, t.grid, t.mult, t.form }; }

// Deterministic P2G of one term: every node of the term's grid sums the
// contributions of the particles of the cells around it, cell by cell in
// cardinal order and in binned order inside a cell, and adds the sum to
// itself (one writer per node, no atomics).  The binning covers every
// particle (cell keys clamped into the owned cells) and lists them through
// perm.
struct PullArgs
{
    MeshDev mesh;
    PFieldDev points;
    // One term, or the MPM set (ScalarValue, VectorValue, TensorDivergence)
    // in one pass; every term's grid has the same extents.
    MultiTermDev term[3];
    int32_t nterms;
    const int32_t* counts;
    const int64_t* offsets;
    const int64_t* perm;
};

// Brick tiling of cell-sorted particles.  A brick is tile[0] x tile[1] x
// tile[2] mesh cells; its particles are the tile[0] * tile[1] cell runs along
// the last dimension (contiguous in the cell-sorted order).  Bricks are cut
// into parts of at most `cap` particles; a workgroup processes one part at a
// time from the part table (filled on the device before the launch).
struct TileArgs
{
    const int64_t* cell_offsets; // exclusive scan, per mesh cell
    const int32_t* cell_counts;
    const int2* parts;           // (brick, part index within the brick)
    const int32_t* num_parts;    // number of entries of `parts`
    int32_t tile[3];             // cells per brick and dimension
    int32_t ntile[3];            // bricks per dimension
    int32_t win[3];              // window nodes per dimension
    int32_t flush_perm[3];       // grid dims from largest to smallest stride
    int32_t max_runs;            // tile[0] * tile[1]
    int32_t max_win_nodes;       // win[0] * win[1] * win[2]
    int32_t cap;                 // particles per part
    int32_t sub;                 // particles of a scatter's records in LDS
    int32_t thin;                // fewer than SCATTER_THIN particles a cell
    int32_t grid;                // workgroups launched (a multiple of 8)
    int64_t bin_begin;           // particle index of cell offset 0
    // Particle at each binned position q (perm[q - bin_begin]) when the
    // binning does not reorder the particles themselves; nullptr: the
    // particle at q is q.
    const int64_t* perm;
    __device__ __forceinline__ int64_t particle( int64_t q ) const
    {
        return perm ? perm[q - bin_begin] : q;
    }
};

// Cell-tiled scatter (ca_scatter.hip).  A pass is of one of two kinds: with
// value-type terms only, or with gradient-type ones (`grad`: three more
// values in a slot of its records).
constexpr int SCATTER_BLOCK = 256;
constexpr bool scatter_grad( int vals ) { return vals >= 3; }
// Weights at the head of a slot row, and the row with its values, even.
constexpr int scatter_row_head( int order, bool grad ) { return order == 1 ? ( grad ? 3 : 1 ) : 2; }
constexpr int scatter_row( int order, int vals )
{
    return ( scatter_row_head( order, scatter_grad( vals ) ) + vals + 1 ) / 2 * 2;
}
// Waves per SIMD the registers of a pass leave room for without spilling
// (a spill of a few registers at one wave more measured 1.2 to 2 times
// slower), and the LDS that lets as many workgroups run on a CU.
constexpr int scatter_waves( bool fp64, bool grad )
{
    return fp64 ? ( grad ? 2 : 3 ) : ( grad ? 3 : 4 );
}
constexpr int scatter_lds( int waves ) { return 160 * 1024 / waves - 512; }
// Particles of a wave's batch of 64 whose records are in LDS at a time.  16
// leave the window more room (and cost a wave per SIMD with value terms if
// they were 64), 32 break fewer runs of one cell apart.  Value terms take 16:
// mass and momentum of 8.4 M clustered particles 0.46 ms against 0.50 ms.
// Gradient terms take 32, the fused MPM P2G below scatter_sparse particles a cell
// 16.  us with 32 and with 16, quadratic, 96^3 cells (80^3 from 10 a cell on):
//   a cell    2        3        4        5        6        7        8        10
//   FP32  435 363  472 424  462 463  481 450  471 475  477 492  485 509  328 341
//   FP64  634 517  680 551  703 566  754 614  755 666  785 722  795 783  510 543
// (cubic splines the same; clustered clouds, FP32 at 4 and 8: 418 420  522 549,
// FP64: 590 571  802 875; linear splines, 2, FP64: 0.51 0.54 ms; the G2P adjoint
// at 3: 0.40 0.42 ms).
constexpr double scatter_sparse( bool fp64 ) { return fp64 ? 8.0 : 6.0; }
// Particles a cell below which the products of an FP32 group of up to four are
// summed in two chains.
constexpr double SCATTER_THIN = 4.0;
constexpr int scatter_sub( bool fp64, int order, bool grad, int nslot, double mean_ppc )
{
    return !grad || ( order > 1 && nslot > 1 && mean_ppc < scatter_sparse( fp64 ) ) ? 16 : 32;
}
// Cells of a scatter brick along k, a compile-time stride of the LDS window
// (linear splines: groups of three cells).
constexpr int scatter_cells_k( int order ) { return order == 1 ? 9 : 8; }
// A scatter record: 16 weights (linear splines: 8) and four slot rows, with a
// stride that puts the 16-byte pieces eight lanes write at a time into
// different LDS banks.
constexpr int scatter_record( bool fp64, int order, int row )
{
    const int len = ( order == 1 ? 8 : 16 ) + 4 * row;
    return len + ( fp64 ? 2 : ( len % 8 == 0 && len % 16 != 0 ? 0 : 4 ) );
}

// Launch-time error/timing context owned by the C-ABI layer.
class Launcher
{
  public:
    virtual ~Launcher() = default;
    // Called around every kernel launch; name is the kernel family.
    virtual void before( const char* name, hipStream_t s ) = 0;
    virtual void after( const char* name, hipStream_t s ) = 0;
};

// Fused term sets with their own kernels; any other multi-term call runs one
// single-form pass per term.
enum Plan : int32_t
{
    PLAN_SINGLE = 0,  // one term, any form
    PLAN_MPM_P2G = 1, // (SV, VV, TD): mass, momentum, stress divergence
    PLAN_MPM_G2P = 2, // (VV, TDT) on one shared grid: velocity + gradient
    PLAN_MASS_MOMENTUM = 3, // (SV, VV): mass and momentum (P2G only)
    // Gather only: the P2G adjoint of (SV, VV, TD) with the position part
    // of the G2P adjoint of (VV, TDT) on one shared grid, in one pass.
    PLAN_MPM_ADJOINT = 4
};

// Kernel launchers (return hipSuccess or the launch error), one set per
// spline order (compiled in separate translation units).
#define CABANA_AMD_DECLARE_LAUNCHERS( SUFFIX )                                 \
    hipError_t launch_gather_##SUFFIX( Launcher& L, bool fp64, int plan,       \
                                       const GatherArgs& a, hipStream_t s );   \
    hipError_t launch_scatter_atomic_##SUFFIX( Launcher& L, bool fp64,         \
                                               int plan, const ScatterArgs& a, \
                                               hipStream_t s );                \
    hipError_t launch_multi_term_##SUFFIX( Launcher& L, bool fp64,             \
                                           const MultiTermArgs& a, hipStream_t s ); \
    hipError_t launch_p2g_pull_##SUFFIX( Launcher& L, bool fp64, const PullArgs& a, \
                                         hipStream_t s );                      \
    hipError_t launch_count_outside_##SUFFIX( Launcher& L, const MeshDev& m,   \
                                              const PFieldDev& pts, int64_t n, \
                                              unsigned long long* skipped,     \
                                              hipStream_t s );
#define CABANA_AMD_DECLARE_TILED( SUFFIX )                                     \
    hipError_t launch_gather_tiled_##SUFFIX( Launcher& L, bool fp64, int plan, \
                                             const GatherArgs& a,              \
                                             const TileArgs& t, size_t lds,    \
                                             hipStream_t s );                  \
    hipError_t launch_scatter_cells_##SUFFIX( Launcher& L, bool fp64,          \
                                              int plan, const ScatterArgs& a,  \
                                              const TileArgs& t, size_t lds,   \
                                              hipStream_t s );
CABANA_AMD_DECLARE_TILED( o1 )
CABANA_AMD_DECLARE_TILED( o2 )
CABANA_AMD_DECLARE_TILED( o3 )
CABANA_AMD_DECLARE_LAUNCHERS( o1 )
CABANA_AMD_DECLARE_LAUNCHERS( o2 )
CABANA_AMD_DECLARE_LAUNCHERS( o3 )
// Orders 0 and 4 to 6 run the per-particle (untiled) kernels only.
CABANA_AMD_DECLARE_LAUNCHERS( o0 )
CABANA_AMD_DECLARE_LAUNCHERS( o4 )
CABANA_AMD_DECLARE_LAUNCHERS( o5 )
CABANA_AMD_DECLARE_LAUNCHERS( o6 )

// Halo kernels on ghosted arrays of one entity (ng arrays that share no
// memory, in one launch).
hipError_t launch_halo_gather( Launcher& L, bool fp64, const MeshDev& m, const GFieldDev* g,
                               int ng, int width, hipStream_t s );
hipError_t launch_halo_scatter_sum( Launcher& L, bool fp64, const MeshDev& m, const GFieldDev* g,
                                    int ng, int width, hipStream_t s );
// Transpose of the fold for a cotangent grid: ghost := owner within the band,
// 0 for every other non-owned node.
hipError_t launch_halo_adjoint_fill( Launcher& L, bool fp64, const MeshDev& m, const GFieldDev* g,
                                     int ng, int width, hipStream_t s );
// Zero every non-owned node.
hipError_t launch_zero_ghosts( Launcher& L, bool fp64, const MeshDev& m, const GFieldDev* g,
                               int ng, hipStream_t s );

// Binning.
struct CartGridDev
{
    double min[3];
    double rdx[3];
    int32_t nx[3];
};
hipError_t launch_exclusive_scan( Launcher& L, const int32_t* in, int64_t* out,
                                  int64_t n, int64_t* block_sums,
                                  int64_t nblock_cap, hipStream_t s );
// Scratch of a sorting build of n particles: keys and values of two buffers
// (n + 64 int32 each), hist of 2^digit_bits * lcl_sort_tiles( n ) int32 and
// the totals of SORT_MAX_DIGITS digits.
constexpr int SORT_MAX_DIGITS = 256;
struct SortScratch
{
    int32_t* keys_a;
    int32_t* keys_b;
    int32_t* vals_a;
    int32_t* vals_b;
    int32_t* hist;
    int64_t* totals;
};
int64_t lcl_sort_tiles( int64_t n );
int lcl_sort_passes( int key_bits, int* digit_bits );
// Bins particles [begin, begin + n): keys (cell index, or bad_key outside the
// grid, counted in *bad), a stable radix sort of them over key_bits bits,
// counts[c] and offsets[c] of bins 0..ncell-1.  The sorted order leaves as
// begin + index in permutes.
hipError_t launch_lcl_build( Launcher& L, const PFieldDev& pos, int64_t begin, int64_t n,
                             const CartGridDev& g, int32_t bad_key, unsigned long long* bad,
                             int key_bits, const SortScratch& w, int64_t* permutes, int64_t ncell,
                             int32_t* counts, int64_t* offsets, hipStream_t s );
// The same with owned-cell keys (clamped into the owned cells) of particles
// [0, n), for the library's own binning.
hipError_t launch_auto_bin_sort( Launcher& L, const PFieldDev& pos, int64_t n, const MeshDev& m,
                                 int key_bits, const SortScratch& w, int64_t* permutes,
                                 int64_t ncell, int32_t* counts, int64_t* offsets, hipStream_t s );
// Row-contiguous members of one particle set, permuted in one fused pass:
// member f's rows are row_words[f] 4-byte words apart, words[f] of them per
// particle, and its block of the scratch starts at n * word_offset[f] words.
constexpr int PERMUTE_MAX_MEMBERS = 16;
struct PermuteMembers
{
    int32_t count;
    int32_t words[PERMUTE_MAX_MEMBERS];
    const uint32_t* src[PERMUTE_MAX_MEMBERS];
    int64_t row_words[PERMUTE_MAX_MEMBERS];
    int64_t word_offset[PERMUTE_MAX_MEMBERS];
};
// Permutes count members in place (field[i] = old field[permutes[i - begin]]
// for i in [begin, end)); scratch holds at least
// sum over members of (elem_size * ncomp) * (end - begin + 1) bytes.
hipError_t launch_permute_members( Launcher& L, const PFieldDev* f,
                                   const int* elem_size, int count,
                                   const int64_t* permutes, int64_t begin,
                                   int64_t end, void* scratch, hipStream_t s );
hipError_t launch_permute_gather( Launcher& L, const PFieldDev& f,
                                  int elem_size, const int64_t* permutes,
                                  int64_t begin, int64_t end, void* scratch,
                                  hipStream_t s );
hipError_t launch_permute_copy_back( Launcher& L, const PFieldDev& f,
                                     int elem_size, int64_t begin,
                                     int64_t end, const void* scratch,
                                     hipStream_t s );
hipError_t launch_fill_i32( Launcher& L, int32_t* dst, int64_t n,
                            int32_t value, hipStream_t s );

// Bounds of particleMigrate on one rank (Cabana_Grid_ParticleDistributor.hpp
// :87-148, :170-221), formed on the host as LocalMesh and GlobalMesh form
// them: the band of migrateCount (ghosted corners moved in by
// min_halo_width cells), the owned corners, the global corners and extent.
struct MigrateBoundsDev
{
    double band_lo[3];
    double band_hi[3];
    double own_lo[3];
    double own_hi[3];
    double global_lo[3];
    double global_hi[3];
    double extent[3];
    int32_t periodic[3];
};
// *count += particles outside the band.
hipError_t launch_migrate_count( Launcher& L, const PFieldDev& pos, int64_t n,
                                 const MigrateBoundsDev& b, unsigned long long* count,
                                 hipStream_t s );
// Periodic shift of the positions in place, keep[p] = 0 for particles
// leaving through a non-periodic boundary, *dropped += their number.
hipError_t launch_migrate_shift( Launcher& L, const PFieldDev& pos, int64_t n,
                                 const MigrateBoundsDev& b, int32_t* keep,
                                 unsigned long long* dropped, hipStream_t s );
// The library's own binning by counting: cells counted with atomics as the
// keys are formed, offsets by a scan, particles placed by their arrival
// number.  Not stable (the order inside a cell varies), so the deterministic
// mode sorts instead.
hipError_t launch_auto_bin_count( Launcher& L, const PFieldDev& pos, int64_t n, const MeshDev& m,
                                  int64_t ncell, int32_t* keys, int32_t* rank, int32_t* counts,
                                  int64_t* offsets, int64_t* block_sums, int64_t nblock_cap,
                                  int64_t* perm, hipStream_t s );
// Whether counting is used: beyond the one-workgroup sort, and where the cells
// are not so few that their counters would be contended.
bool auto_bin_counts( int64_t n, int64_t ncell );
// Block [lo, lo + n) of every dimension of a grid array, packed x fastest
// after the dofs (the BOV data order) into out.
hipError_t launch_bov_pack( Launcher& L, bool fp64, const GFieldDev& g, int lo, const int n[3],
                            void* out, hipStream_t s );
// idx[rank[p]] = p for the kept particles (rank: exclusive scan of keep).
hipError_t launch_compact_index( Launcher& L, const int32_t* keep, const int64_t* rank,
                                 int64_t n, int64_t* idx, hipStream_t s );
// Part table of a brick tiling: brick_nparts (nbricks ints), brick_start
// (nbricks int64), block_sums (scan scratch, nblock_cap int64), parts
// (nbricks + n / cap entries at most) and num_parts (1 int).
hipError_t launch_brick_parts( Launcher& L, const TileArgs& t,
                               const int32_t num_cell[3], int32_t* brick_nparts,
                               int64_t* brick_start, int64_t* block_sums,
                               int64_t nblock_cap, int2* parts,
                               int32_t* num_parts, hipStream_t s );

// p2g with the brick part table of a tiled scatter built in `scratch`
// (scratch_bytes long) instead of the context's allocations; the context's
// device must be current.  Records an error on the context and returns its
// status.
cabana_amd_status p2g_fixed_scratch( cabana_amd_context* ctx, const cabana_amd_mesh* mesh,
                                     int32_t order, const cabana_amd_particle_field* points,
                                     int32_t num_terms, const cabana_amd_p2g_term* terms,
                                     int32_t halo_width, const cabana_amd_binning* bins,
                                     cabana_amd_stream stream, void* scratch,
                                     size_t scratch_bytes );
// Records msg as the context's (and the thread's) last error; returns st.
cabana_amd_status fail_with( cabana_amd_context* ctx, cabana_amd_status st, const char* msg );

// LDS atomic-add throughput probe (ca_probe.hip): iters adds per lane over
// num_groups workgroups of 256 threads; ms = kernel time.
hipError_t probe_lds_add( bool fp64, int iters, int num_groups, void* out, hipStream_t s,
                          float& ms );

} // namespace cabana_amd
