// Cell-tiled scatter of cell-sorted particles on the matrix cores, one spline
// order per translation unit (CA_ORDER set on the compile line): P2G forward
// and the grid part of the G2P adjoint.
//
// Every stencil of a particle of one mesh cell lies in the cell's 4^3 node
// window (linear splines: the window of three cells along k).  With the 1-D
// weights w and gradients g along the window padded by zeros, a node value is
//   G[(i,j),(k,d)] = sum_p  (wx_i wy_j) (wz_k P1_d + gz_k P4_d)
//                         + (gx_i wy_j) (wz_k P2_d) + (wx_i gy_j) (wz_k P3_d)
// which is a matrix product over the particles with 16 rows (i, j) and 16
// columns (k, d): v_mfma_*_16x16x4 takes four particles at a time, one product
// for value-type dofs and three for gradient-type ones.  Particles are taken
// in the order of the binning, so nothing is sorted in the kernel: a wave
// walks its share of the part, 64 particles a batch (one per lane: positions,
// weights and attributes, written to the wave's records in LDS), then the
// batch's runs of equal cell, four particles a step.
//
// Linear splines reach 2 x 2 nodes along (i, j), four rows of the sixteen:
// v_mfma_*_4x4x* takes the same four particles a step with rows (i, j) and
// columns d, a block for every k (and, in FP32, every particle), at a quarter
// of the matrix time.
//
// What bounds it: instruction issue.  FP32 matrix and vector instructions do
// not overlap on a SIMD of this chip (137 and 166 cycles of each alone take 299
// together), so a batch of 64 particles of the MPM P2G, quadratic, FP32, costs
// the 3270 vector and 2340 matrix cycles of its wave one after the other, and
// waits for LDS take most of the remaining 1750.  HBM moves 2.6 GB in 1.57 ms.
// Against the kernel this one replaced, which sorted each task's particles in
// LDS and added their 27 nodes by LDS atomics, spent half its time at barriers:
//   MPM P2G, 33.6 M particles of 128^3 cells, quadratic, FP32  2.47 -> 1.57 ms
//   MPM P2G, odd grid, cubic, FP64                             0.70 -> 0.36 ms
//   mass and momentum, 8.4 M clustered particles, FP32         0.70 -> 0.45 ms
//   MPM P2G, 7.1 M particles of 96^3 cells, linear, FP64       0.49 -> 0.37 ms
// (linear splines in 16 x 16 products: 0.52 ms).
#include "ca_tiles.hpp"

namespace cabana_amd
{
namespace
{

// Columns of the matrix product.  A tile is one 16 x 16 accumulator: columns
// (k, slot) of four window nodes and four slots, each slot a grid dof.  The
// ScalarValue and VectorValue terms of a fused P2G share a tile (slot 0 and
// slots 1 to 3); every other form has its dofs in slots 0 to 2.
template <bool SHARED, int... FORMS>
struct Tiles
{
    using FL = FormList<FORMS...>;
    static constexpr bool PAIR = !SHARED && FL::N >= 2;
    static constexpr int NT = SHARED ? 1 : ( FL::N == 3 ? 2 : 1 );
    static constexpr int first_term( int tile ) { return tile == 0 ? 0 : 2; }
    static constexpr int last_term( int tile )
    {
        return SHARED ? FL::N - 1 : ( tile == 0 ? ( PAIR ? 1 : 0 ) : 2 );
    }
    static constexpr bool value_form( int f ) { return f == FORM_SV || f == FORM_VV; }
    // Slots of a tile that hold a dof.
    static constexpr int nd( int tile )
    {
        return ( PAIR && tile == 0 ) ? 4 : ng_of( FL::v[last_term( tile )] );
    }
    // The tile has value-type (P1) and gradient-type (P2, P3, P4) columns.
    static constexpr bool has_v( int tile )
    {
        bool r = false;
        for ( int t = first_term( tile ); t <= last_term( tile ); ++t )
            r = r || value_form( FL::v[t] );
        return r;
    }
    static constexpr bool has_g( int tile )
    {
        bool r = false;
        for ( int t = first_term( tile ); t <= last_term( tile ); ++t )
            r = r || !value_form( FL::v[t] );
        return r;
    }
    static constexpr bool any_g() { return has_g( 0 ) || has_g( NT - 1 ); }
    // Offset of a tile's values in a record's slot row, after its weights.
    static constexpr int val( int tile )
    {
        int o = scatter_row_head( ORDER, any_g() );
        for ( int i = 0; i < tile; ++i )
            o += ( has_v( i ) ? 1 : 0 ) + ( has_g( i ) ? 3 : 0 );
        return o;
    }
    static constexpr int row_len() { return val( NT ); }
    static constexpr int row() { return ( row_len() + 1 ) / 2 * 2; }
    static constexpr int win_dofs()
    {
        int n = 0;
        for ( int i = 0; i < NT; ++i )
            n += nd( i );
        return n;
    }
};

// Record of a particle: weight and gradient along QUAD and along k of the four
// window nodes, then the four slot rows (weight and gradient along SLOT of the
// node with the slot's number, then the slot's values) in 16-byte chunks,
// [chunk][slot].  Linear splines: weight and gradient along k of the four
// window nodes, then slot rows that begin with the products of the x and y
// weights of the (i, j) node with the slot's number (value, x and y gradient).
// The record stride spreads the four records of a step over
// the LDS banks.
template <class Real, int ROW>
struct Record
{
    // Values before the slot rows (linear splines: along k only).
    static constexpr int HEAD = ORDER == 1 ? 8 : 16;
    static constexpr int CW = 16 / (int)sizeof( Real );
    static constexpr int NC = ( ROW + CW - 1 ) / CW;
    static constexpr int STRIDE = scatter_record( sizeof( Real ) == 8, ORDER, ROW );
    static constexpr int width( int c ) { return ROW - c * CW < CW ? ROW - c * CW : CW; }
    static constexpr int at( int c, int slot ) { return HEAD + 4 * CW * c + slot * width( c ); }
    template <int N>
    struct Vec
    {
        typedef Real type __attribute__( ( ext_vector_type( N ) ) );
    };
    static __device__ __forceinline__ void put_row( Real* rec, int slot, const Real* v )
    {
        static_for<NC>( [&]( auto C ) {
            constexpr int c = C;
            typename Vec<width( c )>::type x;
#pragma unroll
            for ( int e = 0; e < width( c ); ++e )
                x[e] = v[c * CW + e];
            *reinterpret_cast<typename Vec<width( c )>::type*>( rec + at( c, slot ) ) = x;
        } );
    }
    static __device__ __forceinline__ void put_pair( Real* at, Real w, Real g )
    {
        *reinterpret_cast<typename Vec<2>::type*>( at ) = typename Vec<2>::type{ w, g };
    }
    static __device__ __forceinline__ void get_pair( const Real* at, Real& w, Real& g )
    {
        const auto x = *reinterpret_cast<const typename Vec<2>::type*>( at );
        w = x[0];
        g = x[1];
    }
    static __device__ __forceinline__ void get_row( const Real* rec, int slot, Real* v )
    {
        static_for<NC>( [&]( auto C ) {
            constexpr int c = C;
            const auto x = *reinterpret_cast<const typename Vec<width( c )>::type*>( rec + at( c, slot ) );
#pragma unroll
            for ( int e = 0; e < width( c ); ++e )
                v[c * CW + e] = x[e];
        } );
    }
};

// The slot values of form FORM: r[0] = P1 (value-type) or r = (P2, P3, P4).
template <int FORM, class Real>
__device__ __forceinline__ void slot_values( const Real* P, int d, Real* r )
{
    if constexpr ( FORM == FORM_SV || FORM == FORM_VV )
        r[0] = P[d];
    else if constexpr ( FORM == FORM_SG )
    {
        r[0] = d == 0 ? P[0] : Real( 0 );
        r[1] = d == 1 ? P[0] : Real( 0 );
        r[2] = d == 2 ? P[0] : Real( 0 );
    }
    else if constexpr ( FORM == FORM_VD )
    {
#pragma unroll
        for ( int b = 0; b < 3; ++b )
            r[b] = P[b];
    }
    else if constexpr ( FORM == FORM_TD )
    {
#pragma unroll
        for ( int b = 0; b < 3; ++b )
            r[b] = P[3 * d + b];
    }
    else
    {
#pragma unroll
        for ( int b = 0; b < 3; ++b )
            r[b] = P[3 * b + d];
    }
}

// Matrix product of four particles.  Row rho of lane l's accumulator register
// r is 4 (l / 16) + r in FP32 and l / 16 + 4 r in FP64.  Window node i sits in
// lanes l / 16 = i and node j in register r = j either way: rho / 4 and rho % 4
// are (i, j) in FP32 and (j, i) in FP64.  QUAD is the dimension along rho / 4
// (one weight per quad of a row of 16 lanes), SLOT the one along rho % 4.
template <class Real>
struct Mfma;
template <>
struct Mfma<float>
{
    typedef float V4 __attribute__( ( ext_vector_type( 4 ) ) );
    static constexpr int QUAD = 0, SLOT = 1;
    static __device__ __forceinline__ V4 mac( float a, float b, V4 c )
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32( a, b, c, 0, 0, 0 );
    }
};
template <>
struct Mfma<double>
{
    typedef double V4 __attribute__( ( ext_vector_type( 4 ) ) );
    static constexpr int QUAD = 1, SLOT = 0;
    static __device__ __forceinline__ V4 mac( double a, double b, V4 c )
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64( a, b, c, 0, 0, 0 );
    }
};

// Accumulators of a tile and a chunk's sums.  In the 4 x 4 products of linear
// splines lane l holds column l % 4 of block l / 4: in FP32 rows r = (i, j) of
// register r, a block for each particle of the step (l / 16) and each k; in
// FP64 row l / 16 and a block for each k.
template <class Real>
constexpr int acc_regs()
{
    return ORDER == 1 && sizeof( Real ) == 8 ? 1 : 4;
}
[[maybe_unused]] __device__ __forceinline__ Mfma<float>::V4
mac4( float a, float b, Mfma<float>::V4 c )
{
    return __builtin_amdgcn_mfma_f32_4x4x1f32( a, b, c, 0, 0, 0 );
}
[[maybe_unused]] __device__ __forceinline__ Mfma<double>::V4
mac4( double a, double b, Mfma<double>::V4 c )
{
    c[0] = __builtin_amdgcn_mfma_f64_4x4x4f64( a, b, c[0], 0, 0, 0 );
    return c;
}

// DPP move: lane Q of every quad to its four lanes.
template <int CTRL>
__device__ __forceinline__ float dpp( float x )
{
    return __builtin_bit_cast( float, __builtin_amdgcn_update_dpp(
        0, __builtin_bit_cast( int, x ), CTRL, 0xf, 0xf, true ) );
}
template <int CTRL>
__device__ __forceinline__ double dpp( double x )
{
    typedef int I2 __attribute__( ( ext_vector_type( 2 ) ) );
    const I2 v = __builtin_bit_cast( I2, x );
    I2 r;
    r.x = __builtin_amdgcn_update_dpp( 0, v.x, CTRL, 0xf, 0xf, true );
    r.y = __builtin_amdgcn_update_dpp( 0, v.y, CTRL, 0xf, 0xf, true );
    return __builtin_bit_cast( double, r );
}
template <int Q, class Real>
__device__ __forceinline__ Real quad_lane( Real x )
{
    return dpp<Q * 0x55>( x );
}
// The value of lane ^ MASK.
template <int MASK>
__device__ __forceinline__ uint32_t lane_xor( uint32_t v )
{
    if constexpr ( MASK == 1 )
        return __builtin_amdgcn_update_dpp( 0, v, 0xb1, 0xf, 0xf, true );
    else if constexpr ( MASK == 2 )
        return __builtin_amdgcn_update_dpp( 0, v, 0x4e, 0xf, 0xf, true );
    else if constexpr ( MASK == 3 )
        return __builtin_amdgcn_update_dpp( 0, v, 0x1b, 0xf, 0xf, true );
    else if constexpr ( MASK == 7 )
        return __builtin_amdgcn_update_dpp( 0, v, 0x141, 0xf, 0xf, true );
    else if constexpr ( MASK == 15 )
        return __builtin_amdgcn_update_dpp( 0, v, 0x140, 0xf, 0xf, true );
    else if constexpr ( MASK == 8 )
        return __builtin_amdgcn_update_dpp( 0, v, 0x128, 0xf, 0xf, true );
    else
        return __shfl_xor( v, MASK, 64 );
}
// One compare-exchange with lane ^ MASK; BIT is set in the lane that keeps the
// larger value.
template <int MASK, int BIT>
__device__ __forceinline__ uint32_t lane_exchange( uint32_t v )
{
    const uint32_t u = lane_xor<MASK>( v );
    return ( threadIdx.x & BIT ) ? max( u, v ) : min( u, v );
}
// Ascending sort of a wave's 64 values (bitonic).
__device__ __forceinline__ uint32_t sort_lanes( uint32_t v )
{
    static_for<6>( [&]( auto S ) {
        constexpr int s = S;
        v = lane_exchange<( 2 << s ) - 1, 1 << s>( v );
        static_for<s>( [&]( auto T ) {
            constexpr int b = 1 << ( s - 1 - T );
            v = lane_exchange<b, b>( v );
        } );
    } );
    return v;
}
// Attributes of a pass: every term's components in order.
template <int... FORMS>
constexpr int attr_len()
{
    return ( np_of( FORMS ) + ... );
}
template <int... FORMS>
constexpr int attr_of( int t )
{
    constexpr int f[] = { FORMS... };
    int o = 0;
    for ( int i = 0; i < t; ++i )
        o += np_of( f[i] );
    return o;
}

// Global-atomic scatter of one particle (particles whose stencil is outside
// the brick's window, or whose attributes are not finite).  Rare, so its
// loops stay rolled: unrolled, their registers would bound the kernel's.
template <class Real, bool SHARED, int... FORMS>
__device__ __forceinline__ void global_scatter_particle( const ScatterArgs& a, const double x[3],
                                                         const Real* P )
{
    using FL = FormList<FORMS...>;
    Spline3D<ORDER, Real, false> s;
    eval_spline( a.mesh, x, s );
#pragma unroll 1
    for ( int n = 0; n < K * K * K; ++n )
    {
        const int i = n / ( K * K ), j = n / K % K, k = n % K;
        Spline3D<0, Real, false> one;
#pragma unroll
        for ( int q = 0; q < K; ++q )
        {
            one.d[0].w[0] = q == 0 || i == q ? s.d[0].w[q] : one.d[0].w[0];
            one.d[0].g[0] = q == 0 || i == q ? s.d[0].g[q] : one.d[0].g[0];
            one.d[1].w[0] = q == 0 || j == q ? s.d[1].w[q] : one.d[1].w[0];
            one.d[1].g[0] = q == 0 || j == q ? s.d[1].g[q] : one.d[1].g[0];
            one.d[2].w[0] = q == 0 || k == q ? s.d[2].w[q] : one.d[2].w[0];
            one.d[2].g[0] = q == 0 || k == q ? s.d[2].g[q] : one.d[2].g[0];
        }
        const auto nw = node_weights<0, Real, false, false>( one, 0, 0, 0 );
        static_for<FL::N>( [&]( auto I ) {
            constexpr int t = I;
            constexpr int FORM = FL::v[t];
            constexpr int NG = ng_of( FORM );
            const GFieldDev& g = SHARED ? a.t[0].grid : a.t[t].grid;
            Real G[NG];
            form_scatter<FORM>( P + attr_of<FORMS...>( t ), nw, G );
            Real* q = gptr<Real>( g, ( s.d[0].base + i ) * g.s[0] + ( s.d[1].base + j ) * g.s[1] +
                                         ( s.d[2].base + k ) * g.s[2] );
#pragma unroll
            for ( int d = 0; d < NG; ++d )
                atomic_add( q + d * g.s[3], G[d] );
        } );
    }
}

// The run table of a brick in two halves, so its global reads can be issued
// early and committed later: lane r < nruns (<= 64) of wave 0 holds run r's
// raw reads (nothing is computed from them until the commit, so issuing
// them does not wait for them).
struct RunLoad
{
    int64_t start;
    int64_t last_offset;
    int32_t last_count;
};

__device__ __forceinline__ void runs_issue( const TileArgs& ta, const MeshDev& m,
                                            const TileGeom& g, RunLoad& rl )
{
    const int nj = g.c1[1] - g.c0[1];
    const int nruns = ( g.c1[0] - g.c0[0] ) * nj;
    const int r = threadIdx.x;
    rl.start = 0;
    rl.last_offset = 0;
    rl.last_count = 0;
    if ( r < nruns )
    {
        const int ci = g.c0[0] + r / nj, cj = g.c0[1] + r % nj;
        const int64_t cfirst = ( (int64_t)ci * m.num_cell[1] + cj ) * m.num_cell[2] + g.c0[2];
        const int64_t clast = cfirst + ( g.c1[2] - g.c0[2] ) - 1;
        rl.start = ta.cell_offsets[cfirst];
        rl.last_offset = ta.cell_offsets[clast];
        rl.last_count = ta.cell_counts[clast];
    }
}

// Wave 0 writes run_start and the inclusive prefix run_pre (visible after
// the next barrier).
__device__ __forceinline__ void runs_commit( const RunLoad& rl, const TileGeom& g,
                                             int64_t* run_start, int* run_pre )
{
    if ( threadIdx.x >= 64 )
        return;
    const int nruns = ( g.c1[0] - g.c0[0] ) * ( g.c1[1] - g.c0[1] );
    const int lane = threadIdx.x;
    int v = (int)( rl.last_offset + rl.last_count - rl.start );
#pragma unroll
    for ( int o = 1; o < 64; o <<= 1 )
    {
        const int u = __shfl_up( v, o, 64 );
        if ( lane >= o )
            v += u;
    }
    if ( lane < nruns )
    {
        run_start[lane] = rl.start;
        run_pre[lane + 1] = v;
    }
    if ( lane == 0 )
        run_pre[0] = 0;
}

__device__ __forceinline__ float fabs_r( float x ) { return __builtin_fabsf( x ); }
__device__ __forceinline__ double fabs_r( double x ) { return __builtin_fabs( x ); }

// Particles of one batch between their loads and their use (the loads of the
// next batch are in flight while this one is accumulated).
template <class Real, int NP>
struct Batch
{
    double x[3];
    int run;
    Real attr[NP];
};

// Issues the reads of the particle at flattened part position v, run r being a
// run at or before its own.  Every lane reads a particle (past the end, the
// last one), so that nothing of the batch before stays live.
template <class Real, bool CONTIG, int... FORMS>
__device__ __forceinline__ void batch_issue( const ScatterArgs& a, const TileArgs& ta,
                                             const int64_t* run_start, const int* run_pre,
                                             int v, int v1, int& r,
                                             Batch<Real, attr_len<FORMS...>()>& b )
{
    v = min( v, v1 - 1 );
    while ( run_pre[r + 1] <= v )
        ++r;
    b.run = r;
    const int64_t p = ta.particle( ta.bin_begin + run_start[r] + ( v - run_pre[r] ) );
    load_position<CONTIG>( a.points, p, b.x );
    using FL = FormList<FORMS...>;
    static_for<FL::N>( [&]( auto I ) {
        constexpr int t = I;
        a.t[t].pin.template load<Real, np_of( FL::v[t] ), CONTIG>( p,
                                                                   b.attr + attr_of<FORMS...>( t ) );
    } );
}

// Weights along a group's four window nodes, zero outside the stencil, which
// starts off nodes into the window.
template <class Real>
__device__ __forceinline__ void window_weights( const Real* s, int off, Real* w )
{
#pragma unroll
    for ( int n = 0; n < 4; ++n )
    {
        Real v = n < K ? s[n < K ? n : 0] : Real( 0 );
        if constexpr ( ORDER <= 2 )
        {
            const Real v1 = ( n >= 1 && n - 1 < K ) ? s[n >= 1 ? n - 1 : 0] : Real( 0 );
            v = off == 1 ? v1 : v;
        }
        if constexpr ( ORDER == 1 )
        {
            const Real v2 = n >= 2 ? s[n >= 2 ? n - 2 : 0] : Real( 0 );
            v = off == 2 ? v2 : v;
        }
        w[n] = v;
    }
}

// Window nodes along k (a compile-time stride of the LDS window).
constexpr int WK = scatter_cells_k( ORDER ) + ( ORDER == 1 ? 1 : 3 );

// Descending neighbours from which a batch is sorted: each adds about two
// groups, the sort costs about four (2 measured the same, 4 was not tried).
constexpr int SORT_DESCENTS = 3;

// A step's operands as read from the records.
template <class Real, int ROW>
struct Step
{
    Real xz; // one weight of the quad's four (linear splines: wz)
    Real gz; // linear splines
    Real y[ROW];
};

template <class Real, bool CONTIG, bool SHARED, int SUB, int... FORMS>
__global__ __launch_bounds__( SCATTER_BLOCK, ( scatter_waves( sizeof( Real ) == 8, Tiles<SHARED, FORMS...>::any_g() ) ) ) void scatter_cells_kernel(
    ScatterArgs a, TileArgs ta )
{
    using FL = FormList<FORMS...>;
    using TL = Tiles<SHARED, FORMS...>;
    using MF = Mfma<Real>;
    using V4 = typename MF::V4;
    constexpr int NT = TL::NT;
    constexpr int ROW = TL::row();
    using RC = Record<Real, ROW>;
    constexpr int RS = RC::STRIDE;
    constexpr int NP = attr_len<FORMS...>();
    constexpr int NWAVE = SCATTER_BLOCK / 64;
    constexpr int NR = acc_regs<Real>();
    constexpr bool F32 = sizeof( Real ) == 4;
    // Window nodes along k sit in column (node index mod 4), so that the
    // window slides to the next cell without moving the accumulators.  (The
    // windows of the linear spline are three cells apart and do not slide.)
    constexpr bool SLIDE = ORDER != 1;
    // Steps of a chunk at most: the fused passes of sparse particles (records of
    // 16) seldom have more than eight in a group, and chunks of four cost them,
    // and the FP32 P2G of linear splines, 30 to 40 spilled registers.
    constexpr int MAX_STEPS =
        TL::any_g() && ( SUB == 16 || ( ORDER == 1 && F32 && NT == 2 ) ) ? 2 : 4;
    extern __shared__ __align__( 16 ) unsigned char smem[];

    // LDS: the FP64 node window (one block per tile, [node][dof]), the waves'
    // records, the run table.
    const int W[3] = { ta.win[0], ta.win[1], WK };
    const int wnodes = W[0] * W[1] * W[2];
    double* win = reinterpret_cast<double*>( smem );
    size_t off = align16( sizeof( double ) * (size_t)TL::win_dofs() * ta.max_win_nodes );
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane( (int)threadIdx.x >> 6 );
    Real* rec = reinterpret_cast<Real*>( smem + off ) + wave * ( RS * ( SUB + 3 ) );
    off = align16( off + sizeof( Real ) * (size_t)NWAVE * RS * ( SUB + 3 ) );
    int64_t* run_start = reinterpret_cast<int64_t*>( smem + off );
    off = align16( off + sizeof( int64_t ) * ta.max_runs );
    int* run_pre = reinterpret_cast<int*>( smem + off );

    // The lane's place in the products: particle of a step, window row or
    // column, dof slot; and in the accumulators.
    const int pslot = lane >> 4, l16 = lane & 15, kcol = l16 >> 2, slot = lane & 3;

    for ( int e = threadIdx.x; e < TL::win_dofs() * wnodes; e += SCATTER_BLOCK )
        win[e] = 0.0;
    // Records past a group are read (and count zero): they hold finite values.
    for ( int e = lane; e < RS * ( SUB + 3 ); e += 64 )
        rec[e] = Real( 0 );

    // A thirty-second of the largest value: no sum of 16 products overflows
    // where the values do not.
    const Real vmax = Real( sizeof( Real ) == 8 ? 5.6e306 : 1.06e37 ) /
                      ( Real( 1 ) + (Real)a.mesh.rdx[0] + (Real)a.mesh.rdx[1] + (Real)a.mesh.rdx[2] );

    const PartLoop pl( ta );
    for ( int loc = pl.first; pl.more( loc ); loc += pl.stride )
    {
        const int w = pl.part( loc );
        if ( w < 0 )
            continue;
        TileGeom tg;
        part_geometry( ta, a.mesh, w, tg );
        if ( threadIdx.x < 64 )
        {
            RunLoad rl;
            runs_issue( ta, a.mesh, tg, rl );
            runs_commit( rl, tg, run_start, run_pre );
        }
        __syncthreads();
        // Window origin, and the stencil bases (from it) whose nodes lie in the
        // window and in the grid.
        int wlo[3], rmin[3], rcount[3];
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            wlo[d] = tg.c0[d] + a.mesh.halo + BASE_SHIFT;
            rmin[d] = max( 0, -wlo[d] );
            rcount[d] = max( 0, min( W[d], a.mesh.num_node[d] - wlo[d] ) - K + 1 - rmin[d] );
        }
        const int nj = tg.c1[1] - tg.c0[1];
        const int nruns = ( tg.c1[0] - tg.c0[0] ) * nj;
        [[maybe_unused]] const float rnj = 1.0f / (float)nj;
        const int pbeg = tg.part * ta.cap;
        const int pend = min( run_pre[nruns], pbeg + ta.cap );
        // The wave's share: a contiguous range, equal to 16 particles (equal to a
        // batch, one wave of a part of a few batches had little or nothing).
        const int per = ( ( pend - pbeg + NWAVE * 16 - 1 ) / ( NWAVE * 16 ) ) * 16;
        const int v0 = __builtin_amdgcn_readfirstlane( pbeg + wave * per );
        const int v1 = __builtin_amdgcn_readfirstlane( min( pend, v0 + per ) );

        // The open window: key of the group in the accumulators, -1 none.
        int open = -1;
        double acc[NT][NR];
#pragma unroll
        for ( int t = 0; t < NT; ++t )
#pragma unroll
            for ( int r = 0; r < NR; ++r )
                acc[t][r] = 0.0;
        // Adds the accumulators to the LDS window (all columns, or the window's
        // first node along k) and clears them.
        auto retire = [&]( int key, bool all ) {
            const int dk = SLIDE ? ( kcol - key ) & 3 : kcol;
            // Window node of accumulator register r: (i, j) = (lane / 16, r),
            // or for linear splines r (FP32) or lane / 16 (FP64) = 2 i + j.
            const int i0 = ORDER > 1 ? pslot : ( F32 ? 0 : pslot >> 1 );
            const int j0 = ORDER > 1 || F32 ? 0 : pslot & 1;
            const int node = ( ( ( key >> 16 ) + i0 ) * W[1] + ( ( key >> 8 ) & 255 ) + j0 ) * WK +
                             ( key & 255 ) + dk;
            const bool on = all || dk == 0;
            int wo = 0;
            static_for<NT>( [&]( auto T ) {
                constexpr int t = T;
                constexpr int ND = TL::nd( t );
                if ( on && ( ND == 4 || slot < ND ) )
                {
                    double* q = win + ( wo + node * ND + slot );
#pragma unroll
                    for ( int r = 0; r < NR; ++r )
                        atomicAdd( q + ( ORDER > 1 ? r * WK : ( ( r >> 1 ) * W[1] + ( r & 1 ) ) * WK ) * ND,
                                   acc[t][r] );
                }
                wo += ta.max_win_nodes * ND;
            } );
            if ( on )
            {
#pragma unroll
                for ( int t = 0; t < NT; ++t )
#pragma unroll
                    for ( int r = 0; r < NR; ++r )
                        acc[t][r] = 0.0;
            }
        };

        Batch<Real, NP> bt;
        int run = 0;
        if ( v0 < v1 )
        {
            run = find_run( run_pre, nruns, v0 );
            batch_issue<Real, CONTIG, FORMS...>( a, ta, run_start, run_pre, v0 + lane, v1, run, bt );
        }
        for ( int vb = v0; vb < v1; vb += 64 )
        {
            // Particle phase: stencil base, weights, premultiplied attributes.
            // key: window origin of the particle's group, -1 for none.
            int key = -1;
            Real wt[3][4], gt[3][4], P[NP];
            if ( vb + lane < v1 )
            {
                int org[3];
                bool fits = true;
                [[maybe_unused]] int row[2];
                if constexpr ( ORDER == 2 )
                {
                    row[0] = div_small( bt.run, rnj );
                    row[1] = bt.run - row[0] * nj;
                }
#pragma unroll
                for ( int d = 0; d < 3; ++d )
                {
                    // spline_frac without its early returns.
                    const double x0 = logical_coord<ORDER>( bt.x[d], a.mesh.low[d], a.mesh.rdx[d] );
                    const int i0 = (int)x0;
                    const Real fr = (Real)( x0 - (double)i0 );
                    const int rel = i0 - ORDER / 2 - wlo[d];
                    fits = fits & ( x0 >= 0.0 ) & ( x0 < 2147483648.0 ) &
                           ( (unsigned)( rel - rmin[d] ) < (unsigned)rcount[d] );
                    int l = rel;
                    if constexpr ( ORDER == 2 )
                    {
                        // A quadratic stencil takes three of a window's four
                        // nodes, so a particle up to half a cell out of its
                        // binned row of cells still takes the row's window.
                        if ( d < 2 )
                            l = min( max( row[d], rel - 1 ), rel );
                        else
                            l = min( max( rel - ( fr < Real( 0.5 ) ? 1 : 0 ), 0 ), W[d] - 4 );
                    }
                    if constexpr ( ORDER == 1 )
                        l = d == 2 ? (int)( (unsigned)rel / 3u * 3u ) : rel;
                    org[d] = l;
                    Spline1D<ORDER, Real> sd;
                    spline_weights<ORDER, Real, false>( fr, (Real)a.mesh.rdx[d], sd );
                    window_weights( sd.w, rel - l, wt[d] );
                    window_weights( sd.g, rel - l, gt[d] );
                }
                Real big = Real( 0 );
                static_for<FL::N>( [&]( auto I ) {
                    constexpr int t = I;
                    constexpr int o = attr_of<FORMS...>( t );
                    const Real m = (Real)a.t[t].mult;
#pragma unroll
                    for ( int c = 0; c < np_of( FL::v[t] ); ++c )
                    {
                        P[o + c] = bt.attr[o + c] * m;
                        big += fabs_r( P[o + c] );
                    }
                } );
                // A value that is not finite, or overflows against a weight
                // gradient, must not meet the zero weights of window nodes
                // outside its stencil.
                if ( fits && big <= vmax )
                    key = ( org[0] << 16 ) | ( org[1] << 8 ) | org[2];
                else
                {
                    int base[3];
                    if ( stencil_base<ORDER>( a.mesh, bt.x, base ) )
                        global_scatter_particle<Real, SHARED, FORMS...>( a, bt.x, P );
                    else
                        atomicAdd( a.skipped, 1ull );
                }
            }
            const int nb = min( 64, v1 - vb );
            // Positions that changed since the binning leave a batch with keys
            // out of order: its records are then taken in key order, or every
            // misplaced particle would break its neighbours' group in two.  A
            // fresh binning has ascending keys.  Quadratic MPM P2G and G2P
            // adjoint of 128^3 x 16, FP32, positions moved by 0.1 cell: 3.75 and
            // 2.96 ms without this and the row's window above, 2.15 and 1.59 ms
            // with them (fresh: 1.63 and 1.17 ms).
            int before = __shfl_up( key, 1, 64 );
            uint64_t starts = __ballot( key != before ) | 1;
            int skey = key;
            unsigned rank = lane;
            if ( __popcll( __ballot( key < before ) ) >= SORT_DESCENTS )
            {
                const uint32_t o = sort_lanes( (uint32_t)key << 6 | (uint32_t)lane );
                skey = (int)o >> 6;
                rank = __builtin_amdgcn_ds_permute( (int)( o & 63 ) * 4, lane );
                before = __shfl_up( skey, 1, 64 );
                starts = __ballot( skey != before ) | 1;
            }

            Real* rp = rec + __mul24( rank % SUB, RS );
            static_for<64 / SUB>( [&]( auto IS ) {
                constexpr int s0 = IS * SUB;
                if ( s0 >= nb )
                    return;
                if ( rank / SUB == IS && key >= 0 )
                {
#pragma unroll
                    for ( int n = 0; n < 4; ++n )
                    {
                        if constexpr ( ORDER == 1 )
                            RC::put_pair( rp + 2 * n, wt[2][n], gt[2][n] );
                        else
                        {
                            RC::put_pair( rp + 4 * n, wt[MF::QUAD][n], gt[MF::QUAD][n] );
                            RC::put_pair( rp + 4 * ( ( key + n ) & 3 ) + 2, wt[2][n], gt[2][n] );
                        }
                    }
                    static_for<4>( [&]( auto S ) {
                        constexpr int sl = S;
                        Real v[ROW];
#pragma unroll
                        for ( int c = 0; c < ROW; ++c )
                            v[c] = Real( 0 );
                        if constexpr ( ORDER == 1 )
                        {
                            constexpr int i = sl >> 1, j = sl & 1;
                            v[0] = wt[0][i] * wt[1][j];
                            if constexpr ( TL::any_g() )
                            {
                                v[1] = gt[0][i] * wt[1][j];
                                v[2] = wt[0][i] * gt[1][j];
                            }
                        }
                        else
                        {
                            v[0] = wt[MF::SLOT][sl];
                            v[1] = gt[MF::SLOT][sl];
                        }
                        if constexpr ( TL::PAIR )
                        {
                            v[TL::val( 0 )] = P[sl];
                            if constexpr ( NT == 2 && sl < 3 )
                                slot_values<FL::v[FL::N - 1]>( P + 4, sl, v + TL::val( 1 ) );
                        }
                        else
                            static_for<FL::N>( [&]( auto I ) {
                                constexpr int t = I;
                                constexpr int F = FL::v[t];
                                if constexpr ( sl < ng_of( F ) )
                                    slot_values<F>( P + attr_of<FORMS...>( t ), sl,
                                                    v + TL::val( 0 ) + ( SHARED && t == 1 ? 1 : 0 ) );
                            } );
                        RC::put_row( rp, sl, v );
                    } );
                }
                __builtin_amdgcn_fence( __ATOMIC_ACQ_REL, "wavefront" );
                __builtin_amdgcn_wave_barrier();
                // The next batch's reads complete while the last records
                // accumulate (issued here, where this batch's registers are
                // free).
                if constexpr ( s0 + SUB == 64 )
                    batch_issue<Real, CONTIG, FORMS...>( a, ta, run_start, run_pre, vb + 64 + lane,
                                                         v1, run, bt );
                const int s1 = min( s0 + SUB, nb );
                int s = s0;
                while ( s < s1 )
                {
                    const uint64_t rest = s < 63 ? starts >> ( s + 1 ) : 0;
                    const int e = rest ? min( s1, s + 1 + __builtin_ctzll( rest ) ) : s1;
                    const int gk = __builtin_amdgcn_readlane( skey, s );
                    if ( gk < 0 )
                    {
                        s = e;
                        continue;
                    }
                    // The group's window: the open one, or the next along k
                    // (one node leaves the accumulators), or a new one.
                    if ( gk != open )
                    {
                        if ( open >= 0 )
                            retire( open, !( SLIDE && gk == open + 1 ) );
                        open = gk;
                    }
                    int n = e - s;
                    const Real* rp = rec + ( s - s0 + pslot ) * RS;
                    s = e;
                    while ( n > 0 )
                    {
                        // A chunk of one to four steps.  FP32 products are
                        // summed over 8 particles at most for a value-type tile
                        // and over 16 for a gradient-type one, its three kinds
                        // apart, and the sums added in FP64.  (Linear splines
                        // sum the three kinds in one chain, but a lane's chain
                        // is of one particle a step, 12 products at most.)
                        // KINDS is how the kinds of an FP32 gradient-type tile
                        // are summed: 0 apart, 1 in one chain (groups of up to
                        // four: 12 products), 2 in two chains added in FP64
                        // (the same in thin clouds, where such groups are all
                        // there is).  Relative L2 errors, 64^3 cells,
                        // quadratic, of the kernel before this one and of this
                        // one, e-8: momentum at 2, 8, 16 particles a cell 8.87
                        // 9.71 10.3 and 8.84 9.60 9.70; stress divergence at 2,
                        // 4, 8, 16: 9.44 10.0 10.6 11.3 and 9.23 10.0 10.5 11.1
                        // (one chain at 2 a cell: 9.71; two cost the adjoint
                        // 8 us of 98 there).
                        // Each count of steps is code of its own, without
                        // branches, so that its operand reads are issued
                        // together: 1.87 -> 1.62 ms against a loop that read a
                        // step ahead.
                        auto chunk = [&]( auto STEPS, auto KINDS ) {
                            constexpr int NS = STEPS;
                            constexpr int kinds = ORDER == 1 ? 1 : KINDS;
                            V4 D[NT][3];
                            Step<Real, ROW> st[NS];
                            static_for<NS>( [&]( auto C ) {
                                constexpr int c = C;
                                const Real* r = rp + 4 * c * RS;
                                if constexpr ( ORDER == 1 )
                                    RC::get_pair( r + 2 * kcol, st[c].xz, st[c].gz );
                                else
                                    st[c].xz = r[l16];
                                RC::get_row( r, slot, st[c].y );
                            } );
                            __builtin_amdgcn_sched_barrier( 0 );
                            static_for<NS>( [&]( auto C ) {
                                constexpr int c = C;
                                Real wz, gz, A1, AQ, AS;
                                // Particles past the group count zero.
                                const bool in = c < NS - 1 || pslot < n - 4 * c;
                                const Real xz = in ? st[c].xz : Real( 0 );
                                if constexpr ( ORDER == 1 )
                                {
                                    wz = xz;
                                    gz = in ? st[c].gz : Real( 0 );
                                    A1 = st[c].y[0];
                                    if constexpr ( TL::any_g() )
                                    {
                                        AQ = st[c].y[1];
                                        AS = st[c].y[2];
                                    }
                                }
                                else
                                {
                                    const Real wq = quad_lane<0>( xz ), gq = quad_lane<1>( xz );
                                    wz = quad_lane<2>( xz );
                                    gz = quad_lane<3>( xz );
                                    A1 = wq * st[c].y[0];
                                    AQ = gq * st[c].y[0];
                                    AS = wq * st[c].y[1];
                                }
                                static_for<NT>( [&]( auto T ) {
                                    constexpr int t = T;
                                    constexpr int m1 = F32 && kinds > 0 ? 0 : 1;
                                    constexpr int m2 = F32 ? ( kinds == 1 ? 0 : 2 ) : ( ORDER > 1 ? 1 : 2 );
                                    constexpr int dq = ORDER > 1 ? MF::QUAD : 0;
                                    constexpr int ds = ORDER > 1 ? MF::SLOT : 1;
                                    const Real* v = st[c].y + TL::val( t );
                                    const Real* h = v + ( TL::has_v( t ) ? 1 : 0 );
                                    if constexpr ( c == 0 )
                                        D[t][0] = D[t][1] = D[t][2] = V4{ 0, 0, 0, 0 };
                                    auto mac = [&]( Real A, Real B, V4& d ) {
                                        if constexpr ( ORDER == 1 )
                                            d = mac4( A, B, d );
                                        else
                                            d = MF::mac( A, B, d );
                                    };
                                    if constexpr ( !TL::has_g( t ) )
                                        mac( A1, wz * v[0], D[t][F32 ? c / 2 : 0] );
                                    else
                                    {
                                        Real b1 = gz * h[2];
                                        if constexpr ( TL::has_v( t ) )
                                            b1 += wz * v[0];
                                        mac( A1, b1, D[t][0] );
                                        mac( AQ, wz * h[dq], D[t][m1] );
                                        mac( AS, wz * h[ds], D[t][m2] );
                                    }
                                } );
                            } );
                            static_for<NT>( [&]( auto T ) {
                                constexpr int t = T;
#pragma unroll
                                for ( int r = 0; r < NR; ++r )
                                    if constexpr ( !F32 && !TL::has_g( t ) )
                                        // (Chunks summed apart: one chain over all
                                        // groups of a window measured up to 1.2
                                        // times the error.)
                                        acc[t][r] += D[t][0][r];
                                    else if constexpr ( !F32 && ORDER > 1 )
                                        acc[t][r] += D[t][0][r] + D[t][1][r];
                                    else if constexpr ( !F32 )
                                        acc[t][r] += ( D[t][0][r] + D[t][1][r] ) + D[t][2][r];
                                    else if constexpr ( TL::has_g( t ) && kinds == 0 )
                                        acc[t][r] +=
                                            (double)( ( D[t][0][r] + D[t][1][r] ) + D[t][2][r] );
                                    else if constexpr ( TL::has_g( t ) && kinds == 2 )
                                        acc[t][r] += (double)D[t][0][r] + (double)D[t][2][r];
                                    else if constexpr ( !TL::has_g( t ) && NS > 2 )
                                        acc[t][r] += (double)D[t][0][r] + (double)D[t][1][r];
                                    else
                                        acc[t][r] += (double)D[t][0][r];
                            } );
                        };
                        using std::integral_constant;
                        if ( MAX_STEPS == 4 && n > 12 )
                            chunk( integral_constant<int, 4>{}, integral_constant<int, 0>{} );
                        else if ( MAX_STEPS == 4 && n > 8 )
                            chunk( integral_constant<int, 3>{}, integral_constant<int, 0>{} );
                        else if ( n > 4 )
                            chunk( integral_constant<int, 2>{}, integral_constant<int, 0>{} );
                        else if ( F32 && TL::any_g() && ORDER > 1 && ta.thin )
                            chunk( integral_constant<int, 1>{}, integral_constant<int, 2>{} );
                        else
                            chunk( integral_constant<int, 1>{}, integral_constant<int, 1>{} );
                        n -= 4 * MAX_STEPS;
                        rp += 4 * MAX_STEPS * RS;
                    }
                }
                // The records are rewritten by the next sub-batch.
                __builtin_amdgcn_fence( __ATOMIC_ACQ_REL, "wavefront" );
                __builtin_amdgcn_wave_barrier();
            } );
        }
        if ( open >= 0 )
            retire( open, true );
        __syncthreads();

        // Flush the window, one thread per node (the grid's unit-stride
        // dimension fastest across threads): the node's dofs are read and
        // zeroed for the next part, and every non-zero value is added to its
        // grid with one global atomic.
        const float rW[3] = { 1.0f / (float)W[0], 1.0f / (float)W[1], 1.0f / (float)W[2] };
        for ( int f = threadIdx.x; f < wnodes; f += SCATTER_BLOCK )
        {
            int q[3], d0;
            window_coords<1>( ta, f, W, rW, q, d0 );
            const int node = ( q[0] * W[1] + q[1] ) * W[2] + q[2];
            const int gi = wlo[0] + q[0], gj = wlo[1] + q[1], gk = wlo[2] + q[2];
            const bool in = gi >= 0 && gj >= 0 && gk >= 0 && gi < a.mesh.num_node[0] &&
                            gj < a.mesh.num_node[1] && gk < a.mesh.num_node[2];
            int wo = 0;
            static_for<NT>( [&]( auto T ) {
                constexpr int t = T;
                constexpr int ND = TL::nd( t );
                double* src = win + ( wo + node * ND );
                wo += ta.max_win_nodes * ND;
                double v[ND];
#pragma unroll
                for ( int d = 0; d < ND; ++d )
                {
                    v[d] = src[d];
                    src[d] = 0.0;
                }
                if ( in )
                    static_for<ND>( [&]( auto D ) {
                        constexpr int d = D;
                        constexpr bool vec = TL::PAIR && t == 0 && d > 0;
                        const GFieldDev& g = a.t[vec ? 1 : TL::first_term( t )].grid;
                        const Real x = (Real)v[d];
                        if ( x != Real( 0 ) )
                            atomic_add( gptr<Real>( g, gi * g.s[0] + gj * g.s[1] + gk * g.s[2] +
                                                           ( vec ? d - 1 : d ) * g.s[3] ),
                                        x );
                    } );
            } );
        }
        // The next part reuses the window and the run table.
        __syncthreads();
    }
}

template <int F>
constexpr int single_sub()
{
    return scatter_sub( false, ORDER, Tiles<false, F>::any_g(), 1, 0.0 );
}

template <class Real, bool CONTIG>
hipError_t scatter_cells_launch( int plan, const ScatterArgs& a, const TileArgs& t, size_t lds,
                                 hipStream_t s )
{
    if ( plan == PLAN_SINGLE )
    {
        switch ( a.t[0].form )
        {
#define CA_CASE( F )                                                           \
    case F:                                                                    \
        return launch_tile_kernel( scatter_cells_kernel<Real, CONTIG, false, single_sub<F>(), F>, a, t, lds, s, SCATTER_BLOCK );
            CA_CASE( FORM_SV )
            CA_CASE( FORM_VV )
            CA_CASE( FORM_SG )
            CA_CASE( FORM_VD )
            CA_CASE( FORM_TD )
            CA_CASE( FORM_TDT )
#undef CA_CASE
        default:
            return hipErrorInvalidValue;
        }
    }
    if ( plan == PLAN_MPM_P2G )
    {
        if constexpr ( ORDER > 1 )
            if ( t.sub == 16 )
                return launch_tile_kernel(
                    scatter_cells_kernel<Real, CONTIG, false, 16, FORM_SV, FORM_VV, FORM_TD>, a, t,
                    lds, s, SCATTER_BLOCK );
        return launch_tile_kernel(
            scatter_cells_kernel<Real, CONTIG, false, 32, FORM_SV, FORM_VV, FORM_TD>, a, t, lds, s,
            SCATTER_BLOCK );
    }
    if ( plan == PLAN_MASS_MOMENTUM )
        return launch_tile_kernel( scatter_cells_kernel<Real, CONTIG, false, 16, FORM_SV, FORM_VV>,
                                   a, t, lds, s, SCATTER_BLOCK );
    if ( plan == PLAN_MPM_G2P )
        return launch_tile_kernel( scatter_cells_kernel<Real, CONTIG, true, 32, FORM_VV, FORM_TDT>,
                                   a, t, lds, s, SCATTER_BLOCK );
    return hipErrorInvalidValue;
}

template <class Real>
hipError_t scatter_cells_typed( Launcher& L, int plan, const ScatterArgs& a,
                                const TileArgs& t, size_t lds, hipStream_t s )
{
    const char* name = plan == PLAN_MPM_P2G         ? "p2g_mpm_cells"
                       : plan == PLAN_MPM_G2P       ? "g2p_adjoint_mpm_cells"
                       : plan == PLAN_MASS_MOMENTUM ? "p2g_mass_momentum_cells"
                                                    : "scatter_cells";
    L.before( name, s );
    const hipError_t e = a.contig ? scatter_cells_launch<Real, true>( plan, a, t, lds, s )
                                  : scatter_cells_launch<Real, false>( plan, a, t, lds, s );
    L.after( name, s );
    return e;
}

} // namespace

hipError_t CA_CAT( launch_scatter_cells_, CA_SUFFIX )( Launcher& L, bool fp64,
                                                      int plan,
                                                      const ScatterArgs& a,
                                                      const TileArgs& t,
                                                      size_t lds, hipStream_t s )
{
    return fp64 ? scatter_cells_typed<double>( L, plan, a, t, lds, s )
                : scatter_cells_typed<float>( L, plan, a, t, lds, s );
}

} // namespace cabana_amd
