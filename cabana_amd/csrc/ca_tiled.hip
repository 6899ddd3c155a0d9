// Cell-tiled gathers of cell-sorted particles, one spline order per
// translation unit (CA_ORDER set on the compile line): G2P forward, the P2G
// adjoint and the position part of the G2P adjoint.  The node window of every
// grid the pass reads is staged in LDS with coalesced loads; every particle
// then gathers its K^3 stencil from LDS.
#include "ca_tiles.hpp"

namespace cabana_amd
{
namespace
{

// ---------------------------------------------------------------------------
// Tiled gather
// ---------------------------------------------------------------------------

// Waves per SIMD the register allocation of a gather must leave room for:
// three for the FP32 passes that read their inputs late (more than three
// terms; their LDS windows allow four), no bound otherwise.
template <class Real, int... FORMS>
constexpr int gather_min_waves()
{
    return ( sizeof( Real ) == 4 && GatherNeeds<FORMS...>::late() ) ? 3 : 1;
}

template <class Real, int MODE, bool CONTIG, bool SHARED, int... FORMS>
__global__ __launch_bounds__( BLOCK, ( gather_min_waves<Real, FORMS...>() ) ) void gather_tiled_kernel(
    GatherArgs a, TileArgs ta )
{
    using GN = GatherNeeds<FORMS...>;
    constexpr int NSLOT = GN::nslot( SHARED );
    extern __shared__ __align__( 16 ) unsigned char smem[];

    // LDS: one staged window per grid slot (3-dof slots padded to 4), then
    // the run table (capacities of a full brick).
    Real* win[NSLOT];
    size_t off = 0;
    static_for<NSLOT>( [&]( auto I ) {
        constexpr int sl = I;
        win[sl] = reinterpret_cast<Real*>( smem + off );
        off = align16( off + sizeof( Real ) * ta.max_win_nodes *
                                 ( GN::NG( sl, SHARED ) == 1 ? 1 : 4 ) );
    } );
    int64_t* run_start = reinterpret_cast<int64_t*>( smem + off );
    int* run_pre = reinterpret_cast<int*>( run_start + ta.max_runs );

    const PartLoop pl( ta );
    for ( int loc = pl.first; pl.more( loc ); loc += pl.stride )
    {
        const int w = pl.part( loc );
        if ( w < 0 )
            continue;
        TileGeom tg;
        part_geometry( ta, a.mesh, w, tg );
        int wlo[3], W[3];
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            wlo[d] = tg.c0[d] + a.mesh.halo + BASE_SHIFT;
            W[d] = ta.win[d];
        }
        const int wnodes = W[0] * W[1] * W[2];
        const float rW[3] = { 1.0f / (float)W[0], 1.0f / (float)W[1], 1.0f / (float)W[2] };

        // Stage the windows (nodes outside the grid read as zero).
        static_for<NSLOT>( [&]( auto I ) {
            constexpr int sl = I;
            constexpr int NG = GN::NG( sl, SHARED );
            constexpr int NGP = NG == 1 ? 1 : 4;
            const GFieldDev& g = a.t[GN::first_term( sl, SHARED )].grid;
            Real* wp = win[sl];
            for ( int f = threadIdx.x; f < wnodes * NG; f += BLOCK )
            {
                int q[3], d;
                window_coords<NG>( ta, f, W, rW, q, d );
                const int gi = wlo[0] + q[0], gj = wlo[1] + q[1], gk = wlo[2] + q[2];
                Real v = Real( 0 );
                if ( gi >= 0 && gj >= 0 && gk >= 0 && gi < a.mesh.num_node[0] &&
                     gj < a.mesh.num_node[1] && gk < a.mesh.num_node[2] )
                    v = *gptr<const Real>( g, gi * g.s[0] + gj * g.s[1] + gk * g.s[2] +
                                                  d * g.s[3] );
                wp[( ( q[0] * W[1] + q[1] ) * W[2] + q[2] ) * NGP + d] = v;
            }
        } );
        const int nruns = ( tg.c1[0] - tg.c0[0] ) * ( tg.c1[1] - tg.c0[1] );
        const int total = setup_runs( ta, a.mesh, tg, run_start, run_pre );
        const int pbeg = tg.part * ta.cap;
        const int pend = min( total, pbeg + ta.cap );

        // Lanes stride through the part; the cell run of the next particle
        // is found by walking forward, and its position and other global
        // reads are issued one iteration ahead, so their latency overlaps
        // the current particle's stencil work.
        using In = GatherIn<Real, MODE, FORMS...>;
        int v = pbeg + (int)threadIdx.x;
        int r = 0;
        int64_t p = 0;
        double px[3] = { 0.0, 0.0, 0.0 };
        In in;
        if ( v < pend )
        {
            r = find_run( run_pre, nruns, v );
            p = ta.particle( ta.bin_begin + run_start[r] + ( v - run_pre[r] ) );
            load_position<CONTIG>( a.points, p, px );
            gather_load<Real, MODE, CONTIG, FORMS...>( a, p, in );
        }
        while ( v < pend )
        {
            const int vn = v + BLOCK;
            int64_t pn = 0;
            double pxn[3] = { 0.0, 0.0, 0.0 };
            In inn;
            if ( vn < pend )
            {
                while ( run_pre[r + 1] <= vn )
                    ++r;
                pn = ta.particle( ta.bin_begin + run_start[r] + ( vn - run_pre[r] ) );
                load_position<CONTIG>( a.points, pn, pxn );
                gather_load<Real, MODE, CONTIG, FORMS...>( a, pn, inn );
            }
            Spline3D<ORDER, Real, mode_xbar( MODE )> s;
            if ( !eval_spline( a.mesh, px, s ) )
            {
                atomicAdd( a.skipped, 1ull );
            }
            else
            {
                int rel[3];
                bool fits = true;
#pragma unroll
                for ( int d = 0; d < 3; ++d )
                {
                    rel[d] = s.d[d].base - wlo[d];
                    fits = fits && rel[d] >= 0 && rel[d] + K <= W[d];
                }
                // Stencil nodes from the staged window.  A wave with a
                // particle whose stencil is outside the window (not sorted
                // into this brick) reads the grid directly for all of its
                // lanes, so the choice is one uniform branch, not one per
                // node.
                if ( __all( fits ) )
                {
                    const int nb = ( rel[0] * W[1] + rel[1] ) * W[2] + rel[2];
                    const int W1 = W[1], W2 = W[2];
                    auto ld = [&]( auto S, int i, int j, int k, Real* f ) {
                        constexpr int sl = decltype( S )::value;
                        constexpr int NG = GatherNeeds<FORMS...>::NG( sl, SHARED );
                        const int node = nb + ( i * W1 + j ) * W2 + k;
                        if constexpr ( NG == 1 )
                        {
                            f[0] = win[sl][node];
                        }
                        else
                        {
                            const Real* q = win[sl] + node * 4;
                            f[0] = q[0];
                            f[1] = q[1];
                            f[2] = q[2];
                        }
                    };
                    gather_compute<ORDER, Real, MODE, CONTIG, SHARED, FORMS...>( a, p, s, ld, in );
                }
                else
                {
                    GlobalGatherLoad<Real, SHARED, FORMS...> ld{
                        a, { s.d[0].base, s.d[1].base, s.d[2].base } };
                    gather_compute<ORDER, Real, MODE, CONTIG, SHARED, FORMS...>( a, p, s, ld, in );
                }
            }
            v = vn;
            p = pn;
#pragma unroll
            for ( int d = 0; d < 3; ++d )
                px[d] = pxn[d];
            in = inn;
        }
        // The next part restages the windows.
        __syncthreads();
    }
}
template <class Real, bool CONTIG>
hipError_t gather_tiled_launch( int plan, int mode, const GatherArgs& a, const TileArgs& t,
                                size_t lds, hipStream_t s )
{
    if ( plan == PLAN_SINGLE )
    {
        switch ( a.t[0].form )
        {
#define CA_CASE( F )                                                           \
    case F:                                                                    \
        return mode == GATHER_OUT                                              \
                   ? launch_tile_kernel( gather_tiled_kernel<Real, GATHER_OUT, CONTIG, false, F>, \
                                         a, t, lds, s )                        \
               : mode == GATHER_OUT_XBAR                                       \
                   ? launch_tile_kernel(                                       \
                         gather_tiled_kernel<Real, GATHER_OUT_XBAR, CONTIG, false, F>, a, t, \
                         lds, s )                                              \
                   : launch_tile_kernel( gather_tiled_kernel<Real, GATHER_XBAR, CONTIG, false, F>, \
                                         a, t, lds, s );
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
    if ( plan == PLAN_MPM_G2P && mode == GATHER_OUT )
        return launch_tile_kernel(
            gather_tiled_kernel<Real, GATHER_OUT, CONTIG, true, FORM_VV, FORM_TDT>, a, t, lds, s );
    if ( plan == PLAN_MPM_G2P && mode == GATHER_XBAR )
        return launch_tile_kernel(
            gather_tiled_kernel<Real, GATHER_XBAR, CONTIG, true, FORM_VV, FORM_TDT>, a, t, lds, s );
    if ( plan == PLAN_MPM_P2G && mode == GATHER_OUT_XBAR )
        return launch_tile_kernel(
            gather_tiled_kernel<Real, GATHER_OUT_XBAR, CONTIG, false, FORM_SV, FORM_VV, FORM_TD>,
            a, t, lds, s );
    if ( plan == PLAN_MPM_ADJOINT && mode == GATHER_OUT_XBAR )
        return launch_tile_kernel(
            gather_tiled_kernel<Real, GATHER_OUT_XBAR, CONTIG, false, FORM_SV, FORM_VV, FORM_TD,
                                FORM_VV | FORM_XONLY,
                                FORM_TDT | FORM_XONLY | FORM_SHARE_PREV>,
            a, t, lds, s );
    return hipErrorInvalidValue;
}

template <class Real>
hipError_t gather_tiled_typed( Launcher& L, int plan, const GatherArgs& a,
                               const TileArgs& t, size_t lds, hipStream_t s )
{
    const int mode = !a.has_xbar ? GATHER_OUT : ( a.t[0].pout.data ? GATHER_OUT_XBAR : GATHER_XBAR );
    const char* name =
        plan == PLAN_MPM_ADJOINT
            ? "adjoint_mpm_tiled"
            : a.has_xbar ? ( plan == PLAN_MPM_P2G ? "p2g_adjoint_mpm_tiled" : "gather_xbar_tiled" )
                         : ( plan == PLAN_MPM_G2P ? "g2p_mpm_tiled" : "g2p_tiled" );
    L.before( name, s );
    const hipError_t e = a.contig ? gather_tiled_launch<Real, true>( plan, mode, a, t, lds, s )
                                  : gather_tiled_launch<Real, false>( plan, mode, a, t, lds, s );
    L.after( name, s );
    return e;
}

} // namespace

hipError_t CA_CAT( launch_gather_tiled_, CA_SUFFIX )( Launcher& L, bool fp64,
                                                     int plan,
                                                     const GatherArgs& a,
                                                     const TileArgs& t,
                                                     size_t lds, hipStream_t s )
{
    return fp64 ? gather_tiled_typed<double>( L, plan, a, t, lds, s )
                : gather_tiled_typed<float>( L, plan, a, t, lds, s );
}

} // namespace cabana_amd
