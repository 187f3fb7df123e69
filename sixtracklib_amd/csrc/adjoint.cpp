// C API of the differentiable tracker (include/sixtracklib_amd/adjoint.h):
// argument checks and dispatch to the _exact / _fma kernel builds.
#include <hip/hip_runtime.h>

#include <cstring>
#include <string>
#include <vector>

#include "sixtracklib_amd/adjoint.h"
#include "adjoint_launch.h"
#include "lattice_hot.h"

extern "C" void st_internal_set_error( char const* msg );

namespace
{
bool valid( const st_adj_problem_t* p )
{
    if( p == nullptr || p->lat == nullptr || p->rec_off == nullptr || p->mp_index == nullptr ||
        p->target == nullptr || p->ckpt == nullptr || p->n_elem <= 0 || p->K <= 0 ||
        p->n_turns <= 0 || p->n < 0 || p->n >= ( int64_t )1 << 31 )
    {
        st_internal_set_error( "adjoint: invalid problem description" );
        return false;
    }
    return true;
}

// the part of a plan that NS(Adjoint_coefficients) uses
bool valid_multipoles( const st_adj_plan_t* p )
{
    if( p == nullptr || p->lat == nullptr || p->hot == nullptr ||
        p->n_mp < 0 || p->max_order < 0 || p->max_order > ST_ADJ_MAX_ORDER ||
        ( p->n_mp > 0 && ( p->mp_order == nullptr || p->mp_lat == nullptr || p->mp_hot == nullptr ) ) )
    {
        st_internal_set_error( "adjoint: invalid plan" );
        return false;
    }
    return true;
}

bool valid_plan( const st_adj_plan_t* p )
{
    if( !valid_multipoles( p ) || !valid( &p->base ) ) return false;
    if( p->segments == nullptr )
    {
        st_internal_set_error( "adjoint: invalid plan" );
        return false;
    }
    return true;
}

int done( hipError_t e, const char* what )
{
    if( e == hipSuccess ) return 0;
    std::string m = std::string( what ) + ": " + hipGetErrorString( e );
    st_internal_set_error( m.c_str() );
    return -1;
}
}  // namespace

extern "C" {

int64_t NS(Adjoint_checkpoint_doubles)( const st_adj_problem_t* p )
{
    if( p == nullptr || p->K <= 0 ) return -1;
    int64_t const n_seg = ( p->n_elem + p->K - 1 ) / p->K;
    return p->n_turns * n_seg * 9 * p->n;
}

int64_t NS(Adjoint_segment_doubles)( const st_adj_problem_t* p )
{
    if( p == nullptr || p->K <= 0 ) return -1;
    return p->K * 9 * p->n;
}

int NS(Adjoint_forward)( const st_adj_problem_t* p, int fma, const double* coords, double* loss,
    int32_t* status, void* stream )
{
    if( !valid( p ) || coords == nullptr || loss == nullptr || status == nullptr ) return -1;
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_forward_fma( p, coords, loss, status, s )
                     : st_launch_adj_forward_exact( p, coords, loss, status, s ), "adjoint forward" );
}

int NS(Adjoint_backward_turn)( const st_adj_problem_t* p, int fma, int64_t turn,
    const double* grad_out, double* segbuf, double* coef, double* cot, void* stream )
{
    if( !valid( p ) || turn < 0 || turn >= p->n_turns || grad_out == nullptr ||
        segbuf == nullptr || coef == nullptr || cot == nullptr )
    {
        st_internal_set_error( "adjoint backward: invalid arguments" );
        return -1;
    }
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_backward_turn_fma( p, turn, grad_out, segbuf, coef, cot, s )
                     : st_launch_adj_backward_turn_exact( p, turn, grad_out, segbuf, coef, cot, s ),
                 "adjoint backward" );
}

int NS(Adjoint_reduce_coefficients)( const st_adj_problem_t* p, int fma, const int32_t* mp_order,
    int64_t n_mp, const double* coef, double* grad_bal, int64_t stride, void* stream )
{
    if( !valid( p ) || mp_order == nullptr || coef == nullptr || grad_bal == nullptr ||
        stride < 2 * ST_ADJ_MAX_ORDER + 2 )
    {
        st_internal_set_error( "adjoint reduce: invalid arguments (stride >= 22)" );
        return -1;
    }
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_reduce_fma( p, mp_order, n_mp, coef, grad_bal, stride, s )
                     : st_launch_adj_reduce_exact( p, mp_order, n_mp, coef, grad_bal, stride, s ),
                 "adjoint reduce" );
}

int64_t NS(Adjoint_hot_size)( const uint64_t* lat )
{
    return lat == nullptr ? -1 : ( int64_t )st::hot_stream( lat ).size();
}

int NS(Adjoint_hot_build)( const uint64_t* lat, int64_t K, uint64_t* hot, int64_t hot_words,
    st_adj_segment_t* segments, int64_t n_segments, uint32_t* mp_hot, int64_t n_mp )
{
    if( lat == nullptr || K <= 0 || hot == nullptr || segments == nullptr ) return -1;
    st::HotMap map;
    std::vector< uint64_t > const h = st::hot_stream( lat, &map );
    int64_t const n_elem = ( int64_t )map.off.size() - 1;
    if( ( int64_t )h.size() != hot_words || n_segments != ( n_elem + K - 1 ) / K ) return -1;
    std::memcpy( hot, h.data(), h.size() * sizeof( uint64_t ) );
    std::vector< uint32_t > at( n_elem + 1 );               // packed records, byte offsets
    int64_t m = 0;
    uint32_t pos = 0;
    for( int64_t e = 0; e < n_elem; ++e )
    {
        uint64_t const r = lat[ pos / 8u ];
        at[ e ] = pos;
        pos += ST_REC_BYTES( r );
        if( ST_REC_OP( r ) != ST_OP_MULTIPOLE ) continue;
        if( m >= n_mp || mp_hot == nullptr || ST_REC_AUX( r ) > ST_ADJ_MAX_ORDER ) return -1;
        // behind word 0, or behind the Drift's length
        uint32_t const first = map.off[ e ] / 8u + ( ( map.off[ e ] & 1u ) ? 2u : 1u );
        mp_hot[ m++ ] = first + 2u * ST_REC_AUX( r );       // highest order first
    }
    if( m != n_mp ) return -1;
    for( int64_t j = 0; j < n_segments; ++j )
    {
        int64_t const b = j * K, e = b + K < n_elem ? b + K : n_elem;
        st_adj_segment_t s{};
        int64_t first = b;
        if( map.off[ b ] & 1u ) { s.head = at[ b ] + 1u; ++first; }
        s.off = map.off[ first ] & ~1u;
        s.next = map.handler[ first ];
        s.stop = map.off[ e ] & ~1u;
        if( first == e ) s.stop = s.off;
        else if( map.off[ e ] & 1u ) s.tail = at[ e - 1 ] + 1u;
        segments[ j ] = s;
    }
    return 0;
}

int NS(Adjoint_coefficients)( const st_adj_plan_t* p, int fma, const double* knl, const double* ksl,
    int scaled, void* stream )
{
    if( !valid_multipoles( p ) || ( p->n_mp > 0 && ( knl == nullptr || ksl == nullptr ) ) ) return -1;
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_coefficients_fma( p, knl, ksl, scaled, s )
                     : st_launch_adj_coefficients_exact( p, knl, ksl, scaled, s ), "adjoint coefficients" );
}

int NS(Adjoint_loss)( const st_adj_plan_t* p, int fma, const double* coords, double* loss,
    int32_t* status, void* stream )
{
    if( !valid_plan( p ) || coords == nullptr || loss == nullptr || status == nullptr ) return -1;
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_loss_fma( p, coords, loss, status, s )
                     : st_launch_adj_loss_exact( p, coords, loss, status, s ), "adjoint loss" );
}

int64_t NS(Adjoint_gradient_doubles_within)( const st_adj_plan_t* p, int64_t max_doubles )
{
    if( p == nullptr || p->base.n < 0 || p->base.n_elem <= 0 || p->base.K <= 0 || p->n_mp < 0 ||
        p->max_order < 0 ) return -1;
    return st_adj_work_doubles( p, st_adj_group( p, max_doubles ) );
}

int64_t NS(Adjoint_gradient_doubles)( const st_adj_plan_t* p )
{
    return NS(Adjoint_gradient_doubles_within)( p, INT64_MAX );
}

int NS(Adjoint_gradients_within)( const st_adj_plan_t* p, int fma, const double* grad_out, double* work,
    int64_t work_doubles, double* grad_coords, double* grad_knl, double* grad_ksl, void* stream )
{
    if( !valid_plan( p ) || grad_out == nullptr || work == nullptr || grad_coords == nullptr ||
        ( p->n_mp > 0 && ( grad_knl == nullptr || grad_ksl == nullptr ) ) )
    {
        st_internal_set_error( "adjoint gradients: invalid arguments" );
        return -1;
    }
    int64_t const group = st_adj_group( p, work_doubles );
    if( work_doubles < st_adj_work_doubles( p, group ) )
    {
        st_internal_set_error( "adjoint gradients: not enough work memory" );
        return -1;
    }
    hipStream_t const s = static_cast< hipStream_t >( stream );
    return done( fma ? st_launch_adj_gradients_fma( p, grad_out, work, group, grad_coords, grad_knl, grad_ksl, s )
                     : st_launch_adj_gradients_exact( p, grad_out, work, group, grad_coords, grad_knl, grad_ksl, s ),
                 "adjoint gradients" );
}

int NS(Adjoint_gradients)( const st_adj_plan_t* p, int fma, const double* grad_out, double* work,
    double* grad_coords, double* grad_knl, double* grad_ksl, void* stream )
{
    return NS(Adjoint_gradients_within)( p, fma, grad_out, work, INT64_MAX, grad_coords, grad_knl, grad_ksl, stream );
}

}  // extern "C"
