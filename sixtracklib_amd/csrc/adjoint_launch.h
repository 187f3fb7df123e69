// Differentiable tracking: problem descriptor and kernel launchers
// (library-internal; the C API is include/sixtracklib_amd/adjoint.h).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sixtracklib_amd/adjoint.h"

// largest multipole order the coefficient reduction handles
#define ST_ADJ_MAX_ORDER 10

#define ST_DECLARE_ADJ_LAUNCHERS( SUF )                                                   \
    extern "C" hipError_t st_launch_adj_forward##SUF( const st_adj_problem_t* p,         \
        const double* coords, double* loss, int32_t* status, hipStream_t stream );        \
    extern "C" hipError_t st_launch_adj_backward_turn##SUF( const st_adj_problem_t* p,   \
        int64_t turn, const double* grad_out, double* segbuf, double* coef, double* cot, \
        hipStream_t stream );                                                             \
    extern "C" hipError_t st_launch_adj_reduce##SUF( const st_adj_problem_t* p,          \
        const int32_t* mp_order, int64_t n_mp, const double* coef, double* grad_bal,      \
        int64_t stride, hipStream_t stream );                                             \
    extern "C" hipError_t st_launch_adj_coefficients##SUF( const st_adj_plan_t* p,       \
        const double* knl, const double* ksl, int scaled, hipStream_t stream );           \
    extern "C" hipError_t st_launch_adj_loss##SUF( const st_adj_plan_t* p,               \
        const double* coords, double* loss, int32_t* status, hipStream_t stream );        \
    extern "C" hipError_t st_launch_adj_gradients##SUF( const st_adj_plan_t* p,          \
        const double* grad_out, double* work, int64_t group, double* grad_coords,         \
        double* grad_knl, double* grad_ksl, hipStream_t stream );

// Reverse pass (adjoint_kernels.hip): elements of a piece and of the part of
// it whose states are in LDS at a time, doubles of a kept state; the particle
// count up to which the pieces of a group of turns run side by side, and the
// bytes that may take.
#define ST_ADJ_PIECE 64
#define ST_ADJ_SUB 8
#define ST_ADJ_STATE 8
#define ST_ADJ_PARALLEL_MAX 65536
#define ST_ADJ_PARALLEL_BYTES ( int64_t( 1 ) << 32 )

static inline int64_t st_adj_pieces( const st_adj_plan_t* p )
{ return ( p->base.n_elem + ST_ADJ_PIECE - 1 ) / ST_ADJ_PIECE; }
static inline int64_t st_adj_tiles( const st_adj_plan_t* p ) { return ( p->base.n + 63 ) / 64; }
static inline int64_t st_adj_parts( const st_adj_plan_t* p )
{ return ( p->base.n_elem + ST_ADJ_SUB - 1 ) / ST_ADJ_SUB; }
// units whose parts' first states a wave makes: the ranges of the checkpoints,
// or the pieces where K is smaller
static inline int64_t st_adj_units( const st_adj_plan_t* p )
{ return p->base.K > ST_ADJ_PIECE ? ( p->base.n_elem + p->base.K - 1 ) / p->base.K : st_adj_pieces( p ); }
static inline int64_t st_adj_row_doubles( const st_adj_plan_t* p )
{ return p->n_mp * 2 * ( p->max_order + 1 ); }
// work, pieces of a group of turns side by side: Jacobians
// [group][piece][36][64 tiles], end and start cotangents
// [group][piece][6][64 tiles] each, first states of parts
// [group][part][8][64 tiles], partial sums [group][tiles][row];
// one wave through all pieces: first states of the parts of one unit, partial
// sums [tiles][row]
static inline int64_t st_adj_turn_doubles( const st_adj_plan_t* p )
{
    return st_adj_tiles( p ) * ( 64 * ( st_adj_pieces( p ) * ( 36 + 6 + 6 ) + st_adj_parts( p ) * ST_ADJ_STATE ) +
                                 st_adj_row_doubles( p ) );
}
static inline int64_t st_adj_unit_doubles( const st_adj_plan_t* p )
{
    int64_t const unit = p->base.K > ST_ADJ_PIECE ? p->base.K : ST_ADJ_PIECE;
    int64_t const range = unit < p->base.n_elem ? unit : p->base.n_elem;
    return st_adj_tiles( p ) * ( 64 * ( ( range + ST_ADJ_SUB - 1 ) / ST_ADJ_SUB ) * ST_ADJ_STATE +
                                 st_adj_row_doubles( p ) );
}
// turns whose pieces run side by side with at most ``doubles`` of work; 0: one
// wave goes through all pieces
static inline int64_t st_adj_group( const st_adj_plan_t* p, int64_t doubles )
{
    if( p->base.n > ST_ADJ_PARALLEL_MAX || p->base.n <= 0 || doubles < 0 ) return 0;
    int64_t const most = ST_ADJ_PARALLEL_BYTES / 8;
    int64_t const g = ( doubles < most ? doubles : most ) / st_adj_turn_doubles( p );
    return g < p->base.n_turns ? g : p->base.n_turns;
}
static inline int64_t st_adj_work_doubles( const st_adj_plan_t* p, int64_t group )
{ return group > 0 ? group * st_adj_turn_doubles( p ) : st_adj_unit_doubles( p ); }

ST_DECLARE_ADJ_LAUNCHERS( _exact )
ST_DECLARE_ADJ_LAUNCHERS( _fma )
