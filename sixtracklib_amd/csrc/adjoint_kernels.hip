// Differentiable tracking: forward pass with checkpoints and per-turn
// reverse passes (gfx950; compiled twice like track_kernels.hip).
//
// No counterpart in the reference.  The forward pass runs the same element
// maps as the tracker (track_device.h) on one particle per lane; the loss
// is sum over turns t and coordinates c of w_c (X_c(t) - target_c(t))^2,
// X(t) the state at the end of turn t.  Every K elements of every turn the
// lane state is stored (checkpoint).  The reverse pass for turn t walks the
// turn's segments last to first: it recomputes a segment from its
// checkpoint, storing the state before each element, then applies the
// adjoint maps (adjoint_device.h) in reverse order.  Multipoles write
// (chi px_bar, chi py_bar, x, y) per particle; st_k_adj_reduce turns those
// into the gradient of every bal coefficient (one block per multipole).
//
// Memory layouts (n particles, structure of arrays so a wave's accesses are
// contiguous):
//   coords  [6][n]             x, px, y, py, zeta, delta
//   ckpt    [T][S][9][n]       lane state: the six above + rpp, rvv, psigma
//   segbuf  [K][9][n]          states before each element of one segment
//   coef    [M][4][n]          per multipole: chi px_bar, chi py_bar, x, y
//   cot     [6][n]             cotangent of the state (in / out per turn)
#include <hip/hip_runtime.h>

#include "track_device.h"
#include "adjoint_device.h"
#include "track_hot.h"
#include "adjoint_launch.h"

#ifndef ST_KSUFFIX
#error "ST_KSUFFIX (kernel name suffix of this build variant) must be defined"
#endif
#define ST_CAT2( a, b ) a##b
#define ST_CAT( a, b ) ST_CAT2( a, b )
#define KN( n ) ST_CAT( n, ST_KSUFFIX )

using namespace st;

namespace
{
typedef __attribute__( ( address_space( 4 ) ) ) const uint32_t cu32_t;
typedef __attribute__( ( address_space( 4 ) ) ) const int32_t ci32_t;

struct AdjArgs
{
    cptr_t lat;
    cu32_t* rec_off;         // word offset of element e's record
    int64_t n_elem, K, n_seg, n_turns, n;
    LaneConst C;
    double w[ 6 ];
    const double* target;    // [T][6]
    const double* coords;
    double* ckpt;
    double* loss;
    int32_t* status;
    int64_t turn;
    const double* grad_out;  // device scalar
    double* segbuf;
    ci32_t* mp_index;        // element -> multipole slot (-1: none)
    double* coef;
    double* cot;
};

ST_DEV void put_lane( double* b, int64_t n, int64_t i, const Lane& L )
{
    b[ 0 * n + i ] = L.x;    b[ 1 * n + i ] = L.px;   b[ 2 * n + i ] = L.y;
    b[ 3 * n + i ] = L.py;   b[ 4 * n + i ] = L.zeta; b[ 5 * n + i ] = L.delta;
    b[ 6 * n + i ] = L.rpp;  b[ 7 * n + i ] = L.rvv;  b[ 8 * n + i ] = L.psigma;
}

ST_DEV void get_lane( const double* b, int64_t n, int64_t i, Lane& L )
{
    L.x = b[ 0 * n + i ];    L.px = b[ 1 * n + i ];   L.y = b[ 2 * n + i ];
    L.py = b[ 3 * n + i ];   L.zeta = b[ 4 * n + i ]; L.delta = b[ 5 * n + i ];
    L.rpp = b[ 6 * n + i ];  L.rvv = b[ 7 * n + i ];  L.psigma = b[ 8 * n + i ];
    L.s = 0.0;
    L.state = 1;
}

// forward map of one record; returns the aperture predicate
ST_DEV bool apply( cptr_t r, Lane& L, const LaneConst& C )
{
    uint64_t const h = r[ 0 ];
    cptr_t const e = r + ST_REC_PAYLOAD;
    switch( ST_REC_OP( h ) )
    {
    case ST_OP_DRIFT: drift( L, rd( e, 0 ) ); return limit_global_ok( L );
    case ST_OP_MULTIPOLE: multipole( L, C.chi, e, ST_REC_AUX( h ), L.delta ); return true;
    case ST_OP_CAVITY: cavity( L, C, e ); return true;
    case ST_OP_XYSHIFT: xyshift( L, e ); return true;
    case ST_OP_SROTATION: srotation( L, e ); return true;
    case ST_OP_LIMIT_RECT: return limit_rect_ok( L, e );
    case ST_OP_LIMIT_ELLIPSE: return limit_ellipse_ok( L, e );
    case ST_OP_LIMIT_RECT_ELLIPSE: return limit_rect_ellipse_ok( L, e );
    default: return false;                   // excluded when the lattice is prepared
    }
}
}  // namespace

__global__ void __launch_bounds__( 256 ) KN( st_k_adj_forward )( AdjArgs a )
{
    int64_t const i = ( int64_t )blockIdx.x * blockDim.x + threadIdx.x;
    if( i >= a.n ) return;
    int64_t const n = a.n;
    Lane L;
    L.x = a.coords[ 0 * n + i ]; L.px = a.coords[ 1 * n + i ];
    L.y = a.coords[ 2 * n + i ]; L.py = a.coords[ 3 * n + i ];
    L.zeta = a.coords[ 4 * n + i ];
    update_delta( L, a.C, a.coords[ 5 * n + i ] );
    L.s = 0.0;
    L.state = 1;
    double loss = 0.0;
    bool ok = true;
    for( int64_t t = 0; t < a.n_turns; ++t )
    {
        for( int64_t e = 0; e < a.n_elem; ++e )
        {
            if( e % a.K == 0 ) put_lane( a.ckpt + ( ( t * a.n_seg + e / a.K ) * 9 ) * n, n, i, L );
            ok = apply( a.lat + a.rec_off[ e ], L, a.C ) && ok;
        }
        double const X[ 6 ] = { L.x, L.px, L.y, L.py, L.zeta, L.delta };
        for( int c = 0; c < 6; ++c )
        {
            double const d = X[ c ] - a.target[ t * 6 + c ];
            loss += a.w[ c ] * d * d;
        }
    }
    a.loss[ i ] = loss;
    if( !ok ) atomicOr( a.status, -1 );      // an aperture would have removed the particle
}

__global__ void __launch_bounds__( 256 ) KN( st_k_adj_backward_turn )( AdjArgs a )
{
    int64_t const i = ( int64_t )blockIdx.x * blockDim.x + threadIdx.x;
    if( i >= a.n ) return;
    int64_t const n = a.n, t = a.turn;
    double const g = *a.grad_out;
    Cot c;
    c.x = a.cot[ 0 * n + i ]; c.px = a.cot[ 1 * n + i ]; c.y = a.cot[ 2 * n + i ];
    c.py = a.cot[ 3 * n + i ]; c.zeta = a.cot[ 4 * n + i ]; c.delta = a.cot[ 5 * n + i ];
    for( int64_t j = a.n_seg - 1; j >= 0; --j )
    {
        Lane L;
        get_lane( a.ckpt + ( ( t * a.n_seg + j ) * 9 ) * n, n, i, L );
        int64_t const e0 = j * a.K;
        int64_t const e1 = ( e0 + a.K < a.n_elem ) ? e0 + a.K : a.n_elem;
        for( int64_t e = e0; e < e1; ++e )
        {
            put_lane( a.segbuf + ( ( e - e0 ) * 9 ) * n, n, i, L );
            ( void )apply( a.lat + a.rec_off[ e ], L, a.C );
        }
        if( j == a.n_seg - 1 )
        {
            // loss term of this turn: d/dX of w_c (X_c - target_c)^2
            c.x += g * 2.0 * a.w[ 0 ] * ( L.x - a.target[ t * 6 + 0 ] );
            c.px += g * 2.0 * a.w[ 1 ] * ( L.px - a.target[ t * 6 + 1 ] );
            c.y += g * 2.0 * a.w[ 2 ] * ( L.y - a.target[ t * 6 + 2 ] );
            c.py += g * 2.0 * a.w[ 3 ] * ( L.py - a.target[ t * 6 + 3 ] );
            c.zeta += g * 2.0 * a.w[ 4 ] * ( L.zeta - a.target[ t * 6 + 4 ] );
            c.delta += g * 2.0 * a.w[ 5 ] * ( L.delta - a.target[ t * 6 + 5 ] );
        }
        for( int64_t e = e1 - 1; e >= e0; --e )
        {
            cptr_t const r = a.lat + a.rec_off[ e ];
            uint64_t const h = r[ 0 ];
            cptr_t const prm = r + ST_REC_PAYLOAD;
            Lane P;
            get_lane( a.segbuf + ( ( e - e0 ) * 9 ) * n, n, i, P );
            switch( ST_REC_OP( h ) )
            {
            case ST_OP_DRIFT: drift_adj( P, rd( prm, 0 ), a.C.beta0, c ); break;
            case ST_OP_MULTIPOLE:
            {
                int64_t const m = a.mp_index[ e ];
                double* const cb = a.coef + ( m * 4 ) * n;
                cb[ 0 * n + i ] = a.C.chi * c.px;
                cb[ 1 * n + i ] = a.C.chi * c.py;
                cb[ 2 * n + i ] = P.x;
                cb[ 3 * n + i ] = P.y;
                multipole_adj( P, a.C.chi, prm, ( int )( ST_REC_AUX( h ) & 0x7fffu ), c );
                break;
            }
            case ST_OP_CAVITY: cavity_adj( P, a.C, prm, c ); break;
            case ST_OP_SROTATION: srotation_adj( prm, c ); break;
            default: break;                      // XYShift and apertures: identity
            }
        }
    }
    a.cot[ 0 * n + i ] = c.x; a.cot[ 1 * n + i ] = c.px; a.cot[ 2 * n + i ] = c.y;
    a.cot[ 3 * n + i ] = c.py; a.cot[ 4 * n + i ] = c.zeta; a.cot[ 5 * n + i ] = c.delta;
}

// One block per multipole m: grad_bal[m][2k] += sum_i (-cpx Re z^k + cpy Im z^k),
// grad_bal[m][2k+1] += sum_i (cpx Im z^k + cpy Re z^k), z = x + i y.
__global__ void __launch_bounds__( 256 ) KN( st_k_adj_reduce )( int64_t n,
    const int32_t* mp_order, const double* coef, double* grad_bal, int64_t stride )
{
    __shared__ double red[ 256 ];
    int64_t const m = blockIdx.x;
    int const order = mp_order[ m ];
    double acc[ 2 * ST_ADJ_MAX_ORDER + 2 ];
    for( int k = 0; k < 2 * ST_ADJ_MAX_ORDER + 2; ++k ) acc[ k ] = 0.0;
    const double* const cb = coef + ( m * 4 ) * n;
    for( int64_t i = threadIdx.x; i < n; i += blockDim.x )
    {
        double const cpx = cb[ 0 * n + i ], cpy = cb[ 1 * n + i ];
        double const x = cb[ 2 * n + i ], y = cb[ 3 * n + i ];
        double wr = 1.0, wi = 0.0;
#pragma unroll
        for( int k = 0; k <= ST_ADJ_MAX_ORDER; ++k )
        {
            if( k > order ) break;
            acc[ 2 * k ] += -cpx * wr + cpy * wi;
            acc[ 2 * k + 1 ] += cpx * wi + cpy * wr;
            double const nr = wr * x - wi * y;
            wi = wr * y + wi * x;
            wr = nr;
        }
    }
    for( int k = 0; k < 2 * order + 2; ++k )
    {
        red[ threadIdx.x ] = acc[ k ];
        __syncthreads();
        for( int s = blockDim.x / 2; s > 0; s >>= 1 )
        {
            if( ( int )threadIdx.x < s ) red[ threadIdx.x ] += red[ threadIdx.x + s ];
            __syncthreads();
        }
        if( threadIdx.x == 0 ) grad_bal[ m * stride + k ] += red[ 0 ];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------
// The same gradients for all turns in few launches.
//
// What bounds them: the particles of such a problem are few (a few thousand:
// 64 waves on 1,024 SIMDs), and the loop over elements x turns is a chain, so
// the forward pass above takes 390 ns per element and the reverse pass 960.
// Here
//   * the forward pass runs the scheduled record walk (track_hot.h), segment
//     by segment between checkpoints;
//   * the reverse pass is linear in the cotangent.  st_k_adj_jacobian forms
//     the transposed Jacobian of every piece of 64 elements of every turn,
//     all pieces side by side (six cotangents through the piece at once,
//     sharing its states and coefficients); st_k_adj_chain carries the
//     cotangent from piece to piece, 36 multiply-adds each.  Terms of those
//     products cancel, which leaves twice the rounding error of going element
//     by element; so st_k_adj_through goes through every piece so, side by
//     side, from the end cotangent found, and st_k_adj_chain_refine carries
//     on what each piece got wrong (error of the coordinates' gradients
//     against 80-bit arithmetic on the same states, 16 lattices: 4.2e-15
//     without, 1.78e-15 with this, turn by turn 1.83e-15).  st_k_adj_reverse
//     goes through every piece once more for the coefficient gradients.  Above
//     ST_ADJ_PARALLEL_MAX particles the waves fill the chip without that,
//     and st_k_adj_reverse alone goes through the pieces one after another;
//   * a piece's states are made from the checkpoints in parts of 8 elements,
//     the two coordinates each map's Jacobian needs kept in LDS (8 KB a wave;
//     with parts of 16 half as many waves fit a CU: 293 against 237 us for
//     st_k_adj_reverse, 168 and 127 for st_k_adj_through);
//   * the sums over particles are formed in the wave (DPP adds, a fixed
//     order) instead of through four values per particle and multipole.
// 4,096 particles, 1,000 elements, 10 turns, exact build: forward 3.9 -> 0.78
// ms, reverse 9.6 -> 0.75 ms (Jacobians 0.25, chain 0.05, through 0.13, its
// refinement 0.06, coefficients 0.23, sums 0.03).  Backward pass as called,
// before / now: 64 particles, 10 turns 7.2 / 0.36 ms, 16,384 and 10 turns
// 13.7 / 2.7.  Side by side costs three and a half sweeps instead of one and
// wins as long as the particles leave SIMDs idle: 2 turns, 65,536 particles
// side by side 2.3 ms, 70,000 with one wave through all pieces 2.7.
namespace
{
struct PlanArgs
{
    cptr_t lat, hot;
    cu32_t* rec_off;
    ci32_t* mp_index;
    cptr_t segments;             // st_adj_segment_t as three words each
    int64_t n_elem, K, n_seg, n_turns, n, n_mp;
    int32_t no;                  // max_order + 1
    int32_t tiles, pieces;
    int32_t t0, turns;           // turns [t0, t0 + turns) of this launch
    int32_t add;                 // partial sums are added to (not the first group)
    LaneConst C;
    double w[ 6 ];
    const double* target;
    double* ckpt;
    const double* grad_out;
    double *jac, *cend, *cstart, *partial, *grad_coords;
    double* states;              // first states of parts (state_slot)
    int64_t parts, units;
};

// sum over the 64 lanes, in lane 63, in a fixed order (rows of 16 by shifts,
// then the rows)
template< int CTRL, int ROWS >
ST_DEV double dpp_add( double v )
{
    int const lo = __builtin_amdgcn_update_dpp( 0, __double2loint( v ), CTRL, ROWS, 0xf, false );
    int const hi = __builtin_amdgcn_update_dpp( 0, __double2hiint( v ), CTRL, ROWS, 0xf, false );
    return v + __hiloint2double( hi, lo );
}

ST_DEV double wave_sum( double v )
{
    v = dpp_add< 0x111, 0xf >( v );
    v = dpp_add< 0x112, 0xf >( v );
    v = dpp_add< 0x114, 0xf >( v );
    v = dpp_add< 0x118, 0xf >( v );
    v = dpp_add< 0x142, 0xa >( v );
    v = dpp_add< 0x143, 0xc >( v );
    return v;
}

// Elements [b, e) forward; with SAVE the two coordinates the adjoint map of
// each needs go to lds[2 k], lds[2 k + 1] of element b + k (this lane's
// column): px, py of a Drift, x, y of a Multipole, zeta, delta of a Cavity.
template< bool SAVE >
ST_DEV void run_elements( const PlanArgs& a, int64_t b, int64_t e, Lane& L, double* lds )
{
    if( b >= e ) return;
    cptr_t r = a.lat + a.rec_off[ b ];
    uint64_t h = r[ 0 ];
    double* s = lds;
    for( int64_t k = b; k < e; ++k )
    {
        cptr_t const prm = r + ST_REC_PAYLOAD;
        cptr_t const nr = r + ST_REC_LEN( h );
        uint64_t const hn = nr[ 0 ];
        switch( ST_REC_OP( h ) )
        {
        case ST_OP_DRIFT:
            if( SAVE ) { s[ 0 ] = L.px; s[ 64 ] = L.py; }
            drift_xz( L, rd( prm, 0 ) );
            break;
        case ST_OP_MULTIPOLE:
            if( SAVE ) { s[ 0 ] = L.x; s[ 64 ] = L.y; }
            multipole( L, a.C.chi, prm, ST_REC_AUX( h ), L.delta );
            break;
        case ST_OP_CAVITY:
            if( SAVE ) { s[ 0 ] = L.zeta; s[ 64 ] = L.delta; }
            cavity( L, a.C, prm );
            break;
        case ST_OP_XYSHIFT: xyshift( L, prm ); break;
        case ST_OP_SROTATION: srotation( L, prm ); break;
        default: break;                           // apertures: checked by the forward pass
        }
        if( SAVE ) s += 128;
        r = nr;
        h = hn;
    }
}

// The kernels of the reverse pass go through pieces of 64 elements in parts of
// 16, the last first, and each part starts from its first state.  Those are
// made once from the checkpoints and kept (8 doubles a particle, N particles
// apart, part by part): a wave goes through a unit of parts, the range of a
// checkpoint, or a piece where K is smaller, so every element is passed once
// whatever K is.
ST_DEV double* state_slot( const PlanArgs& a, int64_t slot )
{ return a.states + slot * ST_ADJ_STATE * 64 * ( int64_t )a.tiles; }

// first part of unit u
ST_DEV int64_t unit_begin( const PlanArgs& a, int64_t u )
{
    return a.K > ST_ADJ_PIECE ? ( u * a.K + ST_ADJ_SUB - 1 ) / ST_ADJ_SUB
                              : u * ( ST_ADJ_PIECE / ST_ADJ_SUB );
}

// the first states of parts p .. end - 1 of turn t, from slot on
ST_DEV void keep_states( const PlanArgs& a, int64_t t, int64_t p, int64_t end, int64_t i, int64_t tid,
                         int64_t slot )
{
    int64_t const N = 64 * ( int64_t )a.tiles;
    Lane L;
    for( int64_t e = 0, c = -1; p < end; ++p, ++slot )
    {
        int64_t const b = p * ST_ADJ_SUB;
        if( b / a.K != c )
        {
            c = b / a.K;
            e = c * a.K;
            get_lane( a.ckpt + ( ( t * a.n_seg + c ) * 9 ) * a.n, a.n, i, L );
        }
        run_elements< false >( a, e, b, L, nullptr );
        e = b;
        double* const s = state_slot( a, slot ) + tid;
        s[ 0 ] = L.x;        s[ N ] = L.px;         s[ 2 * N ] = L.y;   s[ 3 * N ] = L.py;
        s[ 4 * N ] = L.zeta; s[ 5 * N ] = L.delta;  s[ 6 * N ] = L.rpp; s[ 7 * N ] = L.rvv;
    }
}

ST_DEV Lane kept_state( const PlanArgs& a, int64_t tid, int64_t slot )
{
    int64_t const N = 64 * ( int64_t )a.tiles;
    const double* const s = state_slot( a, slot ) + tid;
    Lane L;
    L.x = s[ 0 ];        L.px = s[ N ];        L.y = s[ 2 * N ];   L.py = s[ 3 * N ];
    L.zeta = s[ 4 * N ]; L.delta = s[ 5 * N ]; L.rpp = s[ 6 * N ]; L.rvv = s[ 7 * N ];
    L.psigma = L.s = 0.0;                           // no map below reads them
    L.state = 1;
    return L;
}

// The adjoint maps of elements [b, e), last first, on COLS cotangents; lds
// as run_elements< true > left it, L the state after the last element.
// COEF: part receives the wave's sums for the coefficient gradients of every
// multipole (rows of 2 no: d loss / d bal[2k], d loss / d bal[2k + 1]).
template< int COLS, bool COEF >
ST_DEV void reverse_elements( const PlanArgs& a, int64_t b, int64_t e, const Lane& L, const double* lds,
                              Cot* c, double* part, bool add )
{
    double delta = L.delta, rpp = L.rpp, drpp = -rpp * rpp;
    double drvv = drvv_ddelta( delta, a.C.beta0 );
    double const chi = a.C.chi;
    for( int64_t k = e - 1; k >= b; --k )
    {
        cptr_t const r = a.lat + a.rec_off[ k ];
        uint64_t const h = r[ 0 ];
        cptr_t const prm = r + ST_REC_PAYLOAD;
        double const s0 = lds[ 128 * ( k - b ) ], s1 = lds[ 128 * ( k - b ) + 64 ];
        switch( ST_REC_OP( h ) )
        {
        case ST_OP_DRIFT:                         // drift_adj, s = (px, py)
        {
            double const len = rd( prm, 0 );
            double const xp = s0 * rpp, yp = s1 * rpp;
            double const px = s0 * drpp, py = s1 * drpp;
            double const dz = fma( -xp, px, fma( -yp, py, drvv ) ), lr = len * rpp;
#pragma unroll
            for( int q = 0; q < COLS; ++q )
            {
                double const d = fma( c[ q ].x, px, fma( c[ q ].y, py, c[ q ].zeta * dz ) );
                c[ q ].delta = fma( len, d, c[ q ].delta );
                c[ q ].px = fma( lr, fma( -c[ q ].zeta, xp, c[ q ].x ), c[ q ].px );
                c[ q ].py = fma( lr, fma( -c[ q ].zeta, yp, c[ q ].y ), c[ q ].py );
            }
            break;
        }
        case ST_OP_MULTIPOLE:                     // multipole_adj, s = (x, y)
        {
            int const order = ( int )( ST_REC_AUX( h ) & 0x7fffu );
            if( COEF )
            {
                int64_t const m = a.mp_index[ k ];
                double* const g = part + m * ( 2 * a.no );
                double const cx = chi * c[ 0 ].px, cy = chi * c[ 0 ].py;
                double wr = 1.0, wi = 0.0;
                for( int n = 0;; ++n )
                {
                    double const gr = wave_sum( fma( cy, wi, -cx * wr ) );
                    double const gi = wave_sum( fma( cx, wi, cy * wr ) );
                    if( __lane_id() == 63 )
                    {
                        g[ 2 * n ] = add ? g[ 2 * n ] + gr : gr;
                        g[ 2 * n + 1 ] = add ? g[ 2 * n + 1 ] + gi : gi;
                    }
                    if( n == order ) break;
                    double const nr = fma( wr, s0, -wi * s1 );
                    wi = fma( wr, s1, wi * s0 );
                    wr = nr;
                }
            }
            double dre = 0.0, dim = 0.0;          // chi P'(z)
            for( int n = order; n >= 1; --n )
            {
                double const nre = fma( dre, s0, fma( -dim, s1, n * rd( prm, 2 * n ) ) );
                dim = fma( dre, s1, fma( dim, s0, n * rd( prm, 2 * n + 1 ) ) );
                dre = nre;
            }
            dre *= chi;
            dim *= chi;
#pragma unroll
            for( int q = 0; q < COLS; ++q )
            {
                c[ q ].x += fma( -c[ q ].px, dre, c[ q ].py * dim );   // one rounding at the
                c[ q ].y += fma( c[ q ].px, dim, c[ q ].py * dre );    // size of x, of y
            }
            break;
        }
        case ST_OP_CAVITY:                        // s = (zeta, delta)
        {
            double const b2 = a.C.beta0 * a.C.beta0;
            Lane P;
            P.zeta = s0;
            P.delta = delta = s1;
            P.rvv = ( 1.0 + delta ) / sqrt( b2 * ( delta * delta + 2.0 * delta ) + 1.0 );
            rpp = 1.0 / ( 1.0 + delta );
            drpp = -rpp * rpp;
            drvv = drvv_ddelta( delta, a.C.beta0 );
            double zz, zd, dz, dd;
            cavity_jacobian( P, a.C, prm, zz, zd, dz, dd );
#pragma unroll
            for( int q = 0; q < COLS; ++q )
            {
                double const zb = c[ q ].zeta, db = c[ q ].delta;
                c[ q ].zeta = fma( zb, zz, db * dz );
                c[ q ].delta = fma( zb, zd, db * dd );
            }
            break;
        }
        case ST_OP_SROTATION:
#pragma unroll
            for( int q = 0; q < COLS; ++q ) srotation_adj( prm, c[ q ] );
            break;
        default: break;                           // XYShift and apertures: identity
        }
    }
}

// Parts begin .. end - 1, the last first; slot holds the first state of part
// begin, those after it the others'.  A part's state is loaded while the part
// behind it is gone through.
template< int COLS, bool COEF >
ST_DEV void reverse_parts( const PlanArgs& a, int64_t begin, int64_t end, int64_t tid, int64_t slot,
                           double* lds, Cot* c, double* part, bool add )
{
    if( begin >= end ) return;
    Lane first = kept_state( a, tid, slot + ( end - 1 - begin ) );
    for( int64_t p = end - 1; p >= begin; --p )
    {
        int64_t const b = p * ST_ADJ_SUB, e = b + ST_ADJ_SUB < a.n_elem ? b + ST_ADJ_SUB : a.n_elem;
        Lane L = first;
        first = kept_state( a, tid, slot + ( p > begin ? p - 1 - begin : 0 ) );
        run_elements< true >( a, b, e, L, lds );
        reverse_elements< COLS, COEF >( a, b, e, L, lds, c, part, add );
    }
}

// Piece j of a turn whose parts' states are from slot on.
template< int COLS, bool COEF >
ST_DEV void reverse_piece( const PlanArgs& a, int64_t j, int64_t tid, int64_t slot, double* lds, Cot* c,
                           double* part, bool add )
{
    constexpr int PARTS = ST_ADJ_PIECE / ST_ADJ_SUB;
    int64_t const first = j * PARTS;
    reverse_parts< COLS, COEF >( a, first, first + PARTS < a.parts ? first + PARTS : a.parts, tid, slot + first,
                                 lds, c, part, add );
}

// component p of the loss terms of turn t, weight w, g = 2 x the loss's cotangent
ST_DEV double loss_term( const PlanArgs& a, double w, int64_t t, int p, int64_t i, double g )
{
    const double* const b = a.ckpt + ( ( t + 1 ) * a.n_seg * 9 ) * a.n;   // the next turn's first
    return g * w * ( b[ p * a.n + i ] - a.target[ t * 6 + p ] );
}

ST_DEV void add_loss_terms( const PlanArgs& a, int64_t t, int64_t i, Cot& c )
{
    double const g = 2.0 * *a.grad_out;
    c.x += loss_term( a, a.w[ 0 ], t, 0, i, g );
    c.px += loss_term( a, a.w[ 1 ], t, 1, i, g );
    c.y += loss_term( a, a.w[ 2 ], t, 2, i, g );
    c.py += loss_term( a, a.w[ 3 ], t, 3, i, g );
    c.zeta += loss_term( a, a.w[ 4 ], t, 4, i, g );
    c.delta += loss_term( a, a.w[ 5 ], t, 5, i, g );
}

ST_DEV void store_cot( double* g, int64_t i, const Cot& c )
{
    g[ 6 * i ] = c.x; g[ 6 * i + 1 ] = c.px; g[ 6 * i + 2 ] = c.y;
    g[ 6 * i + 3 ] = c.py; g[ 6 * i + 4 ] = c.zeta; g[ 6 * i + 5 ] = c.delta;
}
}  // namespace

// bal of every multipole into the packed lattice and the hot stream
__global__ void __launch_bounds__( 256 ) KN( st_k_adj_coefficients )( st_adj_plan_t p,
    const double* knl, const double* ksl, int scaled )
{
    int64_t const j = ( int64_t )blockIdx.x * blockDim.x + threadIdx.x;
    int const no = ( int )p.max_order + 1;
    if( j >= p.n_mp * no ) return;
    int64_t const m = j / no;
    int const k = ( int )( j % no );
    if( k > p.mp_order[ m ] ) return;
    double f = 1.0;
    for( int q = 2; q <= k; ++q ) f *= q;
    double const inv = scaled ? 1.0 : 1.0 / f;
    double const re = scaled ? knl[ j ] : knl[ j ] * inv, im = scaled ? ksl[ j ] : ksl[ j ] * inv;
    double* const lat = reinterpret_cast< double* >( p.lat ) + p.mp_lat[ m ] + 2 * k;
    double* const hot = reinterpret_cast< double* >( p.hot ) + p.mp_hot[ m ] - 2 * k;
    lat[ 0 ] = re; lat[ 1 ] = im;
    hot[ 0 ] = re; hot[ 1 ] = im;
}

// Forward pass through the hot stream: per segment the checkpoint, then its
// records.  A lane that an aperture would remove sets the status and stops.
__global__ void __launch_bounds__( 64, 4 ) KN( st_k_adj_loss )( PlanArgs a, const double* coords,
    double* loss_out, int32_t* status )
{
    int64_t const n = a.n, tid = ( int64_t )blockIdx.x * 64 + threadIdx.x;
    bool const in_range = tid < n;
    int64_t const i = in_range ? tid : n - 1;
    Lane L;
    L.x = coords[ 6 * i ]; L.px = coords[ 6 * i + 1 ];
    L.y = coords[ 6 * i + 2 ]; L.py = coords[ 6 * i + 3 ];
    L.zeta = coords[ 6 * i + 4 ];
    update_delta( L, a.C, coords[ 6 * i + 5 ] );
    L.s = 0.0;
    double loss = 0.0;
    uint64_t act = ballot( in_range );
    bool ok = true;
    for( int64_t t = 0; t < a.n_turns && act != 0u; ++t )
    {
        for( int64_t j = 0; j < a.n_seg && act != 0u; ++j )
        {
            if( in_range ) put_lane( a.ckpt + ( ( t * a.n_seg + j ) * 9 ) * n, n, i, L );
            cptr_t const sg = a.segments + 3 * j;
            uint64_t const s0 = sg[ 0 ], s1 = sg[ 1 ], s2 = sg[ 2 ];
            uint32_t off = ( uint32_t )s0, next = ( uint32_t )( s0 >> 32 );
            uint32_t const stop = ( uint32_t )s1, head = ( uint32_t )( s1 >> 32 ), tail = ( uint32_t )s2;
            if( head != 0u )
            {
                cptr_t const r = rec_at( a.lat, head - 1u );
                multipole( L, a.C.chi, r + ST_REC_PAYLOAD, ST_REC_AUX( r[ 0 ] ), L.delta );
            }
            while( off != stop && act != 0u )
            {
                uint64_t lost;
                uint32_t info;
                hot_run< true >( a.hot, off, next, stop, L, a.C.chi, act, lost, info );
                if( info == ~0u )                 // not run: the packed records of the segment
                {
                    int64_t const b = j * a.K + ( head != 0u ? 1 : 0 );
                    int64_t e = ( j + 1 ) * a.K < a.n_elem ? ( j + 1 ) * a.K : a.n_elem;
                    if( tail != 0u ) --e;
                    for( int64_t k = b; k < e; ++k ) ok = apply( a.lat + a.rec_off[ k ], L, a.C ) && ok;
                    break;
                }
                if( lost != 0u )
                {
                    if( lane_in( lost ) ) ok = false;
                    act &= ~lost;
                    if( info & 1u )
                    {
                        cptr_t const r = rec_at( a.lat, info & ~1u );
                        cptr_t const m = r + ST_REC_LEN( r[ 0 ] );
                        multipole( L, a.C.chi, m + ST_REC_PAYLOAD, ST_REC_AUX( m[ 0 ] ), L.delta );
                    }
                    continue;
                }
                if( off == stop ) break;
                off += 16u;
                ok = apply( rec_at( a.lat, info ), L, a.C ) && ok;
            }
            if( tail != 0u )
            {
                cptr_t const r = rec_at( a.lat, tail - 1u );
                drift_xz( L, rd( r, 2 ) );
                ok = limit_global_ok( L ) && ok;
            }
        }
        double const X[ 6 ] = { L.x, L.px, L.y, L.py, L.zeta, L.delta };
        for( int c = 0; c < 6; ++c )
        {
            double const d = X[ c ] - a.target[ t * 6 + c ];
            loss += a.w[ c ] * d * d;
        }
    }
    if( !in_range ) return;
    put_lane( a.ckpt + ( a.n_turns * a.n_seg * 9 ) * n, n, i, L );
    loss_out[ i ] = loss;
    if( !ok ) report_failure( status );
}

// block (turn, unit, tile), tile fastest: the first states of the unit's
// parts, slot (turn, part)
__global__ void __launch_bounds__( 64, 4 ) KN( st_k_adj_states )( PlanArgs a )
{
    int64_t const tile = blockIdx.x % a.tiles, tu = blockIdx.x / a.tiles;
    int64_t const u = tu % a.units, k = tu / a.units;
    int64_t const tid = tile * 64 + threadIdx.x;
    int64_t const begin = unit_begin( a, u ), next = unit_begin( a, u + 1 );
    keep_states( a, a.t0 + k, begin, next < a.parts ? next : a.parts, tid < a.n ? tid : a.n - 1, tid,
                 k * a.parts + begin );
}

// block (turn, piece, tile), tile fastest: d (cotangent at the piece's
// start) / d (at its end), column q for the unit cotangent q
__global__ void __launch_bounds__( 64, 2 ) KN( st_k_adj_jacobian )( PlanArgs a )
{
    __shared__ double lds[ ST_ADJ_SUB * 128 ];
    int64_t const tile = blockIdx.x % a.tiles, tp = blockIdx.x / a.tiles;
    int64_t const j = tp % a.pieces, k = tp / a.pieces;
    int64_t const tid = tile * 64 + threadIdx.x;
    Cot c[ 6 ];
#pragma unroll
    for( int q = 0; q < 6; ++q )
        c[ q ] = Cot{ q == 0 ? 1.0 : 0.0, q == 1 ? 1.0 : 0.0, q == 2 ? 1.0 : 0.0,
                      q == 3 ? 1.0 : 0.0, q == 4 ? 1.0 : 0.0, q == 5 ? 1.0 : 0.0 };
    if( a.K <= ST_ADJ_PIECE )                          // its unit is this piece
    {
        int64_t const begin = unit_begin( a, j ), next = unit_begin( a, j + 1 );
        keep_states( a, a.t0 + k, begin, next < a.parts ? next : a.parts, tid < a.n ? tid : a.n - 1, tid,
                     k * a.parts + begin );
    }
    reverse_piece< 6, false >( a, j, tid, k * a.parts, lds + threadIdx.x, c, nullptr, false );
    int64_t const N = 64 * ( int64_t )a.tiles;
    double* const J = a.jac + tp * 36 * N + tid;
#pragma unroll
    for( int q = 0; q < 6; ++q )
    {
        J[ ( 6 * q + 0 ) * N ] = c[ q ].x; J[ ( 6 * q + 1 ) * N ] = c[ q ].px;
        J[ ( 6 * q + 2 ) * N ] = c[ q ].y; J[ ( 6 * q + 3 ) * N ] = c[ q ].py;
        J[ ( 6 * q + 4 ) * N ] = c[ q ].zeta; J[ ( 6 * q + 5 ) * N ] = c[ q ].delta;
    }
}

// The cotangent through the pieces of the group's turns, last first; every
// piece's end cotangent is kept.  REFINE: once more, each piece's start
// cotangent from the one that st_k_adj_through found for the kept end
// cotangent, and the Jacobian applied to the little by which the end
// cotangent has changed.
//
// The pieces are a chain, so what bounds it is how fast the CUs that hold it
// take in the Jacobians, and one CU takes in some 35 GB/s, whatever its waves
// have in flight (64 particles a block: 0.5 us a piece, with one wave or with
// six).  So a block has 16 particles, whose rows are a cache line each, and
// two waves of 48 lanes, three components each: 0.34 us a piece, 0.38 with
// REFINE.
template< bool REFINE >
ST_DEV void adj_chain( const PlanArgs& a )
{
    __shared__ double v[ 2 ][ 6 ][ 16 ];               // by turns: what the Jacobian is applied to
    __shared__ double weight[ 6 ];
    if( threadIdx.x < 6 ) weight[ threadIdx.x ] = a.w[ threadIdx.x ];
    __syncthreads();
    int const l = ( int )threadIdx.x & 63, k = l & 15;
    bool const idle = l >= 48;                         // kept for the barriers
    int const p = 3 * ( int )( threadIdx.x >> 6 ) + ( idle ? 0 : l >> 4 );
    int64_t const tid = ( int64_t )blockIdx.x * 16 + k;
    int64_t const i = tid < a.n ? tid : a.n - 1;
    int64_t const N = 64 * ( int64_t )a.tiles;
    double const g = 2.0 * *a.grad_out;
    int64_t const last = ( int64_t )a.turns * a.pieces - 1;
    auto load = [ & ]( int64_t tp, double* into )
    {
        if( tp < 0 || idle ) return;
        const double* const J = a.jac + ( tp * 36 + p ) * N + tid;
#pragma unroll
        for( int q = 0; q < 6; ++q ) into[ q ] = J[ 6 * q * N ];
        if( REFINE )
        {
            into[ 6 ] = a.cend[ ( tp * 6 + p ) * N + tid ];
            into[ 7 ] = a.cstart[ ( tp * 6 + p ) * N + tid ];
        }
    };
    double c = a.add ? a.grad_coords[ 6 * i + p ] : 0.0;
    int t = a.t0 + a.turns, left = 0;                  // turn, pieces of it before this one
    auto step = [ & ]( int64_t tp, const double* M )
    {
        double( *const w )[ 16 ] = v[ tp & 1 ];
        bool const turn_end = left == 0;
        if( turn_end ) { --t; left = a.pieces; }
        --left;
        if( !idle )
        {
            if( turn_end ) c += loss_term( a, weight[ p ], t, p, i, g );
            a.cend[ ( tp * 6 + p ) * N + tid ] = c;
            w[ p ][ k ] = REFINE ? c - M[ 6 ] : c;
        }
        __syncthreads();
        double const r = fma( M[ 0 ], w[ 0 ][ k ], fma( M[ 1 ], w[ 1 ][ k ], fma( M[ 2 ], w[ 2 ][ k ],
                         fma( M[ 3 ], w[ 3 ][ k ], fma( M[ 4 ], w[ 4 ][ k ], M[ 5 ] * w[ 5 ][ k ] ) ) ) ) );
        c = REFINE ? M[ 7 ] + r : r;
    };
    constexpr int AHEAD = 8;
    double M[ AHEAD ][ 8 ] = {};
#pragma unroll
    for( int j = 0; j < AHEAD - 1; ++j ) load( last - j, M[ j ] );
    for( int64_t tp = last; tp >= 0; tp -= AHEAD )
    {
#pragma unroll
        for( int j = 0; j < AHEAD; ++j )
        {
            if( tp - j < 0 ) break;
            load( tp - j - ( AHEAD - 1 ), M[ ( j + AHEAD - 1 ) % AHEAD ] );
            step( tp - j, M[ j ] );
        }
    }
    if( REFINE && !idle && tid < a.n ) a.grad_coords[ 6 * i + p ] = c;
}

__global__ void __launch_bounds__( 128 ) KN( st_k_adj_chain )( PlanArgs a )
{
    adj_chain< false >( a );
}

__global__ void __launch_bounds__( 128 ) KN( st_k_adj_chain_refine )( PlanArgs a )
{
    adj_chain< true >( a );
}

// block (turn, piece, tile): a piece's start cotangent, element by element
// from its end cotangent
__global__ void __launch_bounds__( 64, 2 ) KN( st_k_adj_through )( PlanArgs a )
{
    __shared__ double lds[ ST_ADJ_SUB * 128 ];
    int64_t const tile = blockIdx.x % a.tiles, tp = blockIdx.x / a.tiles;
    int64_t const j = tp % a.pieces, k = tp / a.pieces, N = 64 * ( int64_t )a.tiles;
    int64_t const tid = tile * 64 + threadIdx.x;
    const double* const ce = a.cend + tp * 6 * N + tid;
    Cot c{ ce[ 0 ], ce[ N ], ce[ 2 * N ], ce[ 3 * N ], ce[ 4 * N ], ce[ 5 * N ] };
    reverse_piece< 1, false >( a, j, tid, k * a.parts, lds + threadIdx.x, &c, nullptr, false );
    double* const cs = a.cstart + tp * 6 * N + tid;
    cs[ 0 ] = c.x; cs[ N ] = c.px; cs[ 2 * N ] = c.y;
    cs[ 3 * N ] = c.py; cs[ 4 * N ] = c.zeta; cs[ 5 * N ] = c.delta;
}

// CHAIN: one wave goes through all pieces of all turns, last first, with its
// cotangent; its partial sums gather over the turns.  Otherwise block
// (turn, piece, tile) from the piece's end cotangent.
template< bool CHAIN >
ST_DEV void adj_reverse( const PlanArgs& a, double* lds )
{
    int64_t const tile = blockIdx.x % a.tiles, tp = blockIdx.x / a.tiles;
    int64_t const tid = tile * 64 + threadIdx.x;
    bool const in_range = tid < a.n;
    int64_t const i = in_range ? tid : a.n - 1;
    int64_t const row = a.n_mp * 2 * a.no;
    Cot c{ 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    if( !CHAIN )
    {
        int64_t const j = tp % a.pieces, k = tp / a.pieces, N = 64 * ( int64_t )a.tiles;
        const double* const ce = a.cend + tp * 6 * N + tid;
        if( in_range ) c = Cot{ ce[ 0 ], ce[ N ], ce[ 2 * N ], ce[ 3 * N ], ce[ 4 * N ], ce[ 5 * N ] };
        reverse_piece< 1, true >( a, j, tid, k * a.parts, lds, &c,
                                  a.partial + ( k * a.tiles + tile ) * row, a.add != 0 );
        return;
    }
    for( int64_t t = a.n_turns - 1; t >= 0; --t )
    {
        if( in_range ) add_loss_terms( a, t, i, c );
        // unit by unit, the last first; its states from slot 0 on
        int64_t end = a.parts;
        for( int64_t u = a.units - 1; u >= 0; --u )
        {
            int64_t const begin = unit_begin( a, u );
            keep_states( a, t, begin, end, i, tid, 0 );
            reverse_parts< 1, true >( a, begin, end, tid, 0, lds, &c, a.partial + tile * row, t < a.n_turns - 1 );
            end = begin < end ? begin : end;
        }
    }
    if( in_range ) store_cot( a.grad_coords, i, c );
}

__global__ void __launch_bounds__( 64, 2 ) KN( st_k_adj_reverse )( PlanArgs a )
{
    __shared__ double lds[ ST_ADJ_SUB * 128 ];
    adj_reverse< false >( a, lds + threadIdx.x );
}

__global__ void __launch_bounds__( 64, 2 ) KN( st_k_adj_reverse_chain )( PlanArgs a )
{
    __shared__ double lds[ ST_ADJ_SUB * 128 ];
    adj_reverse< true >( a, lds + threadIdx.x );
}

// one block per multipole: the partial sums added up, times 1 / n!
__global__ void __launch_bounds__( 256 ) KN( st_k_adj_sum )( const double* partial, int64_t partials,
    int64_t n_mp, int no, const int32_t* mp_order, double* grad_knl, double* grad_ksl )
{
    __shared__ double red[ 4 ];
    int64_t const m = blockIdx.x;
    int const order = mp_order[ m ];
    double f = 1.0;
    for( int k = 0; k < no; ++k )
    {
        if( k > 1 ) f *= k;
        for( int c = 0; c < 2; ++c )
        {
            double v = 0.0;
            if( k <= order )
                for( int64_t p = threadIdx.x; p < partials; p += 256 )
                    v += partial[ ( p * n_mp + m ) * ( 2 * no ) + 2 * k + c ];
            v = wave_sum( v );
            if( __lane_id() == 63 ) red[ threadIdx.x >> 6 ] = v;
            __syncthreads();
            if( threadIdx.x == 0 )
                ( c == 0 ? grad_knl : grad_ksl )[ m * no + k ] =
                    ( ( red[ 0 ] + red[ 1 ] ) + ( red[ 2 ] + red[ 3 ] ) ) * ( 1.0 / f );
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------ launchers

namespace
{
AdjArgs make_args( const st_adj_problem_t* p )
{
    AdjArgs a{};
    a.lat = ( cptr_t )p->lat;
    a.rec_off = ( cu32_t* )p->rec_off;
    a.n_elem = p->n_elem; a.K = p->K; a.n_seg = ( p->n_elem + p->K - 1 ) / p->K;
    a.n_turns = p->n_turns; a.n = p->n;
    a.C.q0 = p->q0; a.C.mass0 = p->mass0; a.C.beta0 = p->beta0; a.C.p0c = p->p0c;
    a.C.chi = p->chi; a.C.charge_ratio = p->charge_ratio;
    for( int c = 0; c < 6; ++c ) a.w[ c ] = p->weights[ c ];
    a.target = p->target;
    a.ckpt = p->ckpt;
    a.mp_index = ( ci32_t* )p->mp_index;
    return a;
}
}  // namespace

extern "C" hipError_t KN( st_launch_adj_forward )( const st_adj_problem_t* p, const double* coords,
    double* loss, int32_t* status, hipStream_t stream )
{
    if( p->n <= 0 ) return hipSuccess;
    AdjArgs a = make_args( p );
    a.coords = coords; a.loss = loss; a.status = status;
    hipLaunchKernelGGL( KN( st_k_adj_forward ), dim3( ( unsigned )( ( p->n + 255 ) / 256 ) ), dim3( 256 ),
                        0, stream, a );
    return hipGetLastError();
}

extern "C" hipError_t KN( st_launch_adj_backward_turn )( const st_adj_problem_t* p, int64_t turn,
    const double* grad_out, double* segbuf, double* coef, double* cot, hipStream_t stream )
{
    if( p->n <= 0 ) return hipSuccess;
    AdjArgs a = make_args( p );
    a.turn = turn; a.grad_out = grad_out; a.segbuf = segbuf; a.coef = coef; a.cot = cot;
    hipLaunchKernelGGL( KN( st_k_adj_backward_turn ), dim3( ( unsigned )( ( p->n + 255 ) / 256 ) ),
                        dim3( 256 ), 0, stream, a );
    return hipGetLastError();
}

extern "C" hipError_t KN( st_launch_adj_reduce )( const st_adj_problem_t* p, const int32_t* mp_order,
    int64_t n_mp, const double* coef, double* grad_bal, int64_t stride, hipStream_t stream )
{
    if( n_mp <= 0 || p->n <= 0 ) return hipSuccess;
    hipLaunchKernelGGL( KN( st_k_adj_reduce ), dim3( ( unsigned )n_mp ), dim3( 256 ), 0, stream,
                        p->n, mp_order, coef, grad_bal, stride );
    return hipGetLastError();
}

namespace
{
PlanArgs plan_args( const st_adj_plan_t* p )
{
    PlanArgs a{};
    a.lat = ( cptr_t )p->base.lat; a.hot = ( cptr_t )p->hot;
    a.rec_off = ( cu32_t* )p->base.rec_off; a.mp_index = ( ci32_t* )p->base.mp_index;
    a.segments = ( cptr_t )p->segments;
    a.n_elem = p->base.n_elem; a.K = p->base.K;
    a.n_seg = ( p->base.n_elem + p->base.K - 1 ) / p->base.K;
    a.n_turns = p->base.n_turns; a.n = p->base.n; a.n_mp = p->n_mp;
    a.no = ( int32_t )p->max_order + 1;
    a.tiles = ( int32_t )st_adj_tiles( p ); a.pieces = ( int32_t )st_adj_pieces( p );
    a.parts = st_adj_parts( p ); a.units = st_adj_units( p );
    a.C.q0 = p->base.q0; a.C.mass0 = p->base.mass0; a.C.beta0 = p->base.beta0; a.C.p0c = p->base.p0c;
    a.C.chi = p->base.chi; a.C.charge_ratio = p->base.charge_ratio;
    for( int c = 0; c < 6; ++c ) a.w[ c ] = p->base.weights[ c ];
    a.target = p->base.target;
    a.ckpt = p->base.ckpt;
    return a;
}
}  // namespace

extern "C" hipError_t KN( st_launch_adj_coefficients )( const st_adj_plan_t* p, const double* knl,
    const double* ksl, int scaled, hipStream_t stream )
{
    int64_t const n = p->n_mp * ( p->max_order + 1 );
    if( n <= 0 ) return hipSuccess;
    hipLaunchKernelGGL( KN( st_k_adj_coefficients ), dim3( ( unsigned )( ( n + 255 ) / 256 ) ), dim3( 256 ),
                        0, stream, *p, knl, ksl, scaled );
    return hipGetLastError();
}

extern "C" hipError_t KN( st_launch_adj_loss )( const st_adj_plan_t* p, const double* coords,
    double* loss, int32_t* status, hipStream_t stream )
{
    if( p->base.n <= 0 ) return hipSuccess;
    hipLaunchKernelGGL( KN( st_k_adj_loss ), dim3( ( unsigned )st_adj_tiles( p ) ), dim3( 64 ), 0, stream,
                        plan_args( p ), coords, loss, status );
    return hipGetLastError();
}

extern "C" hipError_t KN( st_launch_adj_gradients )( const st_adj_plan_t* p, const double* grad_out,
    double* work, int64_t group, double* grad_coords, double* grad_knl, double* grad_ksl, hipStream_t stream )
{
    PlanArgs a = plan_args( p );
    a.grad_out = grad_out;
    a.grad_coords = grad_coords;
    int64_t const tiles = st_adj_tiles( p ), pieces = st_adj_pieces( p );
    int64_t const partials = p->base.n > 0 ? ( group > 0 ? group : 1 ) * tiles : 0;
    a.jac = work;
    a.cend = a.jac + group * pieces * 36 * 64 * tiles;
    a.cstart = a.cend + group * pieces * 6 * 64 * tiles;
    a.states = a.cstart + group * pieces * 6 * 64 * tiles;
    a.partial = work + st_adj_work_doubles( p, group ) - partials * st_adj_row_doubles( p );
    if( p->base.n > 0 && group > 0 )
    {
        for( int64_t end = p->base.n_turns; end > 0; end -= group )
        {
            // the last turns first, groups of the same size (a turn's rows of
            // the partial sums are added to by the groups after the first)
            a.t0 = ( int32_t )( end > group ? end - group : 0 );
            a.turns = ( int32_t )( end - a.t0 );
            a.add = end < p->base.n_turns ? 1 : 0;
            unsigned const grid = ( unsigned )( a.turns * pieces * tiles );
            if( a.K > ST_ADJ_PIECE )
                hipLaunchKernelGGL( KN( st_k_adj_states ), dim3( ( unsigned )( a.turns * a.units * tiles ) ),
                                    dim3( 64 ), 0, stream, a );
            hipLaunchKernelGGL( KN( st_k_adj_jacobian ), dim3( grid ), dim3( 64 ), 0, stream, a );
            hipLaunchKernelGGL( KN( st_k_adj_chain ), dim3( ( unsigned )( 4 * tiles ) ), dim3( 128 ), 0, stream, a );
            hipLaunchKernelGGL( KN( st_k_adj_through ), dim3( grid ), dim3( 64 ), 0, stream, a );
            hipLaunchKernelGGL( KN( st_k_adj_chain_refine ), dim3( ( unsigned )( 4 * tiles ) ), dim3( 128 ), 0, stream, a );
            hipLaunchKernelGGL( KN( st_k_adj_reverse ), dim3( grid ), dim3( 64 ), 0, stream, a );
            hipError_t const e = hipGetLastError();
            if( e != hipSuccess ) return e;
        }
    }
    else if( p->base.n > 0 )
    {
        hipLaunchKernelGGL( KN( st_k_adj_reverse_chain ), dim3( ( unsigned )tiles ), dim3( 64 ), 0, stream, a );
        hipError_t const e = hipGetLastError();
        if( e != hipSuccess ) return e;
    }
    if( p->n_mp > 0 )
        hipLaunchKernelGGL( KN( st_k_adj_sum ), dim3( ( unsigned )p->n_mp ), dim3( 256 ), 0, stream,
                            a.partial, partials, p->n_mp, ( int )a.no,
                            p->mp_order, grad_knl, grad_ksl );
    return hipGetLastError();
}
