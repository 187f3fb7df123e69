/* Hot stream: the packed lattice (lattice.h) once more, in the form the
 * scheduled record walk of track_hot.h reads.
 *
 * record:  word 0  bits 0-31 byte offset of the NEXT record's handler
 *                  (its kind * ST_HOT_SPACING, + ST_HOT_SET_B for every
 *                  second record), bits 32-63 byte offset of the element's
 *                  record in the packed lattice
 *          word 1…  parameters; the length follows from the kind
 * A Drift followed by a Multipole is one record.  Multipole coefficients
 * are stored highest order first (re, im of order n, n - 1, … 0).  Records
 * that can lose a particle at an aperture, and EXIT records, end with the
 * path length s after the last drift on a turn that starts at s = 0.
 * Elements without a handler (and the END record) are EXIT records: the
 * walk returns on them and the caller runs the packed lattice's record.
 * The stream starts with a TOUCH record.
 */
#ifndef SIXTRACKLIB_AMD_LATTICE_HOT_H__
#define SIXTRACKLIB_AMD_LATTICE_HOT_H__

#include <stdint.h>

#include "lattice.h"

#define ST_HOT_SPACING      1024   /* bytes between two handlers                */
#define ST_HOT_SET_B        32768  /* handlers of the second register set       */
#define ST_HOT_EXIT         0      /* [s]                                       */
#define ST_HOT_DRIFT        1      /* [L]                                       */
#define ST_HOT_XYSHIFT      2      /* [-dx, -dy]                                */
#define ST_HOT_SROTATION    3      /* [cos, sin]                                */
#define ST_HOT_LIMIT_RECT   4      /* [min_x, max_x, min_y, max_y, s]           */
#define ST_HOT_LIMIT_ELLIPSE 5     /* [a^2, b^2, a^2 b^2, s]                    */
#define ST_HOT_TOUCH        6      /* []                                        */
#define ST_HOT_MULTIPOLE    7      /* + order 0..10: [coefficients]             */
#define ST_HOT_DRIFT_MP     18     /* + order 0..10: [L, coefficients]          */
#define ST_HOT_MAX_ORDER    10
/* TOUCH records: one about every ST_HOT_TOUCH_BYTES of the stream (at most
 * a longest record of 192 bytes more); each reads one word of every 64-byte
 * line from ST_HOT_TOUCH_AHEAD bytes past its end up to where the next one
 * starts to. */
#define ST_HOT_TOUCH_BYTES  1024
#define ST_HOT_TOUCH_AHEAD  128
#define ST_HOT_TOUCH_LINES  20
/* zero words after the stream: the walk loads 128 bytes of the record after
 * the last and touches the lines of a TOUCH interval past the end */
#define ST_HOT_PAD_WORDS    256

#if defined( __cplusplus )
#include <vector>

namespace st
{
/* Where the elements of a lattice are in its hot stream: entry i for element
 * i, one more entry for the end of the lattice. */
struct HotMap
{
    std::vector< uint32_t > off;       /* byte offset of the record that holds it; bit 0
                                          set for the Multipole of a Drift's record  */
    std::vector< uint32_t > handler;   /* handler offset of that record              */
    std::vector< uint64_t > s;         /* path length before it, on a turn from s = 0 */
};

/* hot stream of the packed lattice ``lat`` (END-terminated), padding
 * included */
inline std::vector< uint64_t > hot_stream( const uint64_t* lat, HotMap* map = nullptr )
{
    if( map ) *map = HotMap();
    size_t end = 0;
    while( ST_REC_OP( lat[ end ] ) != ST_OP_END ) end += ST_REC_LEN( lat[ end ] );
    std::vector< uint64_t > w;
    w.reserve( end + end / 16 + ST_HOT_PAD_WORDS + 16 );
    uint64_t s = 0;                               /* bits of +0.0 */
    size_t pos = 0, touched = 0;
    bool first = true;
    size_t last = 0, records = 0;
    uint64_t s_before = 0;
    uint32_t handler = 0;
    auto put = [ & ]( unsigned kind, size_t at )
    {
        // the record before names this one's handler
        handler = ( uint32_t )( kind * ST_HOT_SPACING + ( records % 2 ) * ST_HOT_SET_B );
        if( records > 0 ) w[ last ] |= handler;
        last = w.size();
        ++records;
        w.push_back( ( uint64_t )( at * 8u ) << 32 );
    };
    auto element = [ & ]( unsigned second, uint64_t path )
    {
        if( map == nullptr ) return;
        map->off.push_back( ( uint32_t )( last * 8u ) | second );
        map->handler.push_back( handler );
        map->s.push_back( path );
    };
    auto is_flat_mp = [ & ]( uint64_t h )
    { return ST_REC_OP( h ) == ST_OP_MULTIPOLE && ST_REC_AUX( h ) <= ST_HOT_MAX_ORDER; };
    auto put_mp = [ & ]( size_t at )
    {
        int const order = ( int )ST_REC_AUX( lat[ at ] );
        for( int k = order; k >= 0; --k )
        {
            w.push_back( lat[ at + ST_REC_PAYLOAD + 2 * k ] );
            w.push_back( lat[ at + ST_REC_PAYLOAD + 2 * k + 1 ] );
        }
    };
    for( ;; )
    {
        if( first || ( w.size() - touched ) * 8u >= ST_HOT_TOUCH_BYTES )
        {
            touched = w.size();
            first = false;
            put( ST_HOT_TOUCH, pos );
        }
        s_before = s;
        uint64_t const h = lat[ pos ];
        const uint64_t* const e = lat + pos + ST_REC_PAYLOAD;
        size_t const next = pos + ST_REC_LEN( h );
        switch( ST_REC_OP( h ) )
        {
        case ST_OP_DRIFT:
        {
            s = e[ 1 ];
            if( is_flat_mp( lat[ next ] ) )
            {
                put( ST_HOT_DRIFT_MP + ST_REC_AUX( lat[ next ] ), pos );
                w.push_back( e[ 0 ] );
                put_mp( next );
                element( 0u, s_before );
                element( 1u, s );
                pos = next + ST_REC_LEN( lat[ next ] );
                continue;
            }
            put( ST_HOT_DRIFT, pos );
            w.push_back( e[ 0 ] );
            break;
        }
        case ST_OP_XYSHIFT:
        case ST_OP_SROTATION:
            put( ST_REC_OP( h ) == ST_OP_XYSHIFT ? ST_HOT_XYSHIFT : ST_HOT_SROTATION, pos );
            w.push_back( e[ 0 ] ); w.push_back( e[ 1 ] );
            break;
        case ST_OP_LIMIT_RECT:
            put( ST_HOT_LIMIT_RECT, pos );
            w.insert( w.end(), e, e + 4 );
            w.push_back( s );
            break;
        case ST_OP_LIMIT_ELLIPSE:
            put( ST_HOT_LIMIT_ELLIPSE, pos );
            w.insert( w.end(), e, e + 3 );
            w.push_back( s );
            break;
        default:
            if( is_flat_mp( h ) )
            {
                put( ST_HOT_MULTIPOLE + ST_REC_AUX( h ), pos );
                put_mp( pos );
                break;
            }
            if( ST_REC_OP( h ) == ST_OP_DRIFT_EXACT ) s = e[ 1 ];
            put( ST_HOT_EXIT, pos );
            w.push_back( s );
            break;
        }
        element( 0u, s_before );
        if( ST_REC_OP( h ) == ST_OP_END ) break;
        pos = next;
    }
    w.resize( w.size() + ST_HOT_PAD_WORDS, 0u );
    return w;
}
}  // namespace st
#endif

#endif /* SIXTRACKLIB_AMD_LATTICE_HOT_H__ */
