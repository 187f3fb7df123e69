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

#include <stddef.h>
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
    size_t words = 0, elements = 0;
    for( ; ST_REC_OP( lat[ words ] ) != ST_OP_END; words += ST_REC_LEN( lat[ words ] ) ) ++elements;
    /* no hot record is longer than the packed records it stands for, and a
     * TOUCH record of one word comes before at least ST_HOT_TOUCH_BYTES */
    std::vector< uint64_t > stream( words + 2u + words / ( ST_HOT_TOUCH_BYTES / 8u ) + 2u +
                                    ST_HOT_PAD_WORDS, 0u );
    uint64_t* const begin = stream.data();
    uint64_t* w = begin;                          /* next word to write          */
    uint64_t* last = nullptr;                     /* word 0 of the record before */
    uint64_t* touched = nullptr;                  /* last TOUCH record           */
    uint32_t handler = 0, parity = 0;             /* of the record being written */
    uint32_t *m_off = nullptr, *m_handler = nullptr;
    uint64_t* m_s = nullptr;
    if( map != nullptr )
    {
        map->off.resize( elements + 1u );
        map->handler.resize( elements + 1u );
        map->s.resize( elements + 1u );
        m_off = map->off.data(); m_handler = map->handler.data(); m_s = map->s.data();
    }
    auto put = [ & ]( unsigned kind, size_t at )
    {
        handler = ( uint32_t )( kind * ST_HOT_SPACING ) + parity;
        parity ^= ST_HOT_SET_B;
        if( last != nullptr ) *last |= handler;   /* the record before names it  */
        last = w;
        *w++ = ( uint64_t )( at * 8u ) << 32;
    };
    auto put_mp = [ & ]( const uint64_t* r )
    {
        for( int k = ( int )ST_REC_AUX( r[ 0 ] ); k >= 0; --k )
        {
            *w++ = r[ ST_REC_PAYLOAD + 2 * k ];
            *w++ = r[ ST_REC_PAYLOAD + 2 * k + 1 ];
        }
    };
    auto element = [ & ]( unsigned second, uint64_t path )
    {
        if( map == nullptr ) return;
        *m_off++ = ( uint32_t )( ( last - begin ) * 8 ) | second;
        *m_handler++ = handler;
        *m_s++ = path;
    };
    uint64_t s = 0;                               /* bits of +0.0                */
    for( size_t pos = 0;; )
    {
        if( touched == nullptr || ( size_t )( w - touched ) * 8u >= ST_HOT_TOUCH_BYTES )
        {
            touched = w;
            put( ST_HOT_TOUCH, pos );
        }
        const uint64_t* const r = lat + pos;
        const uint64_t* const e = r + ST_REC_PAYLOAD;
        unsigned const op = ST_REC_OP( r[ 0 ] ), aux = ST_REC_AUX( r[ 0 ] );
        uint64_t const s_before = s;
        pos += ST_REC_LEN( r[ 0 ] );
        switch( op )
        {
        case ST_OP_DRIFT:
        {
            const uint64_t* const m = lat + pos;
            s = e[ 1 ];
            if( ST_REC_OP( m[ 0 ] ) == ST_OP_MULTIPOLE && ST_REC_AUX( m[ 0 ] ) <= ST_HOT_MAX_ORDER )
            {
                put( ST_HOT_DRIFT_MP + ST_REC_AUX( m[ 0 ] ), r - lat );
                *w++ = e[ 0 ];
                put_mp( m );
                element( 0u, s_before );
                element( 1u, s );
                pos += ST_REC_LEN( m[ 0 ] );
                continue;
            }
            put( ST_HOT_DRIFT, r - lat );
            *w++ = e[ 0 ];
            break;
        }
        case ST_OP_XYSHIFT:
        case ST_OP_SROTATION:
            put( op == ST_OP_XYSHIFT ? ST_HOT_XYSHIFT : ST_HOT_SROTATION, r - lat );
            *w++ = e[ 0 ];
            *w++ = e[ 1 ];
            break;
        case ST_OP_LIMIT_RECT:
        case ST_OP_LIMIT_ELLIPSE:
            put( op == ST_OP_LIMIT_RECT ? ST_HOT_LIMIT_RECT : ST_HOT_LIMIT_ELLIPSE, r - lat );
            for( int k = 0; k < ( op == ST_OP_LIMIT_RECT ? 4 : 3 ); ++k ) *w++ = e[ k ];
            *w++ = s;
            break;
        default:
            if( op == ST_OP_MULTIPOLE && aux <= ST_HOT_MAX_ORDER )
            {
                put( ST_HOT_MULTIPOLE + aux, r - lat );
                put_mp( r );
                break;
            }
            if( op == ST_OP_DRIFT_EXACT ) s = e[ 1 ];
            put( ST_HOT_EXIT, r - lat );
            *w++ = s;
            break;
        }
        element( 0u, s_before );
        if( op == ST_OP_END ) break;
    }
    stream.resize( ( size_t )( w - begin ) + ST_HOT_PAD_WORDS );
    return stream;
}
}  // namespace st
#endif

#endif /* SIXTRACKLIB_AMD_LATTICE_HOT_H__ */
