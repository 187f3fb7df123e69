// Host-side prototypes of the kernel launchers (two build variants of
// track_kernels.hip: _exact without FP contraction, _fma with it).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lattice.h"

// A segment of a lattice for track_line through the hot stream
// (lattice_hot.h); byte offsets.
typedef struct st_hot_segment_s
{
    const void* seed;        // descriptor of the set and its lattice (st_batch_seed_t, batch.h)
    int64_t begin;           // first element
    uint32_t off, next;      // first whole record and its handler
    uint32_t stop;           // record after the last whole one
    uint32_t head;           // packed record of a Multipole to run first, 0: none
    uint32_t tail;           // packed record of a Drift to run last + 8, 0: none
    uint32_t unused;
    uint64_t s_begin, s_end; // path length at the segment's ends on a turn from s = 0 (bits)
}
st_hot_segment_t;

#define ST_DECLARE_LAUNCHERS( SUF )                                              \
    extern "C" hipError_t st_launch_track_until##SUF( const st_dev_particles_t* P, \
        const uint64_t* lat, int64_t n_elem, int64_t until_turn, int full,       \
        int32_t* status, int block, hipStream_t stream );                         \
    extern "C" hipError_t st_launch_track_ebe##SUF( const st_dev_particles_t* P,  \
        const uint64_t* lat, int64_t n_elem, int64_t until_turn,                  \
        const st_ebe_config_t* cfg, int64_t cap, const st_dev_particles_t* O,       \
        int32_t* status, int64_t from_turn,                                        \
        int block, hipStream_t stream );                                          \
    extern "C" hipError_t st_launch_track_line##SUF( const st_dev_particles_t* P, \
        const uint64_t* lat, int64_t n_line, int finish_turn, int32_t* status,    \
        int block, hipStream_t stream );                                          \
    extern "C" hipError_t st_launch_track_line_hot##SUF( int64_t n,               \
        const st_hot_segment_t* seg, const uint64_t* lat, int64_t n_line,         \
        int finish_turn, int heavy, int32_t* status, hipStream_t stream );

ST_DECLARE_LAUNCHERS( _exact )
ST_DECLARE_LAUNCHERS( _fma )
