// The record walk of the until-turn loop as one scheduled instruction
// sequence (device code, gfx950), one particle per lane.
//
// What bounds it: a wave issues at most one instruction of any kind per four
// cycles (measured, a scalar add as much as an FP64 multiply-add), so with
// few waves per SIMD a record costs its instructions one after the other,
// scalar work included, plus what it waits for: 41 to 69 cycles for scalar
// loads that hit the scalar cache, 166 for one that misses to L2, about 35
// for a taken jump.  The compiled loop of track_lean.h spends 166 ns (FMA
// build) to 193 ns (exact) per element of a 20,000-element ring, whether 64
// or 65,536 particles are tracked; the FP64 instructions of an average
// element take 25 to 35 ns.  Here
//   * every record of the hot stream (lattice_hot.h) names the handler of
//     the next one: the dispatch is one computed jump, no compare tree, and
//     it does not wait for the next record's words;
//   * the first eight words of the next record are loaded while the current
//     one runs, into the other of two SGPR sets (every handler exists once
//     per set).  Multipole coefficients are stored highest order first, the
//     order Horner reads them, so a long record's further words are loaded
//     while its first steps run;
//   * a Drift and the Multipole after it are one record;
//   * the stream is larger than the scalar cache: TOUCH records, one about
//     every kilobyte, read one word of each of the following lines, so that
//     the misses of a kilobyte overlap instead of stalling record by record
//     (scalar loads complete out of order, so a load in flight is in every
//     wait);
//   * the lanes lost or done are out of exec, so an aperture test needs no
//     mask operation.
// Measured on that ring (ns per element, compiled loop / this): exact build
// 189 / 77 with 1,000 particles, 192 / 77 with 16,000, 193 / 86 with 65,536;
// FMA build 166 / 54, 168 / 55 and 169 / 62.
// Maps are those of track_device.h with the same IEEE operations (each
// fused where that build fuses), so the results are the same bits.
#pragma once

#include "track_lean.h"
#include "lattice_hot.h"

namespace st
{

// Runs hot records from byte offset ``off`` of ``hot`` (``next``: the offset
// of its handler) until a record of the EXIT kind (off stays on it, lost = 0,
// next is that of the record after it) or until lanes of ``act`` are lost at
// a Drift or an aperture: then lost holds them, off and next are those of
// the next record.  info is the byte offset of the element's record in the
// packed lattice, bit 0 set when lanes were lost at the Drift of a record
// whose Multipole is still to run.  info = ~0: nothing was run, because a
// jump target is formed with a 32-bit add and the handlers lie across a
// 4 GiB boundary.
//
// SGPRs: first words of a record s[36:51] and s[52:67], further words
// s[68:99], jump target s[34:35].

#define ST_HOT_SGPRS \
    "s34", "s35", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44", "s45", \
    "s46", "s47", "s48", "s49", "s50", "s51", "s52", "s53", "s54", "s55", "s56", "s57", \
    "s58", "s59", "s60", "s61", "s62", "s63", "s64", "s65", "s66", "s67", "s68", "s69", \
    "s70", "s71", "s72", "s73", "s74", "s75", "s76", "s77", "s78", "s79", "s80", "s81", \
    "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89", "s90", "s91", "s92", "s93", \
    "s94", "s95", "s96", "s97", "s98", "s99"

#if defined( ST_FMA_BUILD )
#define ST_HOT_ARITH R"(
.macro ST_SLOPES
  v_mul_f64 %[t0], %[px], %[rpp]
  v_mul_f64 %[t1], %[py], %[rpp]
.endm
.macro ST_DRIFT X, lw
  v_fma_f64 %[x], %[t0], s[\X+2*\lw:\X+2*\lw+1], %[x]
  v_fma_f64 %[y], %[t1], s[\X+2*\lw:\X+2*\lw+1], %[y]
  v_mul_f64 %[t1], %[t1], %[t1]
  v_cmp_nlt_f64 vcc, |%[x]|, 1.0
  v_cmp_nlt_f64 %[m], |%[y]|, 1.0
  v_fma_f64 %[t0], %[t0], %[t0], %[t1]
  v_fma_f64 %[t0], %[t0], 0.5, 1.0
  v_add_f64 %[t0], %[rvv], -%[t0]
  s_or_b64 vcc, vcc, %[m]
  v_fma_f64 %[z], %[t0], s[\X+2*\lw:\X+2*\lw+1], %[z]
.endm
.macro ST_FIRST X, wr, wi, vr, vi
  v_mov_b64 %[t1], s[\X+2*\wi:\X+2*\wi+1]
  v_fma_f64 %[t3], %[t1], %[x], s[\X+2*\vi:\X+2*\vi+1]
  v_fma_f64 %[t2], -%[t1], %[y], s[\X+2*\vr:\X+2*\vr+1]
  v_fma_f64 %[t1], s[\X+2*\wr:\X+2*\wr+1], %[y], %[t3]
  v_fma_f64 %[t0], s[\X+2*\wr:\X+2*\wr+1], %[x], %[t2]
.endm
.macro ST_STEP X, vr, vi
  v_fma_f64 %[t3], %[t1], %[x], s[\X+2*\vi:\X+2*\vi+1]
  v_fma_f64 %[t2], -%[t1], %[y], s[\X+2*\vr:\X+2*\vr+1]
  v_fma_f64 %[t1], %[t0], %[y], %[t3]
  v_fma_f64 %[t0], %[t0], %[x], %[t2]
.endm
.macro ST_KICK
  v_fma_f64 %[px], -%[chi], %[t0], %[px]
  v_fma_f64 %[py], %[chi], %[t1], %[py]
.endm
.macro ST_KICK0 X, wr, wi
  v_fma_f64 %[px], -%[chi], s[\X+2*\wr:\X+2*\wr+1], %[px]
  v_fma_f64 %[py], %[chi], s[\X+2*\wi:\X+2*\wi+1], %[py]
.endm
.macro ST_ROT X, a, b
  v_mul_f64 %[t0], s[\X+4:\X+5], \b
  v_mul_f64 %[t1], s[\X+4:\X+5], \a
  v_fma_f64 \a, s[\X+2:\X+3], \a, %[t0]
  v_fma_f64 \b, s[\X+2:\X+3], \b, -%[t1]
.endm
)"
#else
#define ST_HOT_ARITH R"(
.macro ST_SLOPES
  v_mul_f64 %[t0], %[px], %[rpp]
  v_mul_f64 %[t1], %[py], %[rpp]
.endm
.macro ST_DRIFT X, lw
  v_mul_f64 %[t2], %[t0], s[\X+2*\lw:\X+2*\lw+1]
  v_mul_f64 %[t3], %[t1], s[\X+2*\lw:\X+2*\lw+1]
  v_add_f64 %[x], %[x], %[t2]
  v_add_f64 %[y], %[y], %[t3]
  v_mul_f64 %[t0], %[t0], %[t0]
  v_mul_f64 %[t1], %[t1], %[t1]
  v_cmp_nlt_f64 vcc, |%[x]|, 1.0
  v_cmp_nlt_f64 %[m], |%[y]|, 1.0
  v_add_f64 %[t0], %[t0], %[t1]
  v_mul_f64 %[t0], %[t0], 0.5
  v_add_f64 %[t0], %[t0], 1.0
  s_or_b64 vcc, vcc, %[m]
  v_add_f64 %[t0], %[rvv], -%[t0]
  v_mul_f64 %[t0], %[t0], s[\X+2*\lw:\X+2*\lw+1]
  v_add_f64 %[z], %[z], %[t0]
.endm
.macro ST_SUMS X, vr, vi
  v_add_f64 %[t1], %[t1], %[t2]
  v_add_f64 %[t0], %[t0], -%[t3]
  v_add_f64 %[t1], %[t1], s[\X+2*\vi:\X+2*\vi+1]
  v_add_f64 %[t0], %[t0], s[\X+2*\vr:\X+2*\vr+1]
.endm
.macro ST_FIRST X, wr, wi, vr, vi
  v_mul_f64 %[t2], s[\X+2*\wr:\X+2*\wr+1], %[y]
  v_mul_f64 %[t1], s[\X+2*\wi:\X+2*\wi+1], %[x]
  v_mul_f64 %[t0], s[\X+2*\wr:\X+2*\wr+1], %[x]
  v_mul_f64 %[t3], s[\X+2*\wi:\X+2*\wi+1], %[y]
  ST_SUMS \X, \vr, \vi
.endm
.macro ST_STEP X, vr, vi
  v_mul_f64 %[t3], %[t1], %[y]
  v_mul_f64 %[t1], %[t1], %[x]
  v_mul_f64 %[t2], %[t0], %[y]
  v_mul_f64 %[t0], %[t0], %[x]
  ST_SUMS \X, \vr, \vi
.endm
.macro ST_KICK
  v_mul_f64 %[t0], -%[chi], %[t0]
  v_mul_f64 %[t1], %[chi], %[t1]
  v_add_f64 %[px], %[px], %[t0]
  v_add_f64 %[py], %[py], %[t1]
.endm
.macro ST_KICK0 X, wr, wi
  v_mul_f64 %[t0], -%[chi], s[\X+2*\wr:\X+2*\wr+1]
  v_mul_f64 %[t1], %[chi], s[\X+2*\wi:\X+2*\wi+1]
  v_add_f64 %[px], %[px], %[t0]
  v_add_f64 %[py], %[py], %[t1]
.endm
.macro ST_ROT X, a, b
  v_mul_f64 %[t0], s[\X+2:\X+3], \a
  v_mul_f64 %[t1], s[\X+4:\X+5], \b
  v_mul_f64 %[t2], -s[\X+4:\X+5], \a
  v_mul_f64 %[t3], s[\X+2:\X+3], \b
  v_add_f64 \a, %[t0], %[t1]
  v_add_f64 \b, %[t2], %[t3]
.endm
)"
#endif

// One handler per record kind and SGPR set: X the set that holds the first
// eight words of the record, Y the other.  ST_PRO waits for the record's
// words, starts the loads of its words from the eighth on (into s[68:99])
// and of the next record's first eight (size: bytes of this one), and forms
// the jump target from the record's own word 0, which names the next
// record's handler: the jump does not wait for the next record's words.
// Handlers are laid out ST_HOT_SPACING bytes apart in the order of their
// kind, those of the second set ST_HOT_SET_B bytes after the first's
// (lattice_hot.h).  A word's first register is X + 2 w below word 8 and
// 52 + 2 w from there on.  exec is the mask of lanes still tracked, so that
// the aperture tests give the lost lanes directly.
#define ST_HOT_HANDLERS R"(
.macro ST_PRO X, Y, size
.if %c[stops]
  s_cmp_eq_u32 %[off], %[stop]
  s_cbranch_scc1 .Lstop%=
.endif
  s_waitcnt lgkmcnt(0)
.if \size > 128
  s_load_dwordx16 s[68:83], %[hot], %[off] offset:64
  s_load_dwordx16 s[84:99], %[hot], %[off] offset:128
.elseif \size > 96
  s_load_dwordx16 s[68:83], %[hot], %[off] offset:64
.elseif \size > 80
  s_load_dwordx8 s[68:75], %[hot], %[off] offset:64
.elseif \size > 64
  s_load_dwordx4 s[68:71], %[hot], %[off] offset:64
.endif
  s_add_u32 %[off], %[off], \size
  s_load_dwordx16 s[\Y:\Y+15], %[hot], %[off] offset:0
  s_add_u32 s34, %[base], s[\X]
.endm
.macro ST_MP X, N, c0
.if \N == 0
  ST_KICK0 \X, \c0, (\c0+1)
.else
  ST_FIRST \X, \c0, (\c0+1), (\c0+2), (\c0+3)
  .set st_j, 2
  .rept \N - 1
  .if st_j == 3
  s_waitcnt lgkmcnt(0)
  .endif
  .if \c0+2*st_j < 7
  ST_STEP \X, (\c0+2*st_j), (\c0+2*st_j+1)
  .elseif \c0+2*st_j == 7
  ST_STEP \X, 7, ((68-\X)/2)
  .else
  ST_STEP 52, (\c0+2*st_j), (\c0+2*st_j+1)
  .endif
  .set st_j, st_j+1
  .endr
  ST_KICK
.endif
.endm
.macro ST_HANDLERS X, Y, T
.p2align 10
.L\T\()table%=:
  s_waitcnt lgkmcnt(0)
  s_mov_b64 %[lost], 0
  s_mov_b32 %[info], s[\X+1]
  s_mov_b32 %[next], s[\X]
  s_branch .Lend%=
.p2align 10
  ST_SLOPES
  ST_PRO \X, \Y, 16
  ST_DRIFT \X, 1
  s_cbranch_scc1 .L\T\()lost%=
  s_setpc_b64 s[34:35]
.p2align 10
  ST_PRO \X, \Y, 24
  v_add_f64 %[x], %[x], s[\X+2:\X+3]
  v_add_f64 %[y], %[y], s[\X+4:\X+5]
  s_setpc_b64 s[34:35]
.p2align 10
  ST_PRO \X, \Y, 24
  ST_ROT \X, %[x], %[y]
  ST_ROT \X, %[px], %[py]
  s_setpc_b64 s[34:35]
.p2align 10
  ST_PRO \X, \Y, 48
  v_cmp_nge_f64 vcc, %[x], s[\X+2:\X+3]
  v_cmp_nle_f64 %[m], %[x], s[\X+4:\X+5]
  v_cmp_nge_f64 %[lost], %[y], s[\X+6:\X+7]
  s_or_b64 vcc, vcc, %[m]
  v_cmp_nle_f64 %[m], %[y], s[\X+8:\X+9]
  s_or_b64 vcc, vcc, %[lost]
  s_or_b64 vcc, vcc, %[m]
  s_cbranch_scc1 .L\T\()lost%=
  s_setpc_b64 s[34:35]
.p2align 10
  v_mul_f64 %[t0], %[x], %[x]
  v_mul_f64 %[t1], %[y], %[y]
  ST_PRO \X, \Y, 40
  v_mul_f64 %[t0], %[t0], s[\X+4:\X+5]
  v_mul_f64 %[t1], %[t1], s[\X+2:\X+3]
  v_add_f64 %[t0], %[t0], %[t1]
  v_cmp_nle_f64 vcc, %[t0], s[\X+6:\X+7]
  s_cbranch_vccnz .L\T\()lost%=
  s_setpc_b64 s[34:35]
.p2align 10
  ST_PRO \X, \Y, 8
  .set st_j, 0
  .rept %c[lines]
  s_load_dword s68, %[hot], %[off] offset:%c[ahead]+64*st_j
  .set st_j, st_j+1
  .endr
  s_setpc_b64 s[34:35]
  .set st_n, 0
  .rept 11
.p2align 10
  ST_PRO \X, \Y, (24+16*st_n)
  ST_MP \X, st_n, 1
  s_setpc_b64 s[34:35]
  .set st_n, st_n+1
  .endr
  .set st_n, 0
  .rept 11
.p2align 10
  ST_SLOPES
  ST_PRO \X, \Y, (32+16*st_n)
  ST_DRIFT \X, 1
  s_cbranch_scc1 .L\T\()lostm%=
  ST_MP \X, st_n, 2
  s_setpc_b64 s[34:35]
  .set st_n, st_n+1
  .endr
.p2align 10
.L\T\()lostm%=:
  s_or_b32 s[\X+1], s[\X+1], 1
.L\T\()lost%=:
  s_mov_b64 %[lost], vcc
  s_mov_b32 %[info], s[\X+1]
  s_mov_b32 %[next], s[\X]
  s_waitcnt lgkmcnt(0)
  s_branch .Lend%=
.endm
  s_mov_b64 %[exec], exec
  s_mov_b64 exec, %[act]
  s_load_dwordx16 s[36:51], %[hot], %[off] offset:0
  s_load_dwordx16 s[52:67], %[hot], %[off] offset:0
  s_getpc_b64 s[34:35]
.Lpc%=:
  s_add_u32 %[base], s34, .Latable%=-.Lpc%=
  s_addc_u32 s35, s35, 0
  s_add_u32 s34, %[base], 0xffff
  s_cselect_b32 %[info], -1, 0
  s_cbranch_scc1 .Lnone%=
  s_add_u32 s34, %[base], %[next]
  s_setpc_b64 s[34:35]
  ST_HANDLERS 36, 52, a
.org .Latable%=+%c[setb]
  ST_HANDLERS 52, 36, b
.Lstop%=:
.Lnone%=:
  s_mov_b64 %[lost], 0
  s_waitcnt lgkmcnt(0)
.Lend%=:
  s_mov_b64 exec, %[exec]
.purgem ST_SLOPES
.purgem ST_DRIFT
.purgem ST_FIRST
.purgem ST_STEP
.purgem ST_KICK
.purgem ST_KICK0
.purgem ST_ROT
.purgem ST_PRO
.purgem ST_MP
.purgem ST_HANDLERS
)"
#if defined( ST_FMA_BUILD )
#define ST_HOT_PURGE ""
#else
#define ST_HOT_PURGE ".purgem ST_SUMS\n"
#endif

// With STOP the walk also returns at the record at byte offset ``stop``,
// before running it (off = stop, lost = 0): one compare and branch more per
// record, for segments of a lattice.
template< bool STOP >
ST_DEV void hot_run( cptr_t hot, uint32_t& off, uint32_t& next, uint32_t const stop, Lane& L,
                     double const chi, uint64_t const act, uint64_t& lost, uint32_t& info )
{
#if defined( __HIP_DEVICE_COMPILE__ )
    double t0, t1, t2, t3;
    uint64_t m, exec;
    uint32_t base;
    asm volatile( ST_HOT_ARITH ST_HOT_HANDLERS ST_HOT_PURGE
        : [ x ] "+v"( L.x ), [ y ] "+v"( L.y ), [ px ] "+v"( L.px ), [ py ] "+v"( L.py ),
          [ z ] "+v"( L.zeta ), [ off ] "+s"( off ), [ next ] "+s"( next ), [ lost ] "=&s"( lost ),
          [ info ] "=&s"( info ), [ m ] "=&s"( m ), [ exec ] "=&s"( exec ), [ base ] "=&s"( base ), [ t0 ] "=&v"( t0 ),
          [ t1 ] "=&v"( t1 ), [ t2 ] "=&v"( t2 ), [ t3 ] "=&v"( t3 )
        : [ rpp ] "v"( L.rpp ), [ rvv ] "v"( L.rvv ), [ chi ] "v"( chi ), [ hot ] "s"( hot ),
          [ act ] "s"( act ), [ stop ] "s"( stop ), [ stops ] "n"( STOP ? 1 : 0 ),
          [ lines ] "n"( ST_HOT_TOUCH_LINES ), [ ahead ] "n"( ST_HOT_TOUCH_AHEAD ),
          [ setb ] "n"( ST_HOT_SET_B )
        : "vcc", "scc", ST_HOT_SGPRS );
#endif
}

// The one-set walk of track_hot2.h (eight waves per SIMD).
ST_DEV void hot_run_one( cptr_t hot, uint32_t& off, uint32_t& next, Lane& L, double const chi,
                         uint64_t const act, uint64_t& lost, uint32_t& info );

// The lanes ``lost`` leave at the element of the packed record r: their
// state is stored, with path length s (bits).
template< class PA >
ST_DEV void hot_lose( const PA& pa, int64_t i, Lane& L, uint64_t lost, uint64_t& act, uint64_t s,
                      int64_t at_element, int64_t at_turn )
{
    if( lane_in( lost ) )
    {
        L.s = __longlong_as_double( ( long long )s );
        store_lane_state( pa.view(), i, L, 0, at_element, at_turn );
    }
    act &= ~lost;
}

// The hot records from byte offset off (handler offset next) to the END
// record, or with STOP to the record at byte offset stop, for lanes that
// came to off with the path length the stream holds for it: the element loop
// of track_lean.h's lean_turn<HEAVY, false> with the records of the hot
// kinds run by hot_run.  False when nothing was run (hot_run, info = ~0).
template< bool HEAVY, bool STOP, bool ONE_SET = false, class PA >
ST_DEV bool hot_walk( const PA& pa, int64_t i, int64_t li, cptr_t lat, cptr_t hot, uint32_t off,
                      uint32_t next, uint32_t stop, Lane& L, double chi, uint64_t& act,
                      int32_t& status, int64_t start, int64_t at_turn )
{
    while( act != 0u )
    {
        if( STOP && off == stop ) break;
        uint64_t lost;
        uint32_t info;
        if constexpr( ONE_SET ) hot_run_one( hot, off, next, L, chi, act, lost, info );
        else hot_run< STOP >( hot, off, next, stop, L, chi, act, lost, info );
        if( info == ~0u ) return false;
        if( lost != 0u )                              // at a Drift or an aperture
        {
            cptr_t const r = rec_at( lat, info & ~1u );
            uint64_t const s = ST_REC_OP( r[ 0 ] ) == ST_OP_DRIFT ? r[ 3 ] : rec_at( hot, off - 8u )[ 0 ];
            hot_lose( pa, i, L, lost, act, s, start + ri( r, 1 ), at_turn );
            if( info & 1u )                           // the Multipole of the same hot record
            {
                cptr_t const m = r + ST_REC_LEN( r[ 0 ] );
                multipole( L, chi, m + ST_REC_PAYLOAD, ST_REC_AUX( m[ 0 ] ), L.delta );
            }
            continue;
        }
        if( STOP && off == stop ) break;
        cptr_t const x = rec_at( hot, off );
        cptr_t const r = rec_at( lat, info );
        uint64_t const h = r[ 0 ];
        unsigned const op = ST_REC_OP( h );
        if( op == ST_OP_END ) break;
        off += 16u;
        if( op == ST_OP_MULTIPOLE )                   // curvature or a high order
        {
            multipole( L, chi, r + ST_REC_PAYLOAD, ST_REC_AUX( h ), L.delta );
            continue;
        }
        bool fail = false;
        // a monitor stores the particle's s
        if constexpr( HEAVY ) L.s = __longlong_as_double( ( long long )x[ 1 ] );
        bool const ok = lean_other< HEAVY >( op, ST_REC_AUX( h ), r + ST_REC_PAYLOAD, L, pa, li,
                                             lane_in( act ), start + ri( r, 1 ), at_turn, fail );
        L.s = 0.0;
        uint64_t const gone = ballot( !ok ) & act;
        if( gone != 0u )
        {
            if( lane_in( gone ) && fail ) status = -1;
            hot_lose( pa, i, L, gone, act, x[ 1 ], start + ri( r, 1 ), at_turn );
        }
    }
    return true;
}

// As track_lean_lane, the turns through the hot stream.  A turn on which
// some lane starts at s != 0 (the first of a call that starts mid-lattice)
// runs the loop with a per-lane s.
template< bool HEAVY, bool ONE_SET = false, class PA >
ST_DEV void track_hot_lane( const PA& pa, const int32_t* list, int64_t n_lanes, int64_t tid, cptr_t lat,
                            cptr_t hot, int64_t n_elem, int64_t until_turn, int64_t max_turns,
                            int32_t* status_out, const WavePrio& wp )
{
    track_lean_lane< HEAVY >( pa, list, n_lanes, tid, lat, n_elem, until_turn, max_turns, status_out, wp,
        [ & ]( int64_t i, int64_t li, Lane& L, double chi, uint64_t& act, int32_t& status, int64_t start,
               int64_t at_turn )
        {
            // a stream starts with a TOUCH record
            if( !hot_walk< HEAVY, false, ONE_SET >( pa, i, li, lat, hot, 0u, ST_HOT_TOUCH * ST_HOT_SPACING, 0u, L,
                                           chi, act, status, start, at_turn ) )
                lean_turn< HEAVY, true >( pa, i, li, lat, L, chi, act, status, start, at_turn );
        } );
}

}  // namespace st
