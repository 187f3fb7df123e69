// The scheduled record walk (track_hot.h) for launches that fill the chip:
// one or two particles per lane at eight waves per SIMD (device code,
// gfx950).
//
// With eight waves on a SIMD the other waves cover what one waits for, and
// the FP64 instructions themselves are the bound; what counts is that little
// else is issued.  So a record's words are read when it runs, exactly as
// many as it has, into one set of 32 SGPRs (words past the 16th replace the
// first ones once those are used): 64 VGPRs and 80 SGPRs hold the walk, and
// the scalar cache, which returns one dword per cycle, is asked for no more
// than the record.  The hot stream, its jumps and the maps are those of
// track_hot.h; a handler's place is twice its offset there
// (ST_HOT2_SPACING), both of that walk's register sets map to one.
//
// Bound by the FP64 issue: two particles per lane, every SIMD with eight
// waves, 1,048,576 particles on the 20,000-element ring take 480 ns per
// element in the FMA build and 777 in the exact one (the compiled loop for
// two: 506 to 515 and 790); one per lane, 524,288 particles, FMA: 261 (two
// register sets 301, the compiled loop 298).
#pragma once

#include "track_hot.h"

#define ST_HOT2_SPACING 2048

namespace st
{
// Arithmetic of particle P (operand names end in P), as in track_hot.h: the
// same operations in the same order.  W: first SGPR of the record's words.
#if defined( ST_FMA_BUILD )
#define ST_HOT2_ARITH( P )                                                                       \
    ".macro ST_SLOPES" #P "\n"                                                                   \
    " v_mul_f64 %[a" #P "], %[px" #P "], %[rpp" #P "]\n"                                         \
    " v_mul_f64 %[b" #P "], %[py" #P "], %[rpp" #P "]\n"                                         \
    ".endm\n"                                                                                    \
    ".macro ST_DRIFT" #P " l\n"                                                                  \
    " v_fma_f64 %[x" #P "], %[a" #P "], s[\\l:\\l+1], %[x" #P "]\n"                              \
    " v_fma_f64 %[y" #P "], %[b" #P "], s[\\l:\\l+1], %[y" #P "]\n"                              \
    " v_mul_f64 %[b" #P "], %[b" #P "], %[b" #P "]\n"                                            \
    " v_cmp_nlt_f64 vcc, |%[x" #P "]|, 1.0\n"                                                    \
    " v_cmp_nlt_f64 %[l" #P "], |%[y" #P "]|, 1.0\n"                                             \
    " v_fma_f64 %[a" #P "], %[a" #P "], %[a" #P "], %[b" #P "]\n"                                \
    " v_fma_f64 %[a" #P "], %[a" #P "], 0.5, 1.0\n"                                              \
    " v_add_f64 %[a" #P "], %[rvv" #P "], -%[a" #P "]\n"                                         \
    " s_or_b64 %[l" #P "], %[l" #P "], vcc\n"                                                    \
    " v_fma_f64 %[z" #P "], %[a" #P "], s[\\l:\\l+1], %[z" #P "]\n"                              \
    ".endm\n"                                                                                    \
    ".macro ST_FIRST" #P " wr, t, vr, vi\n"                                                      \
    " v_fma_f64 %[d" #P "], \\t, %[x" #P "], s[\\vi:\\vi+1]\n"                                   \
    " v_fma_f64 %[c" #P "], -\\t, %[y" #P "], s[\\vr:\\vr+1]\n"                                  \
    ".endm\n"                                                                                    \
    ".macro ST_SECOND" #P " wr\n"                                                                \
    " v_fma_f64 %[b" #P "], s[\\wr:\\wr+1], %[y" #P "], %[d" #P "]\n"                            \
    " v_fma_f64 %[a" #P "], s[\\wr:\\wr+1], %[x" #P "], %[c" #P "]\n"                            \
    ".endm\n"                                                                                    \
    ".macro ST_STEP" #P " vr, vi\n"                                                              \
    " v_fma_f64 %[d" #P "], %[b" #P "], %[x" #P "], s[\\vi:\\vi+1]\n"                            \
    " v_fma_f64 %[c" #P "], -%[b" #P "], %[y" #P "], s[\\vr:\\vr+1]\n"                           \
    " v_fma_f64 %[b" #P "], %[a" #P "], %[y" #P "], %[d" #P "]\n"                                \
    " v_fma_f64 %[a" #P "], %[a" #P "], %[x" #P "], %[c" #P "]\n"                                \
    ".endm\n"                                                                                    \
    ".macro ST_KICK" #P "\n"                                                                     \
    " v_fma_f64 %[px" #P "], -%[chi" #P "], %[a" #P "], %[px" #P "]\n"                           \
    " v_fma_f64 %[py" #P "], %[chi" #P "], %[b" #P "], %[py" #P "]\n"                            \
    ".endm\n"                                                                                    \
    ".macro ST_KICKZ" #P " wr, wi\n"                                                             \
    " v_fma_f64 %[px" #P "], -%[chi" #P "], s[\\wr:\\wr+1], %[px" #P "]\n"                       \
    " v_fma_f64 %[py" #P "], %[chi" #P "], s[\\wi:\\wi+1], %[py" #P "]\n"                        \
    ".endm\n"                                                                                    \
    ".macro ST_ROT" #P " c, s, u, v\n"                                                           \
    " v_mul_f64 %[a" #P "], s[\\s:\\s+1], \\v\n"                                                 \
    " v_mul_f64 %[b" #P "], s[\\s:\\s+1], \\u\n"                                                 \
    " v_fma_f64 \\u, s[\\c:\\c+1], \\u, %[a" #P "]\n"                                            \
    " v_fma_f64 \\v, s[\\c:\\c+1], \\v, -%[b" #P "]\n"                                           \
    ".endm\n"
#else
#define ST_HOT2_ARITH( P )                                                                       \
    ".macro ST_SLOPES" #P "\n"                                                                   \
    " v_mul_f64 %[a" #P "], %[px" #P "], %[rpp" #P "]\n"                                         \
    " v_mul_f64 %[b" #P "], %[py" #P "], %[rpp" #P "]\n"                                         \
    ".endm\n"                                                                                    \
    ".macro ST_DRIFT" #P " l\n"                                                                  \
    " v_mul_f64 %[c" #P "], %[a" #P "], s[\\l:\\l+1]\n"                                          \
    " v_mul_f64 %[d" #P "], %[b" #P "], s[\\l:\\l+1]\n"                                          \
    " v_add_f64 %[x" #P "], %[x" #P "], %[c" #P "]\n"                                            \
    " v_add_f64 %[y" #P "], %[y" #P "], %[d" #P "]\n"                                            \
    " v_mul_f64 %[a" #P "], %[a" #P "], %[a" #P "]\n"                                            \
    " v_mul_f64 %[b" #P "], %[b" #P "], %[b" #P "]\n"                                            \
    " v_cmp_nlt_f64 vcc, |%[x" #P "]|, 1.0\n"                                                    \
    " v_cmp_nlt_f64 %[l" #P "], |%[y" #P "]|, 1.0\n"                                             \
    " v_add_f64 %[a" #P "], %[a" #P "], %[b" #P "]\n"                                            \
    " v_mul_f64 %[a" #P "], %[a" #P "], 0.5\n"                                                   \
    " v_add_f64 %[a" #P "], %[a" #P "], 1.0\n"                                                   \
    " s_or_b64 %[l" #P "], %[l" #P "], vcc\n"                                                    \
    " v_add_f64 %[a" #P "], %[rvv" #P "], -%[a" #P "]\n"                                         \
    " v_mul_f64 %[a" #P "], %[a" #P "], s[\\l:\\l+1]\n"                                          \
    " v_add_f64 %[z" #P "], %[z" #P "], %[a" #P "]\n"                                            \
    ".endm\n"                                                                                    \
    ".macro ST_SUMS" #P " vr, vi\n"                                                              \
    " v_add_f64 %[b" #P "], %[b" #P "], %[c" #P "]\n"                                            \
    " v_add_f64 %[a" #P "], %[a" #P "], -%[d" #P "]\n"                                           \
    " v_add_f64 %[b" #P "], %[b" #P "], s[\\vi:\\vi+1]\n"                                        \
    " v_add_f64 %[a" #P "], %[a" #P "], s[\\vr:\\vr+1]\n"                                        \
    ".endm\n"                                                                                    \
    ".macro ST_FIRST" #P " wr, wi, vr, vi\n"                                                     \
    " v_mul_f64 %[c" #P "], s[\\wr:\\wr+1], %[y" #P "]\n"                                        \
    " v_mul_f64 %[b" #P "], s[\\wi:\\wi+1], %[x" #P "]\n"                                        \
    " v_mul_f64 %[a" #P "], s[\\wr:\\wr+1], %[x" #P "]\n"                                        \
    " v_mul_f64 %[d" #P "], s[\\wi:\\wi+1], %[y" #P "]\n"                                        \
    " ST_SUMS" #P " \\vr, \\vi\n"                                                                \
    ".endm\n"                                                                                    \
    ".macro ST_STEP" #P " vr, vi\n"                                                              \
    " v_mul_f64 %[d" #P "], %[b" #P "], %[y" #P "]\n"                                            \
    " v_mul_f64 %[b" #P "], %[b" #P "], %[x" #P "]\n"                                            \
    " v_mul_f64 %[c" #P "], %[a" #P "], %[y" #P "]\n"                                            \
    " v_mul_f64 %[a" #P "], %[a" #P "], %[x" #P "]\n"                                            \
    " ST_SUMS" #P " \\vr, \\vi\n"                                                                \
    ".endm\n"                                                                                    \
    ".macro ST_KICK" #P "\n"                                                                     \
    " v_mul_f64 %[a" #P "], -%[chi" #P "], %[a" #P "]\n"                                         \
    " v_mul_f64 %[b" #P "], %[chi" #P "], %[b" #P "]\n"                                          \
    " v_add_f64 %[px" #P "], %[px" #P "], %[a" #P "]\n"                                          \
    " v_add_f64 %[py" #P "], %[py" #P "], %[b" #P "]\n"                                          \
    ".endm\n"                                                                                    \
    ".macro ST_KICKZ" #P " wr, wi\n"                                                             \
    " v_mul_f64 %[a" #P "], -%[chi" #P "], s[\\wr:\\wr+1]\n"                                     \
    " v_mul_f64 %[b" #P "], %[chi" #P "], s[\\wi:\\wi+1]\n"                                      \
    " v_add_f64 %[px" #P "], %[px" #P "], %[a" #P "]\n"                                          \
    " v_add_f64 %[py" #P "], %[py" #P "], %[b" #P "]\n"                                          \
    ".endm\n"                                                                                    \
    ".macro ST_ROT" #P " c, s, u, v\n"                                                           \
    " v_mul_f64 %[a" #P "], s[\\c:\\c+1], \\u\n"                                                 \
    " v_mul_f64 %[b" #P "], s[\\s:\\s+1], \\v\n"                                                 \
    " v_mul_f64 %[c" #P "], -s[\\s:\\s+1], \\u\n"                                                \
    " v_mul_f64 %[d" #P "], s[\\c:\\c+1], \\v\n"                                                 \
    " v_add_f64 \\u, %[a" #P "], %[b" #P "]\n"                                                   \
    " v_add_f64 \\v, %[c" #P "], %[d" #P "]\n"                                                   \
    ".endm\n"
#endif

// The other maps of particle P, and the macros' removal.
#define ST_HOT2_MAPS( P )                                                                        \
    ".macro ST_SHIFT" #P " dx, dy\n"                                                             \
    " v_add_f64 %[x" #P "], %[x" #P "], s[\\dx:\\dx+1]\n"                                        \
    " v_add_f64 %[y" #P "], %[y" #P "], s[\\dy:\\dy+1]\n"                                        \
    ".endm\n"                                                                                    \
    ".macro ST_TURN" #P " c, s\n"                                                                \
    " ST_ROT" #P " \\c, \\s, %[x" #P "], %[y" #P "]\n"                                           \
    " ST_ROT" #P " \\c, \\s, %[px" #P "], %[py" #P "]\n"                                         \
    ".endm\n"                                                                                    \
    ".macro ST_RECT" #P " w\n"                                                                   \
    " v_cmp_nge_f64 vcc, %[x" #P "], s[\\w:\\w+1]\n"                                             \
    " v_cmp_nle_f64 %[l" #P "], %[x" #P "], s[\\w+2:\\w+3]\n"                                    \
    " v_cmp_nge_f64 %[m], %[y" #P "], s[\\w+4:\\w+5]\n"                                          \
    " s_or_b64 %[l" #P "], %[l" #P "], vcc\n"                                                    \
    " v_cmp_nle_f64 vcc, %[y" #P "], s[\\w+6:\\w+7]\n"                                           \
    " s_or_b64 %[l" #P "], %[l" #P "], %[m]\n"                                                   \
    " s_or_b64 %[l" #P "], %[l" #P "], vcc\n"                                                    \
    ".endm\n"                                                                                    \
    ".macro ST_ELL" #P " w\n"                                                                    \
    " v_mul_f64 %[a" #P "], %[x" #P "], %[x" #P "]\n"                                            \
    " v_mul_f64 %[b" #P "], %[y" #P "], %[y" #P "]\n"                                            \
    " v_mul_f64 %[a" #P "], %[a" #P "], s[\\w+2:\\w+3]\n"                                        \
    " v_mul_f64 %[b" #P "], %[b" #P "], s[\\w:\\w+1]\n"                                          \
    " v_add_f64 %[a" #P "], %[a" #P "], %[b" #P "]\n"                                            \
    " v_cmp_nle_f64 %[l" #P "], %[a" #P "], s[\\w+4:\\w+5]\n"                                    \
    ".endm\n"
#if defined( ST_FMA_BUILD )
#define ST_HOT2_PURGE_SUMS( P ) ".purgem ST_SECOND" #P "\n"
#else
#define ST_HOT2_PURGE_SUMS( P ) ".purgem ST_SUMS" #P "\n"
#endif
#define ST_HOT2_PURGE( P )                                                                       \
    ".purgem ST_SLOPES" #P "\n.purgem ST_DRIFT" #P "\n.purgem ST_FIRST" #P "\n.purgem ST_STEP" #P \
    "\n.purgem ST_KICK" #P "\n.purgem ST_KICKZ" #P "\n.purgem ST_ROT" #P "\n.purgem ST_SHIFT" #P \
    "\n.purgem ST_TURN" #P "\n.purgem ST_RECT" #P "\n.purgem ST_ELL" #P "\n" ST_HOT2_PURGE_SUMS( P )

// A map for one particle, or for both.
#define ST_HOT2_ONE( NAME, ARGS, CALL )                                                          \
    ".macro ST_" NAME " " ARGS "\n ST_" NAME "0 " CALL "\n.endm\n"
#define ST_HOT2_TWO( NAME, ARGS, CALL )                                                          \
    ".macro ST_" NAME " " ARGS "\n ST_" NAME "0 " CALL "\n ST_" NAME "1 " CALL "\n.endm\n"
#define ST_HOT2_EACH( F )                                                                        \
    F( "SLOPES", "", "" )                                                                        \
    F( "DRIFT", "l", "\\l" )                                                                     \
    F( "STEP", "vr, vi", "\\vr, \\vi" )                                                          \
    F( "KICK", "", "" )                                                                          \
    F( "KICKZ", "wr, wi", "\\wr, \\wi" )                                                         \
    F( "SHIFT", "dx, dy", "\\dx, \\dy" )                                                         \
    F( "TURN", "c, s", "\\c, \\s" )                                                              \
    F( "RECT", "w", "\\w" )                                                                      \
    F( "ELL", "w", "\\w" )

// First step of Horner's rule, from the highest coefficient (wr, wi).  A
// VALU instruction reads one SGPR operand: the FMA build needs wi in a VGPR
// (one copy for both particles).
#if defined( ST_FMA_BUILD )
#define ST_HOT2_FIRST_ONE                                                                        \
    ".macro ST_FIRST wr, wi, vr, vi\n v_mov_b64 %[b0], s[\\wi:\\wi+1]\n"                         \
    " ST_FIRST0 \\wr, %[b0], \\vr, \\vi\n ST_SECOND0 \\wr\n.endm\n"
#define ST_HOT2_FIRST_TWO                                                                        \
    ".macro ST_FIRST wr, wi, vr, vi\n v_mov_b64 %[b0], s[\\wi:\\wi+1]\n"                         \
    " ST_FIRST0 \\wr, %[b0], \\vr, \\vi\n ST_FIRST1 \\wr, %[b0], \\vr, \\vi\n"                  \
    " ST_SECOND0 \\wr\n ST_SECOND1 \\wr\n.endm\n"
#else
#define ST_HOT2_FIRST_ONE ST_HOT2_ONE( "FIRST", "wr, wi, vr, vi", "\\wr, \\wi, \\vr, \\vi" )
#define ST_HOT2_FIRST_TWO ST_HOT2_TWO( "FIRST", "wr, wi, vr, vi", "\\wr, \\wi, \\vr, \\vi" )
#endif

// Lanes lost (l0, l1 of the lanes tracked) -> SCC.
#define ST_HOT2_LOST_ONE                                                                         \
    ".macro ST_LOST\n s_and_b64 %[l0], %[l0], %[act0]\n.endm\n"
#define ST_HOT2_LOST_TWO                                                                         \
    ".macro ST_LOST\n s_and_b64 %[l0], %[l0], %[act0]\n s_and_b64 %[l1], %[l1], %[act1]\n"       \
    " s_or_b64 vcc, %[l0], %[l1]\n.endm\n"
#define ST_HOT2_EXEC_ONE ".macro ST_EXEC\n s_mov_b64 exec, %[act0]\n.endm\n"
#define ST_HOT2_EXEC_TWO ".macro ST_EXEC\n s_or_b64 exec, %[act0], %[act1]\n.endm\n"
#define ST_HOT2_NONE_ONE ".macro ST_NONE\n s_mov_b64 %[l0], 0\n.endm\n"
#define ST_HOT2_NONE_TWO ".macro ST_NONE\n s_mov_b64 %[l0], 0\n s_mov_b64 %[l1], 0\n.endm\n"

// The walk.  Words of the record: s[36:67], word w (mod 16) at 36 + 2 w.
// Jump target s[34:35], code base s68.  The handlers stand in a section of
// their own: 60 KB between a function's blocks would put its branches out of
// reach.  Jumps set the low half of the target only, so the walk runs where
// the handlers and the place to return to lie in one 4 GiB block, and
// otherwise returns info = ~0.
#define ST_HOT2_WALK R"(
.macro ST_LOAD size
.if \size > 96
  s_load_dwordx16 s[36:51], %[hot], %[off] offset:0
  s_load_dwordx16 s[52:67], %[hot], %[off] offset:64
.elseif \size > 80
  s_load_dwordx16 s[36:51], %[hot], %[off] offset:0
  s_load_dwordx8 s[52:59], %[hot], %[off] offset:64
.elseif \size > 64
  s_load_dwordx16 s[36:51], %[hot], %[off] offset:0
  s_load_dwordx4 s[52:55], %[hot], %[off] offset:64
.elseif \size > 32
  s_load_dwordx16 s[36:51], %[hot], %[off] offset:0
.elseif \size > 16
  s_load_dwordx8 s[36:43], %[hot], %[off] offset:0
.elseif \size > 8
  s_load_dwordx4 s[36:39], %[hot], %[off] offset:0
.else
  s_load_dwordx2 s[36:37], %[hot], %[off] offset:0
.endif
.endm
.macro ST_GOT size
  s_waitcnt lgkmcnt(0)
  s_add_u32 %[off], %[off], \size
  s_and_b32 %[next], s36, 0x7fff
  s_mov_b32 %[info], s37
  s_lshl1_add_u32 s34, %[next], s68
.endm
.macro ST_MP N, c0, size
.if \N == 0
  ST_KICKZ (36+2*\c0), (38+2*\c0)
.else
  ST_FIRST (36+2*\c0), (38+2*\c0), (40+2*\c0), (42+2*\c0)
  .set st_j, 2
  .rept \N - 1
  .if (\c0+2*\N+1 > 15) && (st_j == 4)
  s_add_u32 %[info], %[off], 128-\size
  s_load_dwordx16 s[36:51], %[hot], %[info] offset:0
  .endif
  .if (\c0+2*\N+1 > 15) && (st_j == 7)
  s_waitcnt lgkmcnt(0)
  .endif
  ST_STEP (36+2*((\c0+2*st_j)&15)), (36+2*((\c0+2*st_j+1)&15))
  .set st_j, st_j+1
  .endr
  ST_KICK
.endif
.endm
  s_mov_b64 %[exec], exec
  ST_EXEC
  s_getpc_b64 s[34:35]
.Lpc%=:
  s_add_u32 s68, s34, .Ltable%=@rel32@lo+4
  s_addc_u32 s36, s35, .Ltable%=@rel32@hi+12
  s_add_u32 %[ret], s34, .Lend%=-.Lpc%=
  s_cselect_b32 %[info], -1, 0
  s_cmp_lg_u32 s35, s36
  s_cselect_b32 %[info], -1, %[info]
  s_add_u32 s34, s68, 0x1ffff
  s_cselect_b32 %[info], -1, %[info]
  s_cmp_eq_u32 %[info], -1
  s_cbranch_scc1 .Lnone%=
  s_and_b32 %[next], %[next], 0x7fff
  s_lshl1_add_u32 s34, %[next], s68
  s_setpc_b64 s[34:35]
.Lnone%=:
  ST_NONE
.Lend%=:
  s_mov_b64 exec, %[exec]
.pushsection .text.st_hot2,"ax",@progbits
.p2align 11
.Ltable%=:
  ST_LOAD 16
  s_waitcnt lgkmcnt(0)
  s_mov_b32 %[info], s37
  s_and_b32 %[next], s36, 0x7fff
  ST_NONE
  s_branch .Lback%=
.p2align 11
  ST_LOAD 16
  ST_SLOPES
  ST_GOT 16
  ST_DRIFT 38
  ST_LOST
  s_cbranch_scc1 .Lback%=
  s_setpc_b64 s[34:35]
.p2align 11
  ST_LOAD 24
  ST_GOT 24
  ST_SHIFT 38, 40
  s_setpc_b64 s[34:35]
.p2align 11
  ST_LOAD 24
  ST_GOT 24
  ST_TURN 38, 40
  s_setpc_b64 s[34:35]
.p2align 11
  ST_LOAD 48
  ST_GOT 48
  ST_RECT 38
  ST_LOST
  s_cbranch_scc1 .Lback%=
  s_setpc_b64 s[34:35]
.p2align 11
  ST_LOAD 40
  ST_GOT 40
  ST_ELL 38
  ST_LOST
  s_cbranch_scc1 .Lback%=
  s_setpc_b64 s[34:35]
.p2align 11
  ST_LOAD 8
  ST_GOT 8
  s_setpc_b64 s[34:35]
  .set st_n, 0
  .rept 11
.p2align 11
  ST_LOAD (24+16*st_n)
  ST_GOT (24+16*st_n)
  ST_MP st_n, 1, (24+16*st_n)
  s_setpc_b64 s[34:35]
  .set st_n, st_n+1
  .endr
  .set st_n, 0
  .rept 11
.p2align 11
  ST_LOAD (32+16*st_n)
  ST_SLOPES
  ST_GOT (32+16*st_n)
  ST_DRIFT 38
  ST_LOST
  s_cbranch_scc1 .Llostm%=
  ST_MP st_n, 2, (32+16*st_n)
  s_setpc_b64 s[34:35]
  .set st_n, st_n+1
  .endr
.Llostm%=:
  s_or_b32 %[info], %[info], 1
.Lback%=:
  s_mov_b32 s34, %[ret]
  s_setpc_b64 s[34:35]
.popsection
.purgem ST_LOAD
.purgem ST_GOT
.purgem ST_MP
.purgem ST_LOST
.purgem ST_EXEC
.purgem ST_NONE
.purgem ST_SLOPES
.purgem ST_DRIFT
.purgem ST_FIRST
.purgem ST_STEP
.purgem ST_KICK
.purgem ST_KICKZ
.purgem ST_SHIFT
.purgem ST_TURN
.purgem ST_RECT
.purgem ST_ELL
)"

#define ST_HOT2_SGPRS                                                                            \
    "s34", "s35", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44", "s45", "s46",   \
    "s47", "s48", "s49", "s50", "s51", "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59",   \
    "s60", "s61", "s62", "s63", "s64", "s65", "s66", "s67", "s68"
// Runs hot records as hot_run (track_hot.h) does, from either walk's
// position, for one particle per lane or two.  info = ~0: nothing was run.
ST_DEV void hot_run_one( cptr_t hot, uint32_t& off, uint32_t& next, Lane& L, double const chi,
                         uint64_t const act, uint64_t& lost, uint32_t& info )
{
#if defined( __HIP_DEVICE_COMPILE__ )
    double a0, b0, c0, d0;
    uint64_t m, exec;
    uint32_t ret;
    asm volatile( ST_HOT2_ARITH( 0 ) ST_HOT2_MAPS( 0 ) ST_HOT2_EACH( ST_HOT2_ONE ) ST_HOT2_FIRST_ONE ST_HOT2_LOST_ONE
                  ST_HOT2_EXEC_ONE ST_HOT2_NONE_ONE ST_HOT2_WALK ST_HOT2_PURGE( 0 )
        : [ x0 ] "+v"( L.x ), [ y0 ] "+v"( L.y ), [ px0 ] "+v"( L.px ), [ py0 ] "+v"( L.py ),
          [ z0 ] "+v"( L.zeta ), [ off ] "+s"( off ), [ next ] "+s"( next ), [ l0 ] "=&s"( lost ),
          [ info ] "=&s"( info ), [ m ] "=&s"( m ), [ exec ] "=&s"( exec ), [ ret ] "=&s"( ret ), [ a0 ] "=&v"( a0 ),
          [ b0 ] "=&v"( b0 ), [ c0 ] "=&v"( c0 ), [ d0 ] "=&v"( d0 )
        : [ rpp0 ] "v"( L.rpp ), [ rvv0 ] "v"( L.rvv ), [ chi0 ] "v"( chi ), [ hot ] "s"( hot ),
          [ act0 ] "s"( act )
        : "vcc", "scc", ST_HOT2_SGPRS );
#endif
}

ST_DEV void hot_run_two( cptr_t hot, uint32_t& off, uint32_t& next, Lane& L0, Lane& L1, double const chi0,
                         double const chi1, uint64_t const act0, uint64_t const act1, uint64_t& lost0,
                         uint64_t& lost1, uint32_t& info )
{
#if defined( __HIP_DEVICE_COMPILE__ )
    double a0, b0, c0, d0, a1, b1, c1, d1;
    uint64_t m, exec;
    uint32_t ret;
    asm volatile( ST_HOT2_ARITH( 0 ) ST_HOT2_MAPS( 0 ) ST_HOT2_ARITH( 1 ) ST_HOT2_MAPS( 1 )
                  ST_HOT2_EACH( ST_HOT2_TWO ) ST_HOT2_FIRST_TWO ST_HOT2_LOST_TWO ST_HOT2_EXEC_TWO ST_HOT2_NONE_TWO
                  ST_HOT2_WALK ST_HOT2_PURGE( 0 ) ST_HOT2_PURGE( 1 )
        : [ x0 ] "+v"( L0.x ), [ y0 ] "+v"( L0.y ), [ px0 ] "+v"( L0.px ), [ py0 ] "+v"( L0.py ),
          [ z0 ] "+v"( L0.zeta ), [ x1 ] "+v"( L1.x ), [ y1 ] "+v"( L1.y ), [ px1 ] "+v"( L1.px ),
          [ py1 ] "+v"( L1.py ), [ z1 ] "+v"( L1.zeta ), [ off ] "+s"( off ), [ next ] "+s"( next ),
          [ l0 ] "=&s"( lost0 ), [ l1 ] "=&s"( lost1 ), [ info ] "=&s"( info ), [ m ] "=&s"( m ),
          [ exec ] "=&s"( exec ), [ ret ] "=&s"( ret ), [ a0 ] "=&v"( a0 ), [ b0 ] "=&v"( b0 ), [ c0 ] "=&v"( c0 ),
          [ d0 ] "=&v"( d0 ), [ a1 ] "=&v"( a1 ), [ b1 ] "=&v"( b1 ), [ c1 ] "=&v"( c1 ),
          [ d1 ] "=&v"( d1 )
        : [ rpp0 ] "v"( L0.rpp ), [ rvv0 ] "v"( L0.rvv ), [ chi0 ] "v"( chi0 ), [ rpp1 ] "v"( L1.rpp ),
          [ rvv1 ] "v"( L1.rvv ), [ chi1 ] "v"( chi1 ), [ hot ] "s"( hot ), [ act0 ] "s"( act0 ),
          [ act1 ] "s"( act1 )
        : "vcc", "scc", ST_HOT2_SGPRS );
#endif
}

// Two particles per lane: lane l of a wave tracks the particles of slots
// base + l and base + 64 + l (list entries, or indices without a list)
// through the same hot records (hot_run_two).  Each particle's maps, loss
// handling and stored values are those of track_lean_lane, bit for bit; what
// the pair shares is the record walk (scalar loads, jumps, apertures'
// branches).  Only the state the Drift and Multipole records use stays in
// registers (x, px, y, py, zeta, rpp, rvv and chi: 16 VGPRs a particle), so
// that the pair fits the 64 VGPRs of eight waves per SIMD:
//   * delta and psigma stay in memory: Cavity and DriftExact read delta
//     there, Cavity writes both back, and a store leaves them as they are;
//   * every turn starts at s = +0 and s after a drift is the record's, as
//     in lean_turn's turns without a per-lane s;
//   * at_element and at_turn are read back at a store (memory holds their
//     values at the start of the launch until then); the turns a lane has
//     left are a 32-bit count against the wave's turn counter.
// A tile with a particle that starts its turn at s != 0 runs through
// track_lean_lane, one half after the other, and so does one whose walk
// cannot run (hot_run, info = ~0).  That stands once, behind the turns: with
// a copy of it inside them the registers of every return from the walk (two
// a turn at least, END and a Cavity) went through scratch, nine doubles a
// lane.  FMA build, 1,048,576 particles, ns per element: 50 elements 864 ->
// 553, 402 elements 381 -> 361, 20,000 elements 501 and 500.
template< class PA >
ST_DEV void track_lean_lane2( const PA& pa, const int32_t* list, int64_t n_lanes,
                               int64_t base, cptr_t lat, cptr_t hot, int64_t n_elem, int64_t until_turn,
                               int64_t max_turns, int32_t* status_out, const WavePrio& wp = WavePrio() )
{
    constexpr int K = 2;
    int32_t idx[ K ], left[ K ];               // particle index, turns this launch
    double chi[ K ];
    Lane L[ K ];
    uint64_t act[ K ];
    bool mid = false;                          // a particle starts at s != 0
#pragma unroll
    for( int k = 0; k < K; ++k )
    {
        auto const& P = pa.view();
        int64_t const tid = base + 64 * k + __lane_id();
        bool const in_range = tid < n_lanes;
        int64_t const i = ( list != nullptr && in_range ) ? ( int64_t )list[ tid ] : tid;
        int64_t const li = in_range ? i : 0;
        idx[ k ] = ( int32_t )li;
        L[ k ].x = P.x[ li ]; L[ k ].px = P.px[ li ]; L[ k ].y = P.y[ li ];
        L[ k ].py = P.py[ li ]; L[ k ].zeta = P.zeta[ li ];
        L[ k ].rpp = P.rpp[ li ]; L[ k ].rvv = P.rvv[ li ];
        chi[ k ] = P.chi[ li ];
        int64_t const at_turn = P.at_turn[ li ];
        bool const active0 = in_range && n_elem > 0 && until_turn > at_turn && P.state[ li ] == 1;
        int64_t const stop = ( max_turns > 0 && until_turn - at_turn > max_turns ) ? at_turn + max_turns
                                                                                     : until_turn;
        left[ k ] = active0 ? ( int32_t )( stop - at_turn < INT32_MAX ? stop - at_turn : INT32_MAX ) : 0;
        mid = mid || ( active0 && __double_as_longlong( P.s[ li ] ) != 0 );
        act[ k ] = ballot( active0 );
    }
    bool one_by_one = ballot( mid ) != 0u || n_elem <= 0;
    bool failed = false;                       // a lane met a disabled / unknown map
    int64_t turns_done = 0;                    // by this wave, in this call
    // particle k's lanes ``lost`` at the element of the packed record r,
    // with path length s (bits)
    auto lose = [ & ]( int k, uint64_t lost, cptr_t r, uint64_t s )
    {
        if( lost == 0u ) return;
        if( lane_in( lost ) )
        {
            int64_t const j = idx[ k ];
            auto const& P = pa.view();
            store_hot_state( P, j, L[ k ], __longlong_as_double( ( long long )s ), 0,
                             P.at_element[ j ] + ri( r, 1 ), P.at_turn[ j ] + turns_done );
        }
        act[ k ] &= ~lost;
    };
    // a Multipole of any order, with or without curvature terms
    auto kick = [ & ]( cptr_t r )
    {
        unsigned const aux = ST_REC_AUX( r[ 0 ] );
#pragma unroll
        for( int k = 0; k < K; ++k )
        {
            double delta = 0.0;
            if( aux & ST_MP_CURV_FLAG )
            {
                int64_t j = idx[ k ];
                asm volatile( "" : "+v"( j ) );
                delta = pa.view().delta[ j ];
            }
            multipole( L[ k ], chi[ k ], r + ST_REC_PAYLOAD, aux, delta );
        }
    };
    if( !one_by_one ) wave_priority( wp, 0 );
    while( !one_by_one && ( act[ 0 ] | act[ 1 ] ) != 0u )
    {
        uint32_t off = 0, next = ST_HOT_TOUCH * ST_HOT_SPACING;  // a stream starts with a TOUCH
        while( ( act[ 0 ] | act[ 1 ] ) != 0u )
        {
            uint64_t lost[ K ];
            uint32_t info;
            hot_run_two( hot, off, next, L[ 0 ], L[ 1 ], chi[ 0 ], chi[ 1 ], act[ 0 ], act[ 1 ],
                         lost[ 0 ], lost[ 1 ], info );
            one_by_one = info == ~0u;          // nothing was run, in the first turn
            if( one_by_one ) break;
            cptr_t const r = rec_at( lat, info & ~1u );
            if( ( lost[ 0 ] | lost[ 1 ] ) != 0u )     // at a Drift or an aperture
            {
                uint64_t const s = ST_REC_OP( r[ 0 ] ) == ST_OP_DRIFT ? r[ 3 ] : rec_at( hot, off - 8u )[ 0 ];
                lose( 0, lost[ 0 ], r, s );
                lose( 1, lost[ 1 ], r, s );
                if( info & 1u ) kick( r + ST_REC_LEN( r[ 0 ] ) );   // the Multipole of the same hot record
                continue;
            }
            unsigned const op = ST_REC_OP( r[ 0 ] );
            if( op == ST_OP_END ) break;
            uint64_t const s = rec_at( hot, off )[ 1 ];
            off += 16u;
            if( op == ST_OP_MULTIPOLE ) { kick( r ); continue; }
            bool fail = false, ok[ K ];
            lean_other_hot2( op, r + ST_REC_PAYLOAD, L[ 0 ], L[ 1 ], pa, idx[ 0 ], idx[ 1 ],
                             lane_in( act[ 0 ] ), lane_in( act[ 1 ] ), fail, ok[ 0 ], ok[ 1 ] );
#pragma unroll
            for( int k = 0; k < K; ++k )
            {
                uint64_t const gone = ballot( !ok[ k ] ) & act[ k ];
                // fail depends on the record alone: the same in every lane
                if( gone != 0u ) failed = failed || fail;
                lose( k, gone, r, s );
            }
        }
        if( one_by_one ) break;
        ++turns_done;
#pragma unroll
        for( int k = 0; k < K; ++k )
        {
            uint64_t const fin = ballot( turns_done >= left[ k ] ) & act[ k ];
            if( fin != 0u )
            {
                if( lane_in( fin ) )
                {
                    int64_t const j = idx[ k ];
                    auto const& P = pa.view();
                    store_hot_state( P, j, L[ k ], 0.0, 1, P.at_element[ j ], P.at_turn[ j ] + turns_done );
                }
                act[ k ] &= ~fin;
            }
        }
        if( ( act[ 0 ] | act[ 1 ] ) != 0u ) wave_priority( wp, turns_done );
    }
    if( one_by_one )
    {
#pragma unroll 1
        for( int k = 0; k < K; ++k )
            track_lean_lane< false >( pa, list, n_lanes, base + 64 * k + __lane_id(), lat, n_elem,
                                      until_turn, max_turns, status_out, k == 0 ? wp : WavePrio() );
        return;
    }
    wave_priority_leave( wp, turns_done );
    if( failed && __lane_id() == 0 ) report_failure( status_out );
}

}  // namespace st
