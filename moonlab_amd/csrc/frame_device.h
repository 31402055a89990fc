// frame_device.h -- device side of the Pauli-rotation engine
// (frame_program.h): 16 tile amplitudes per thread in registers, rotations
// on them, LDS only to change the layout.
#pragma once

#include <hip/hip_runtime.h>

#include "frame_program.h"
#include "sv_device.h"

namespace mlx {

// One register value: a complex amplitude as a vector the compiler keeps in
// consecutive registers.
template <typename R> struct FVec;
template <> struct FVec<double> { using t = mlx_v2d; };
template <> struct FVec<float> { using t = mlx_v2f; };

template <typename R, bool NT>
__device__ __forceinline__ typename FVec<R>::t frame_ld(const cplx_t<R> *p)
{
    const cplx_t<R> x = ld<NT>(p);
    return typename FVec<R>::t{x.x, x.y};
}
template <typename R, bool NT>
__device__ __forceinline__ void frame_st(cplx_t<R> *p, const typename FVec<R>::t &x)
{
    st<NT>(p, cplx_t<R>{x.x, x.y});
}

// The rotation interpreter: the phases of a pass on one tile.
//
// 16 values per thread move between two fixed register sets V and W: each
// rotation reads one set and writes the other (two FMAs a value, nothing
// copied).  The arms are equally long blocks of straight code reached by a
// computed jump.  A compiled switch over the 81 arms became a tree of about
// twenty branches per rotation, which cost several times the 32 FMAs, and the
// compiler kept a third copy of the values around it; HIP C++ has neither a
// computed jump nor a way to hold values in given registers, so this part is
// assembly.  The assembler's macros write the arms out from the numbering
// FrameArm gives the planner: mlx_d the register bit the rotation pairs
// values across, mlx_z its sign functional; value j sits at I + 2 w j and
// goes to O + 2 w j, w registers a component.
//
// A rotation costs its arm, one 32-byte scalar load issued while the one
// before it runs, its sign (parities of a thread and a tile mask) and two
// jumps.  A layout change is 16 LDS writes, a barrier and 16 reads per
// thread.  The block leaves nothing in flight that it has started: every load
// is waited for inside it.  Global loads the caller has in flight stay so.  It
// reads and writes the tile's LDS and runs barriers ("memory": the caller's
// accesses stay on their side of it).
#define MLX_FRAME_MACROS \
    ".ifndef mlx_frame_macros\n"                                                                          \
    ".set mlx_frame_macros, 1\n"                                                                          \
    /* mlx_p = parity(mlx_z & mlx_j) */                                                                   \
    ".macro mlx_parity\n"                                                                                 \
    ".set mlx_p, mlx_z & mlx_j\n"                                                                         \
    ".set mlx_p, mlx_p ^ (mlx_p >> 1)\n"                                                                  \
    ".set mlx_p, (mlx_p ^ (mlx_p >> 2)) & 1\n"                                                            \
    ".endm\n"                                                                                             \
    /* v[o] = v[a] + T v[b], or minus */                                                                  \
    ".macro mlx_fma w, neg, T, o, b, a\n"                                                                 \
    ".if \\w == 2 && \\neg\n"                                                                             \
    "v_fma_f64 v[\\o:\\o+1], -v[\\T:\\T+1], v[\\b:\\b+1], v[\\a:\\a+1]\n"                                 \
    ".elseif \\w == 2\n"                                                                                  \
    "v_fma_f64 v[\\o:\\o+1], v[\\T:\\T+1], v[\\b:\\b+1], v[\\a:\\a+1]\n"                                  \
    ".elseif \\neg\n"                                                                                     \
    "v_fma_f32 v[\\o], -v[\\T], v[\\b], v[\\a]\n"                                                         \
    ".else\n"                                                                                             \
    "v_fma_f32 v[\\o], v[\\T], v[\\b], v[\\a]\n"                                                          \
    ".endif\n"                                                                                            \
    ".endm\n"                                                                                             \
    /* one arm: form 0 X y = a - i t s b, 1 Y y = a + t s b, 2 Z y = a (1 - i t s) */                     \
    ".macro mlx_rot w, I, O, T, form, tail\n"                                                             \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 16\n"                                                                                          \
    "mlx_parity\n"                                                                                        \
    ".set mlx_a, \\I + 2 * \\w * mlx_j\n"                                                                 \
    ".set mlx_o, \\O + 2 * \\w * mlx_j\n"                                                                 \
    ".if \\form == 2\n"                                                                                   \
    ".set mlx_b, mlx_a\n"                                                                                 \
    ".else\n"                                                                                             \
    ".set mlx_b, \\I + 2 * \\w * (mlx_j ^ (1 << mlx_d))\n"                                                \
    ".endif\n"                                                                                            \
    ".if \\form == 1\n"                                                                                   \
    "mlx_fma \\w, mlx_p, \\T, mlx_o, mlx_b, mlx_a\n"                                                      \
    "mlx_fma \\w, mlx_p, \\T, (mlx_o + \\w), (mlx_b + \\w), (mlx_a + \\w)\n"                              \
    ".else\n"                                                                                             \
    "mlx_fma \\w, mlx_p, \\T, mlx_o, (mlx_b + \\w), mlx_a\n"                                              \
    "mlx_fma \\w, (1 - mlx_p), \\T, (mlx_o + \\w), mlx_b, (mlx_a + \\w)\n"                                \
    ".endif\n"                                                                                            \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    "s_branch \\tail\n"                                                                                   \
    ".endm\n"                                                                                             \
    /* all arms from set I to set O, in FrameArm order */                                                 \
    ".macro mlx_arms w, I, O, T, tail\n"                                                                  \
    ".set mlx_f, 0\n"                                                                                     \
    ".rept 2\n"                                                                                           \
    ".set mlx_d, 0\n"                                                                                     \
    ".rept 4\n"                                                                                           \
    ".set mlx_k, 0\n"                                                                                     \
    ".rept 8\n"                                                                                           \
    ".set mlx_z, (mlx_k & ((1 << mlx_d) - 1)) | ((mlx_k >> mlx_d) << (mlx_d + 1)) | (mlx_f << mlx_d)\n"   \
    "mlx_rot \\w, \\I, \\O, \\T, mlx_f, \\tail\n"                                                         \
    ".set mlx_k, mlx_k + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".set mlx_d, mlx_d + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".set mlx_f, mlx_f + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".set mlx_z, 0\n"                                                                                     \
    ".rept 16\n"                                                                                          \
    "mlx_rot \\w, \\I, \\O, \\T, 2, \\tail\n"                                                             \
    ".set mlx_z, mlx_z + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 32\n"                                                                                          \
    ".if \\w == 2\n"                                                                                      \
    "v_mul_f64 v[\\O+2*mlx_j:\\O+2*mlx_j+1], v[\\T:\\T+1], v[\\I+2*mlx_j:\\I+2*mlx_j+1]\n"                \
    ".else\n"                                                                                             \
    "v_mul_f32_e64 v[\\O+mlx_j], v[\\T], v[\\I+mlx_j]\n"                                                  \
    ".endif\n"                                                                                            \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    "s_branch \\tail\n"                                                                                   \
    ".endm\n"                                                                                             \
    /* T = tangent of the unit in s[H:H+7], sign: parities of its thread and tile masks; then jump to */  \
    /* arm s[H] of the table at s[B:B+1] (an arm is 32 x 8 + 4 bytes) */                                  \
    ".macro mlx_go w, H, T, B, tid, base\n"                                                               \
    "v_and_b32 v[\\T], s[\\H+1], \\tid\n"                                                                 \
    "s_and_b64 s[92:93], s[\\H+2:\\H+3], \\base\n"                                                        \
    "s_bcnt1_i32_b64 s92, s[92:93]\n"                                                                     \
    "v_bcnt_u32_b32 v[\\T], v[\\T], s92\n"                                                                \
    "s_mul_i32 s90, s[\\H], 260\n"                                                                        \
    "v_lshlrev_b32 v[\\T], 31, v[\\T]\n"                                                                  \
    "s_add_u32 s90, s90, s[\\B]\n"                                                                        \
    "s_addc_u32 s91, s[\\B+1], 0\n"                                                                       \
    ".if \\w == 2\n"                                                                                      \
    "v_xor_b32 v[\\T+1], s[\\H+5], v[\\T]\n"                                                              \
    "v_mov_b32 v[\\T], s[\\H+4]\n"                                                                        \
    ".else\n"                                                                                             \
    "v_xor_b32 v[\\T], s[\\H+6], v[\\T]\n"                                                                \
    ".endif\n"                                                                                            \
    "s_setpc_b64 s[90:91]\n"                                                                              \
    ".endm\n"                                                                                             \
    /* write set I to the LDS slots of the layout before (s[36:51]), addresses in A.. */                  \
    ".macro mlx_put w, I, A, S, lds\n"                                                                    \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 16\n"                                                                                          \
    "v_xad_u32 v[\\A+mlx_j], v[\\S], s[36+mlx_j], \\lds\n"                                                \
    ".if \\w == 2\n"                                                                                      \
    "ds_write_b128 v[\\A+mlx_j], v[\\I+4*mlx_j:\\I+4*mlx_j+3]\n"                                          \
    ".else\n"                                                                                             \
    "ds_write_b64 v[\\A+mlx_j], v[\\I+2*mlx_j:\\I+2*mlx_j+1]\n"                                           \
    ".endif\n"                                                                                            \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".endm\n"                                                                                             \
    /* the thread's slot in the new layout, a barrier, and set O from the slots of s[52:67] */            \
    ".macro mlx_get w, O, A, S, tid, lds\n"                                                               \
    "v_and_b32 v[\\A], s78, \\tid\n"                                                                      \
    "v_add_u32 v[\\S], \\tid, v[\\A]\n"                                                                   \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 3\n"                                                                                           \
    "v_and_b32 v[\\A], s[79+mlx_j], v[\\S]\n"                                                             \
    "v_add_u32 v[\\S], v[\\S], v[\\A]\n"                                                                  \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".set mlx_k, 5 - \\w\n"                                                                               \
    "v_lshrrev_b32 v[\\A], mlx_k, v[\\S]\n"                                                               \
    "v_lshrrev_b32 v[\\A+1], 2 * mlx_k, v[\\S]\n"                                                         \
    "v_xor_b32 v[\\A], v[\\A], v[\\A+1]\n"                                                                \
    "v_lshrrev_b32 v[\\A+1], 3 * mlx_k, v[\\S]\n"                                                         \
    "v_xor_b32 v[\\A], v[\\A], v[\\A+1]\n"                                                                \
    ".if \\w == 2\n"                                                                                      \
    "v_lshrrev_b32 v[\\A+1], 12, v[\\S]\n"                                                                \
    "v_xor_b32 v[\\A], v[\\A], v[\\A+1]\n"                                                                \
    ".endif\n"                                                                                            \
    "v_and_b32 v[\\A], (1 << mlx_k) - 1, v[\\A]\n"                                                        \
    "v_xor_b32 v[\\S], v[\\S], v[\\A]\n"                                                                  \
    "v_lshlrev_b32 v[\\S], 2 + \\w, v[\\S]\n"                                                             \
    "s_waitcnt lgkmcnt(0)\n"                                                                              \
    "s_barrier\n"                                                                                         \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 16\n"                                                                                          \
    "v_xad_u32 v[\\A+mlx_j], v[\\S], s[52+mlx_j], \\lds\n"                                                \
    ".if \\w == 2\n"                                                                                      \
    "ds_read_b128 v[\\O+4*mlx_j:\\O+4*mlx_j+3], v[\\A+mlx_j]\n"                                           \
    ".else\n"                                                                                             \
    "ds_read_b64 v[\\O+2*mlx_j:\\O+2*mlx_j+1], v[\\A+mlx_j]\n"                                            \
    ".endif\n"                                                                                            \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    "s_waitcnt lgkmcnt(0)\n"                                                                              \
    ".endm\n"                                                                                             \
    /* header of the next phase, its offsets and its first rotation */                                    \
    ".macro mlx_head\n"                                                                                   \
    "s_load_dwordx8 s[76:83], s[86:87], 0x0\n"                                                            \
    "s_load_dwordx16 s[36:51], s[86:87], 0x20\n"                                                          \
    "s_load_dwordx16 s[52:67], s[86:87], 0x60\n"                                                          \
    "s_load_dwordx8 s[68:75], s[86:87], 0xa0\n"                                                           \
    "s_waitcnt lgkmcnt(0)\n"                                                                              \
    ".endm\n"                                                                                             \
    ".macro mlx_copy w, I, O\n"                                                                           \
    ".set mlx_j, 0\n"                                                                                     \
    ".rept 16 * \\w\n"                                                                                    \
    "v_mov_b64 v[\\O+2*mlx_j:\\O+2*mlx_j+1], v[\\I+2*mlx_j:\\I+2*mlx_j+1]\n"                              \
    ".set mlx_j, mlx_j + 1\n"                                                                             \
    ".endr\n"                                                                                             \
    ".endm\n"                                                                                             \
    ".endif\n"                                                                                           

// V, W: first registers of the sets; T: the tangent; S: the thread's LDS slot
#define MLX_FRAME_LOOP(CW, V, W, T, S) \
    "s_mov_b64 s[86:87], %[p]\n"                                           \
    "s_mov_b32 s85, %[n]\n"                                                \
    "s_getpc_b64 s[88:89]\n"                                               \
    ".LfP%=:\n"                                                            \
    "s_add_u32 s94, s88, .LfA%= - .LfP%=\n"                                \
    "s_addc_u32 s95, s89, 0\n"                                             \
    "s_add_u32 s96, s88, .LfB%= - .LfP%=\n"                                \
    "s_addc_u32 s97, s89, 0\n"                                             \
    /* a phase entered with the values in V */                             \
    ".LfV%=:\n"                                                            \
    "mlx_head\n"                                                           \
    "s_cmp_eq_u32 s77, 0\n"                                                \
    "s_cbranch_scc1 .LfR%=\n"                                              \
    "mlx_put " CW ", " V ", " W ", " S ", %[lds]\n"                        \
    "s_branch .LfX%=\n"                                                    \
    /* a phase entered with the values in W (it changes the layout) */     \
    ".LfW%=:\n"                                                            \
    "mlx_head\n"                                                           \
    "mlx_put " CW ", " W ", " V ", " S ", %[lds]\n"                        \
    ".LfX%=:\n"                                                            \
    "mlx_get " CW ", " V ", " W ", " S ", %[tid], %[lds]\n"                \
    ".LfR%=:\n"                                                            \
    "s_mov_b32 s84, s76\n"                                                 \
    "s_add_u32 s86, s86, 0xa0\n"                                           \
    "s_addc_u32 s87, s87, 0\n"                                             \
    /* two rotations a turn, each fetched while the one before it runs */  \
    ".LfN%=:\n"                                                            \
    "s_load_dwordx8 s[76:83], s[86:87], 0x20\n"                            \
    "mlx_go " CW ", 68, " T ", 94, %[tid], %[base]\n"                      \
    ".LfA%=:\n"                                                            \
    "mlx_arms " CW ", " V ", " W ", " T ", .LfTA%=\n"                      \
    ".LfTA%=:\n"                                                           \
    "s_sub_u32 s84, s84, 1\n"                                              \
    "s_cmp_eq_u32 s84, 0\n"                                                \
    "s_cbranch_scc1 .LfEW%=\n"                                             \
    "s_waitcnt lgkmcnt(0)\n"                                               \
    "s_load_dwordx8 s[68:75], s[86:87], 0x40\n"                            \
    "s_add_u32 s86, s86, 64\n"                                             \
    "s_addc_u32 s87, s87, 0\n"                                             \
    "mlx_go " CW ", 76, " T ", 96, %[tid], %[base]\n"                      \
    ".LfB%=:\n"                                                            \
    "mlx_arms " CW ", " W ", " V ", " T ", .LfTB%=\n"                      \
    ".LfTB%=:\n"                                                           \
    "s_sub_u32 s84, s84, 1\n"                                              \
    "s_cmp_eq_u32 s84, 0\n"                                                \
    "s_waitcnt lgkmcnt(0)\n"                                               \
    "s_cbranch_scc0 .LfN%=\n"                                              \
    "s_sub_u32 s85, s85, 1\n"                                              \
    "s_cmp_eq_u32 s85, 0\n"                                                \
    "s_cbranch_scc0 .LfV%=\n"                                              \
    "s_branch .LfZ%=\n"                                                    \
    ".LfEW%=:\n"                                                           \
    "s_waitcnt lgkmcnt(0)\n"                                               \
    "s_add_u32 s86, s86, 32\n"                                             \
    "s_addc_u32 s87, s87, 0\n"                                             \
    "s_sub_u32 s85, s85, 1\n"                                              \
    "s_cmp_eq_u32 s85, 0\n"                                                \
    "s_cbranch_scc0 .LfW%=\n"                                              \
    "mlx_copy " CW ", " W ", " V "\n"                                      \
    ".LfZ%=:\n"                                                           

#define MLX_FRAME_SCALARS \
    "memory", "scc", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44", "s45", "s46", "s47", "s48", \
        "s49", "s50", "s51", "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59", "s60", "s61", "s62", \
        "s63", "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76", \
        "s77", "s78", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89", "s90", \
        "s91", "s92", "s93", "s94", "s95", "s96", "s97"

// n >= 1 phases from p on; slot: the thread's LDS byte offset in the layout
// the values are in, before and after; lds: byte address of the tile's LDS.
// Threads beyond the tile's 2^(nbits-4) run along on LDS slots of their own,
// past the tile's.
__device__ __forceinline__ void frame_phases(mlx_v2d (&v)[16], const FOp *p, int n, uint32_t tid, uint64_t base,
                                             uint32_t &slot, uint32_t lds)
{
    asm volatile(MLX_FRAME_MACROS MLX_FRAME_LOOP("2", "64", "128", "62", "61")
        : "={v[64:67]}"(v[0]), "={v[68:71]}"(v[1]), "={v[72:75]}"(v[2]), "={v[76:79]}"(v[3]),
          "={v[80:83]}"(v[4]), "={v[84:87]}"(v[5]), "={v[88:91]}"(v[6]), "={v[92:95]}"(v[7]),
          "={v[96:99]}"(v[8]), "={v[100:103]}"(v[9]), "={v[104:107]}"(v[10]), "={v[108:111]}"(v[11]),
          "={v[112:115]}"(v[12]), "={v[116:119]}"(v[13]), "={v[120:123]}"(v[14]), "={v[124:127]}"(v[15]),
          "={v61}"(slot)
        : "{v[64:67]}"(v[0]), "{v[68:71]}"(v[1]), "{v[72:75]}"(v[2]), "{v[76:79]}"(v[3]),
          "{v[80:83]}"(v[4]), "{v[84:87]}"(v[5]), "{v[88:91]}"(v[6]), "{v[92:95]}"(v[7]),
          "{v[96:99]}"(v[8]), "{v[100:103]}"(v[9]), "{v[104:107]}"(v[10]), "{v[108:111]}"(v[11]),
          "{v[112:115]}"(v[12]), "{v[116:119]}"(v[13]), "{v[120:123]}"(v[14]), "{v[124:127]}"(v[15]),
          "{v61}"(slot), [p] "s"(p), [n] "s"(n), [tid] "v"(tid), [base] "s"(base), [lds] "v"(lds)
        : MLX_FRAME_SCALARS, "v62", "v63",
          "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143",
          "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159",
          "v160", "v161", "v162", "v163", "v164", "v165", "v166", "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175",
          "v176", "v177", "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188", "v189", "v190", "v191");
}
__device__ __forceinline__ void frame_phases(mlx_v2f (&v)[16], const FOp *p, int n, uint32_t tid, uint64_t base,
                                             uint32_t &slot, uint32_t lds)
{
    asm volatile(MLX_FRAME_MACROS MLX_FRAME_LOOP("1", "32", "64", "31", "30")
        : "={v[32:33]}"(v[0]), "={v[34:35]}"(v[1]), "={v[36:37]}"(v[2]), "={v[38:39]}"(v[3]),
          "={v[40:41]}"(v[4]), "={v[42:43]}"(v[5]), "={v[44:45]}"(v[6]), "={v[46:47]}"(v[7]),
          "={v[48:49]}"(v[8]), "={v[50:51]}"(v[9]), "={v[52:53]}"(v[10]), "={v[54:55]}"(v[11]),
          "={v[56:57]}"(v[12]), "={v[58:59]}"(v[13]), "={v[60:61]}"(v[14]), "={v[62:63]}"(v[15]),
          "={v30}"(slot)
        : "{v[32:33]}"(v[0]), "{v[34:35]}"(v[1]), "{v[36:37]}"(v[2]), "{v[38:39]}"(v[3]),
          "{v[40:41]}"(v[4]), "{v[42:43]}"(v[5]), "{v[44:45]}"(v[6]), "{v[46:47]}"(v[7]),
          "{v[48:49]}"(v[8]), "{v[50:51]}"(v[9]), "{v[52:53]}"(v[10]), "{v[54:55]}"(v[11]),
          "{v[56:57]}"(v[12]), "{v[58:59]}"(v[13]), "{v[60:61]}"(v[14]), "{v[62:63]}"(v[15]),
          "{v30}"(slot), [p] "s"(p), [n] "s"(n), [tid] "v"(tid), [base] "s"(base), [lds] "v"(lds)
        : MLX_FRAME_SCALARS, "v31",
          "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79",
          "v80", "v81", "v82", "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95");
}

// Program data through the constant address space: the program does not
// change while a kernel runs, and the compiler, which cannot see that past
// the assembly below, would otherwise fetch wave-uniform entries with vector
// loads in the middle of a tile.
template <typename T> using FConst = const __attribute__((address_space(4))) T *;
template <typename T> __device__ __forceinline__ FConst<T> frame_const(const FOp *p)
{
    return (FConst<T>)(uintptr_t)p;
}

// The lowest bits of x spread over the set bits of mask, lowest first.
__device__ __forceinline__ uint64_t frame_deposit(uint64_t x, uint64_t mask)
{
    uint64_t o = 0;
    for (; mask && x; mask &= mask - 1, x >>= 1)
        if (x & 1ull) o |= mask & (0ull - mask);
    return o;
}

// a + b where both are numbers spread over the clear bits of mask
__device__ __forceinline__ uint64_t frame_step(uint64_t a, uint64_t b, uint64_t mask)
{
    return ((a | mask) + b) & ~mask;
}

// What a thread keeps over the tiles of a pass: the output layout's LDS
// address and its word of the sign table.
struct FrameThread {
    uint32_t out_slot;
    uint32_t sign;
};

__device__ __forceinline__ FrameThread frame_thread(FConst<FPass> P, const FOp *prog, int tid, int tbits, bool active)
{
    FrameThread f{0, 0};
    if (P->flags & FP_OUT) {
        const FConst<FOut> o = frame_const<FOut>(prog + P->out);
        for (int b = 0; b < tbits; b++) f.out_slot ^= ((tid >> b) & 1) ? o->col[b] : 0u;
    }
    if (P->table >= 0 && active) f.sign = ((const uint16_t *)(prog + P->table))[tid];
    return f;
}

// byte address of a __shared__ variable
#define MLX_FRAME_LDS(var) ((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&(var))

// x, known to be the same on every lane, in scalar registers
__device__ __forceinline__ uint64_t frame_uniform(uint64_t x)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// The phases of a pass on one tile, then the signs, the scale and the output
// layout: v enters and leaves in the IO layout (register bits = top four tile
// bits).  Every thread of the workgroup calls it (barriers); lds: byte address
// (MLX_FRAME_LDS) of 16 amplitudes per thread of the workgroup, whatever the
// tile's size.
template <typename R>
__device__ __forceinline__ void frame_tile(uint32_t lds, typename FVec<R>::t (&v)[16], FConst<FPass> P,
                                           const FOp *prog, const FrameThread &ft, uint64_t base, int tid,
                                           int nbits)
{
    using V = typename FVec<R>::t;
    // the thread's slot in the current layout; thread bits past the tile's
    // go above its index
    const int x0 = tid + 15 * (tid & -(1 << (nbits - kFrameRegBits)));
    uint32_t slot = (uint32_t)lds_slot<(int)sizeof(V)>(x0) * (uint32_t)sizeof(V);
    if (P->nphases > 0)
        frame_phases(v, (const FOp *)frame_uniform((uint64_t)(uintptr_t)(prog + P->first)),
                     __builtin_amdgcn_readfirstlane(P->nphases), (uint32_t)tid, frame_uniform(base), slot,
                     lds);
    if (P->flags & (FP_SIGN | FP_SCALE | FP_CSCALE)) {
        uint32_t s = ft.sign;
        for (int c = 0; c < P->ncross; c++) {
            const FConst<FCross> x = frame_const<FCross>(prog + P->cross) + c;
            const uint32_t a = (uint32_t)__popcll(x->ga & base) & 1u, b = (uint32_t)__popcll(x->gb & base) & 1u;
            const uint32_t fa = x->wa ^ (0u - ((uint32_t)__popc(x->ta & tid) & 1u));
            const uint32_t fb = x->wb ^ (0u - ((uint32_t)__popc(x->tb & tid) & 1u));
            s ^= (a ? fb : 0u) ^ (b ? fa : 0u) ^ (a & b ? 0xFFFFu : 0u);
        }
        const R sr = (R)P->scale_r, si = (R)P->scale_i;
        if (P->flags & FP_CSCALE) {
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const bool neg = (s >> j) & 1u;
                const cplx_t<R> y = cmul(cplx_t<R>{v[j].x, v[j].y}, neg ? -sr : sr, neg ? -si : si);
                v[j].x = y.x;
                v[j].y = y.y;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const R r = (s >> j) & 1u ? -sr : sr;
                v[j].x *= r;
                v[j].y *= r;
            }
        }
    }
    if (P->flags & FP_OUT) {
        const FConst<FOut> o = frame_const<FOut>(prog + P->out);
        using SharedV = __attribute__((address_space(3))) V;
#pragma unroll
        for (int j = 0; j < 16; j++) *(SharedV *)(uintptr_t)(lds + (slot ^ o->from[j])) = v[j];
        uint32_t os = ft.out_slot;
        for (int c = 0; c < P->nshift; c++) {
            const FConst<FShift> x = frame_const<FShift>(prog + P->shift) + c;
            os ^= (__popcll(x->gmask & base) & 1) ? x->off : 0u;
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = *(const SharedV *)(uintptr_t)(lds + (os ^ o->off[j]));
        // Between two changes a thread writes only slots that it alone has
        // read; the output's permutation breaks that, so nothing is written
        // (by the next tile) before every thread has read.
        lds_barrier();
    }
}

}  // namespace mlx
