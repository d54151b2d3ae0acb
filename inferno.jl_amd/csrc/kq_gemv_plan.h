// kq_gemv_plan.h -- which GEMV kernel takes a weight, by its format, row length
// and (where no other launch has to give the same bits) row count.  Shared by
// the launchers (kq_gemv.hip) and the CPU tests (tests/native).
#pragma once

#include <algorithm>

#include "kq_common.h"

namespace ihip {

// Rows of at most 16 blocks with at least four 8-wave row groups per wave
// over one workgroup per CU take the wide kernels' persistent form.
inline bool kwide_takes_kpers(int nblk, int outer) { return nblk <= 16 && outer >= 4 * 8 * 256; }

// No more one-row workgroups of 8 waves than CUs: one row per wave.
inline bool kwide_one_row(int outer, int ncu) { return (outer + 7) / 8 <= ncu; }

// Which rows k_gemv_mdig takes, by format, length and (gate/up) kind only: a
// row's sum is the same whatever launch it is in, and the two kernels' differ.
// The wide kernels spread a row's blocks over 16 lane positions, this one over
// 4 a step, and it starts later (x goes through LDS twice).  So the wide
// kernels keep the Q4_K / Q5_K rows that fill their lanes, and the short Q4_K
// ones.  Measured on MI355X (us, graph replays over weights in HBM, wide / this):
// Q4_K 2560 x 9728 8.6 / 6.3, 5120 x 5120 7.8 / 5.6, 4096 x 14336 10.6 / 9.9,
// 4096 x 4096 4.1 / 4.6, 12288 x 4096 7.4 / 7.8, 3584 x 2560 3.45 / 3.73; Q5_K
// 4096 x 2048 4.1 / 3.5, 9728 x 2560 7.4 / 6.5, 4096 x 4096 4.8 / 5.1; gate/up
// Q4_K 6144 x 2048 7.2 / 5.7, 13824 x 5120 20.6 / 17.2, 10240 x 3584 11.0 / 10.5,
// 12288 x 4096 12.8 / 13.0; Q5_K 9728 x 2560 12.3 / 9.7, 12288 x 4096 15.8 / 15.5.
// Q6_K (streamed / this) 4096 x 12288 12.4 / 11.7, 2560 x 9728 12.1 / 7.9, 5120 x
// 13824 26.9 / 15.9, 1024 x 4096 4.9 / 3.6, 12288 x 4096 10.8 / 10.8; Q8_0 5003 x
// 2720 8.4 / 5.8, 2560 x 9728 11.2 / 8.3; IQ4_NL 5120 x 5120 10.7 / 6.8, 5003 x 2720
// 8.8 / 5.1, 20000 x 6144 24.3 / 17.7.  What going by length costs: few rows of Q5_K
// (1024 x 2560 2.90 / 3.17, 1024 x 3072 2.92 / 3.17, 1024 x 1024 2.87 / 2.81).
constexpr int kMdMaxSteps = 16, kMdMaxBlocks = 4 * kMdMaxSteps;
constexpr bool mdig_takes(int type, int nblk, bool gateup)
{
    if (nblk > kMdMaxBlocks)
        return false;
    if (type == kQ6_K || nblk > 16)
        return true;
    if (gateup)
        return type == kQ5_K || nblk <= 14;
    return type == kQ5_K && nblk <= 12;
}

// Q8_0 and IQ4_NL rows of whole 256-column units on the wide lane layout, by
// length only (as mdig_takes).  Measured on MI355X (us, graph replays over weights
// in HBM, wide / k_gemv_mdig): Q8_0 1024 x 4096 3.41 / 3.63, 4096 x 4096 5.97 / 6.10,
// 12288 x 4096 11.45 / 12.01, 2048 x 2560 3.41 / 3.79, 8192 x 2560 6.93 / 6.96, 2048 x
// 2048 3.37 / 3.65, 12288 x 2048 7.66 / 7.59, 1024 x 1024 2.90 / 2.94, and many rows of
// 1024 columns the other way (12288 6.98 / 5.08); IQ4_NL 4096 x 4096 5.0 / 5.4, 1024 x
// 3584 3.18 / 3.52, 4096 x 3328 4.81 / 5.21, 12288 x 3328 9.80 / 9.37, and where
// k_gemv_mdig has it 1024 x 2560 3.21 / 3.35, 2048 x 3072 3.64 / 3.76, 4096 x 3072 4.72 /
// 4.44, 12288 x 2560 9.50 / 7.54.  IQ4_NL rows too long for the others too (4096 x 20480).
inline bool b32_takes_wide(int type, int inner)
{
    if (inner % 256)
        return false;
    if (type == kQ8_0)
        return inner <= 4096;
    return (inner > 3072 && inner <= 4096) || inner > 1024 * kMdMaxSteps;
}

// k_gemv_mdig's launch: groups of four rows per workgroup (`steps` of 1024
// columns a group, gate and up together), one workgroup per CU where the units
// it can hold allow.
constexpr int kMdUnits = 512; // units (four rows x one step) per workgroup
inline int mdig_groups(int outer, int steps, int ncu)
{
    const int ngroups = (outer + 3) / 4;
    return std::min((ngroups + ncu - 1) / ncu, kMdUnits / steps);
}
// Waves, ring slots per wave and the most steps the instantiation takes, by the
// row's steps and the format's slot (3 to 5 KB a wave and slot, beside 4 KB of
// digits a step).  Q6_K rows of four steps, four groups or more per workgroup,
// run on 12 waves: measured on MI355X (us, graph replays over weights in HBM, 8
// waves x 3 slots / 12 x 2) 12288 x 4096 11.25 / 10.8 (the streamed kernel 10.8),
// 4096 x 4096 6.2 / 5.5, 8192 x 3328 7.85 / 7.36; 10 and 11 waves x 3 slots 11.6
// and 11.8 at 12288 x 4096, 16 x 2 11.5.  Fewer steps or groups leave the added
// waves idle: 4096 x 2560 4.64 / 4.84, 2048 x 4096 4.33 / 4.63.
struct MdPlan {
    int nw, d, maxs;
};
constexpr int kMdManyGroups = 4;
constexpr MdPlan mdig_plan(int type, int nstep, int groups)
{
    if (type == kQ6_K && nstep == 4 && groups >= kMdManyGroups)
        return {12, 2, 4};
    if (nstep <= 4)
        return {8, 3, 4};
    if (type == kQ6_K && nstep <= 12)
        return {12, 2, 12};
    return type == kQ6_K || type == kQ8_0 ? MdPlan{8, 2, 16} : MdPlan{12, 2, 16};
}

// ---- k_gemv_mdig's index arithmetic, which tests/native/mdig_check.hip walks ----
// Bytes of a block and blocks of a step; 16-byte pieces of a row's step (PHASED:
// from the 16-byte unit its first byte lies in, at an even phase of 0 .. 14);
// pieces between two rows in a ring slot (one more: 13 of 16 lanes' 128-bit reads then hit
// distinct banks, 8 without); 1 KB copies of a slot.
template <int FMT>
struct MdFmt;
template <>
struct MdFmt<kQ4_K> {
    static constexpr int BYTES = 144, BLOCKS = 4, PIECES = 36, PITCH = 37, COPIES = 3;
    static constexpr bool PHASED = false;
};
template <>
struct MdFmt<kQ5_K> {
    static constexpr int BYTES = 176, BLOCKS = 4, PIECES = 44, PITCH = 45, COPIES = 3;
    static constexpr bool PHASED = false;
};
template <>
struct MdFmt<kQ6_K> {
    static constexpr int BYTES = 210, BLOCKS = 4, PIECES = 54, PITCH = 55, COPIES = 4;
    static constexpr bool PHASED = true;
};
template <>
struct MdFmt<kQ8_0> {
    static constexpr int BYTES = 34, BLOCKS = 32, PIECES = 69, PITCH = 70, COPIES = 5;
    static constexpr bool PHASED = true;
};
template <>
struct MdFmt<kIQ4_NL> {
    static constexpr int BYTES = 18, BLOCKS = 32, PIECES = 37, PITCH = 38, COPIES = 3;
    static constexpr bool PHASED = true;
};

// A unit is one step of a group of four rows (of its gate or of its up rows);
// wave w of nwv takes units w, w + nwv, ...
__host__ __device__ inline int md_wave_units(int units, int wave, int nwv)
{
    return wave < units ? (units - wave - 1) / nwv + 1 : 0;
}
// Quotients by nstep of numbers up to 16: inv = ceil(65536 / nstep).
__host__ __device__ inline uint32_t md_inv(int nstep) { return (65536u + (uint32_t)nstep - 1) / (uint32_t)nstep; }
__host__ __device__ inline int md_div(int a, uint32_t inv) { return (int)(((uint32_t)a * inv) >> 16); }

// x (and, NORM, the norm's weights) in 1 KB copies, a wave those that its own
// threads convert: how many, how many of each the ring's last slots hold at a
// time, the slots that takes, and a thread's byte offset in its copy k (threads
// past the row, in rows of no whole 256 columns, copy its end).
__host__ __device__ inline int md_x_copies(int inner, int wave, int nt)
{
    return (inner / 4 - 64 * wave + nt - 1) / nt;
}
__host__ __device__ constexpr int md_x_chunk(int nx, int d, int copies, bool norm)
{
    return nx < d * copies / (norm ? 2 : 1) ? nx : d * copies / (norm ? 2 : 1);
}
__host__ __device__ inline int md_raw_slots(int xc, bool norm, int copies)
{
    return ((norm ? 2 : 1) * xc + copies - 1) / copies;
}
__host__ __device__ inline uint32_t md_x_off(int inner, int tid, int nt, int k)
{
    return (uint32_t)min(16 * tid, 4 * inner - 16 - 16 * nt * k);
}

// Piece q of a slot (copy q / 64, lane q % 64): its row of the group and its
// byte offset in that row's step.
__host__ __device__ inline int md_piece_row(int q, int pitch) { return min(q / pitch, 3); }
__host__ __device__ inline uint32_t md_piece_off(int q, int row, int pitch, int pieces)
{
    return 16u * (uint32_t)min(q - row * pitch, pieces - 1);
}
// Byte offset, from the group's first row's step (PHASED: from the 16-byte unit
// `phase` bytes below it), of the piece at `piece` of the row `row` bytes
// further: the row's nbytes, the last piece of them again past their end.
template <bool PHASED>
__host__ __device__ inline uint32_t md_copy_off(uint32_t row, uint32_t piece, uint32_t nbytes, uint32_t phase)
{
    if constexpr (PHASED) { // from the 16-byte unit of the row's first byte
        const uint32_t o = row + phase;
        return (o & ~15u) + min(piece, ((o & 15u) + nbytes - 1u) & ~15u);
    } else {
        return row + min(piece, nbytes - 16u);
    }
}

// The folded norm on a single weight of at most 16 blocks a row: whether the
// wide kernels take it.  By row count too (no other call promises these bits):
// the wide kernels are ahead while one round of their workgroups holds the rows
// (one row per wave up to 8 rows per CU, two up to 16) or where they run
// persistent, and behind where a second round starts; longer rows fill their
// lanes better.  Measured on MI355X (us, graph replays over weights in HBM, wide
// / k_gemv_mdig): Q4_K 1024 x 1024 3.00 / 3.02, 1024 x 1536 3.06 / 3.28, 1024 x 2560
// 3.04 / 3.37, 2048 x 4096 4.08 / 4.47, 4096 x 2048 3.91 / 3.80, 3072 x 2304 3.78 /
// 4.12, 4096 x 4096 4.49 / 5.14, 6144 x 4096 6.45 / 5.80, 12288 x 3072 6.71 / 6.55,
// 12288 x 3328 6.81 / 7.47, 12288 x 4096 7.22 / 8.12; Q5_K 1024 x 2048 3.27 / 3.28,
// 1024 x 2304 3.23 / 3.48, 2048 x 4096 4.42 / 4.56, 4096 x 3072 5.00 / 4.64, 4096 x
// 3328 4.93 / 5.22, 6144 x 4096 7.27 / 6.38, 12288 x 3072 8.02 / 7.69, 12288 x 4096
// 8.76 / 9.33.
inline bool norm_takes_wide(int type, int nblk, int outer, int ncu)
{
    const bool one = kwide_one_row(outer, ncu), two = (outer + 15) / 16 <= ncu;
    if (type == kQ4_K)
        return one ? nblk > 4 : two ? nblk > 8 : nblk > 12 && kwide_takes_kpers(nblk, outer);
    return one ? nblk > 8 : nblk > 12 && (two || kwide_takes_kpers(nblk, outer));
}

// Gate/up (one wide workgroup has eight rows of each): whether the wide kernels
// take it although mdig_takes does, by row count as above: while one round of
// their workgroups holds the rows and, but for the longest Q4_K ones, a
// workgroup of k_gemv_mdig has more than one group of four.  Measured likewise:
// Q4_K 1536 x 2048 3.41 / 3.42, 1024 x 2816 3.69 / 3.45, 1536 x 2304 3.63 / 3.91, 2048 x
// 2816 3.82 / 4.02, 1024 x 3328 3.61 / 3.95, 1536 x 3584 3.90 / 4.62, 2304 x 2560 5.07 /
// 4.53, 4096 x 3584 5.93 / 6.05; Q5_K 1024 x 3584 4.37 / 4.09, 1536 x 3328 4.49 / 4.91,
// 2048 x 4096 5.05 / 5.27, 1536 x 3072 4.50 / 4.26, 2304 x 4096 6.84 / 6.02.
inline bool gate_up_takes_wide(int type, int nblk, int outer, int ncu)
{
    if (!mdig_takes(type, nblk, true))
        return true;
    if (nblk > 16 || !kwide_one_row(outer, ncu))
        return false;
    const bool groups = outer > 4 * ncu;
    return type == kQ4_K ? nblk > 12 || (nblk > 8 && groups) : nblk > 12 && groups;
}

} // namespace ihip
