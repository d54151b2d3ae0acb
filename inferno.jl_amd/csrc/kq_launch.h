// kq_launch.h -- internal launchers shared by the kernel files and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace ihip {

// kq_gemv.hip
// resid != nullptr: y = epi_apply(resid, W x, epi) per row (kq_common.h: the
// residual add, or the SwiGLU of an unfused gate/up pair); resid may be y.
hipError_t launch_gemv(int type, const void *w, const float *x, float *y, int inner, int outer,
                       hipStream_t s, const float *resid = nullptr, int epi = 0);
// y = W (rmsnorm(x) .* nw) in one launch (the folded norm of the wide kernels or
// of k_gemv_mdig) for Q4_K / Q5_K rows of at most 16 blocks; hipErrorNotSupported
// otherwise.
bool gemv_norm_fusable(int type, int inner, int outer);
hipError_t launch_gemv_norm(int type, const void *w, const float *x, const float *nw, float eps,
                            float *y, int inner, int outer, hipStream_t s);
bool gate_up_fusable(int gate_type, int up_type);
// norm_w != nullptr: the input is rmsnorm(x) .* norm_w (eps inside the root).
hipError_t launch_gate_up_swiglu(int type, const void *wg, const void *wu, const float *x,
                                 float *h, int hidden, int inter, hipStream_t s,
                                 const float *norm_w = nullptr, float eps = 0.0f);
// Whether the argmax can be fused into the lm_head GEMV: Q6_K / Q8_0 rows of
// at most 16 segments of 2048 columns (any vocabulary: the grid is capped at
// kArgMaxParts workgroups, one partial each).
bool lm_head_fusable(int type, int hidden);
// Argmax partials (16 bytes each) one lm_head call writes: fused into the
// streamed GEMV, or the standalone argmax after the GEMV.
int lm_head_argmax_parts(int type, int hidden, int vocab, bool fused);
hipError_t launch_lm_head_argmax(int type, const void *w, const float *x, float *logits,
                                 int32_t *token, uint32_t *flags, int hidden, int vocab,
                                 void *ws, hipStream_t s);
hipError_t launch_argmax(const float *v, int64_t n, int32_t *token, uint32_t *flags, void *ws,
                         hipStream_t s);

// kq_dequant.hip
hipError_t launch_gemv_generic(int type, const void *w, const float *x, float *y, int inner,
                               int outer, hipStream_t s, const float *resid = nullptr, int epi = 0);
// rmsnorm_cpu! (src/ModelCPU.jl:111-123): out = x * (1/sqrt(mean(x^2) + eps)) .* w
hipError_t launch_rmsnorm(const float *x, const float *w, float eps, float *out, int n,
                          hipStream_t s);
hipError_t launch_dequant(int type, const void *src, float *dst, int64_t n, bool aligned,
                          hipStream_t s);
hipError_t launch_mlp_gate_mul(float *gate, const float *up, int64_t n, hipStream_t s);
hipError_t launch_silu_gate_mul(float *out, const float *x, const float *gate, int64_t n,
                                hipStream_t s);

// CUs of the current device (queried once per device)
int device_cus();

// kq_prefill.hip
// The prefill GEMM addresses its operands as 32-bit byte offsets from the
// start of Xh (T x inner fp16) and W (outer Q4_K rows), and counts its
// output tiles in ints.
inline bool prefill_fits(int T, int inner, int outer)
{
    return 2 * (int64_t)T * inner <= (int64_t)UINT32_MAX &&
           (int64_t)outer * (inner / 256) * 144 <= (int64_t)UINT32_MAX &&
           (int64_t)T * outer <= (int64_t)INT32_MAX; // tile counts stay ints
}
// Rows of at most this many columns run on fp32 operands (k_prefill_q4k_split).
constexpr int kPrefillF32MaxK = 512;
// Longer rows of at most this many columns take fp16 weights rounded once
// from their exact values (k_prefill_q4k<true>).
constexpr int kPrefillExactWMaxK = 2048;
// The caller's scratch xh: the fp16 activations (T x inner), one int per
// token (its power-of-two scale) from the next 16-byte boundary, then, from
// the next 16-byte boundary, the partial sums of a split over K.  A split
// keeps nsplit x (64-token x 128-row tiles) <= kPrefillMaxTiles, so its
// nsplit - 1 partial planes of T x outer floats hold at most
// T x 128 x kPrefillMaxTiles / ceil(T / 64) floats whatever outer is.
constexpr int kPrefillMaxTiles = 256;
constexpr int kPrefillBM = 64, kPrefillBN = 128; // workgroup tile: tokens x weight rows
inline size_t prefill_scale_offset(int T, int inner)
{
    return ((size_t)2 * (size_t)T * (size_t)inner + 15) & ~(size_t)15;
}
inline size_t prefill_part_offset(int T, int inner)
{
    return (prefill_scale_offset(T, inner) + (size_t)4 * (size_t)T + 15) & ~(size_t)15;
}
inline size_t prefill_part_floats(int T)
{
    const size_t mtiles = ((size_t)T + kPrefillBM - 1) / kPrefillBM;
    return (size_t)T * kPrefillBN * (size_t)kPrefillMaxTiles / mtiles;
}
// XCD-aware order: workgroup bid's place `lin` in tile order, so that the
// consecutive workgroups of one XCD (bid mod 8) take consecutive places and
// share the operand bytes of those tiles in their L2 (tile order below).
// The grid is prefill_grid workgroups; lin >= tiles x nsplit exits.
__host__ __device__ inline int prefill_grid(int tiles, int nsplit)
{
    return (tiles * nsplit + 7) / 8 * 8;
}
__host__ __device__ inline int prefill_lin(int bid, int tiles, int nsplit)
{
    const int per_xcd = (tiles * nsplit + 7) / 8;
    return (bid % 8) * per_xcd + bid / 8;
}
// Workgroup `lin` (in tile order) of a launch of mtiles x ntiles tiles and
// nsplit splits over K: its split, its tile and the split's block columns
// kb0 .. kb0 + nk - 1 of the nblk.  Tile order within a split: groups of
// kPrefillGroupM M tiles (token bands), the group's M tiles fastest, then N.
// An XCD's 32 consecutive tiles at 512 tokens are then 4 token bands x 8
// weight bands, 2 MB of fp16 activations and 2.4 MB of weight blocks per
// 4 MB L2, where all 8 token bands of 4 weight bands (M fastest over all of
// them) need 4 MB + 1.2 MB.  Measured on MI355X (us per call, stream
// launches, two runs each, interleaved): 512 x 4096 x 4096 30.5 against
// 31.4-31.5, 512 x 14336 x 4096 102.8-103.0 against 104.7-105.0, 512 x 4096
// x 14336 84.1-84.6 against 84.4-84.9; groups of 2 M tiles were no better at
// 512 tokens and 0.7 us slower at 256 (2 x 16 bands per XCD).
constexpr int kPrefillGroupM = 4;
struct PrefillSplit {
    int sp, mt, nt, kb0, nk;
};
__host__ __device__ inline PrefillSplit prefill_split_of(int lin, int mtiles, int ntiles, int nblk,
                                                        int nsplit)
{
    PrefillSplit s;
    const int tiles = mtiles * ntiles;
    s.sp = lin / tiles;
    const int tl = lin - s.sp * tiles;
    const int g = tl / (kPrefillGroupM * ntiles);
    const int gm = mtiles - kPrefillGroupM * g < kPrefillGroupM ? mtiles - kPrefillGroupM * g : kPrefillGroupM;
    const int idx = tl - g * kPrefillGroupM * ntiles;
    s.mt = kPrefillGroupM * g + idx % gm;
    s.nt = idx / gm;
    s.kb0 = s.sp * nblk / nsplit;
    s.nk = (s.sp + 1) * nblk / nsplit - s.kb0;
    return s;
}
inline size_t prefill_scratch_bytes(int T, int inner)
{
    return prefill_part_offset(T, inner) + 4 * prefill_part_floats(T);
}
// Splits over K of one prefill launch on a device of ncu CUs (1: none).  A
// weight of few rows leaves most CUs without a tile (512 x 512 x 4096 is 32
// tiles for 256 CUs), so each tile's block columns are shared out over
// nsplit workgroups, as many as keep nsplit x tiles within the CUs (and
// within the partial planes the scratch holds) and at least two columns per
// split, and a second launch adds the partial sums.  Rows of fewer than 8
// block columns are not split: a workgroup's fixed cost (the launch, the
// first copies, the partial-sum exchange and the 32 KB of stores) is then
// most of its time, and the summing launch adds to it (measured on MI355X,
// us per call: 512 x 512 x 4096 18.9-21.4 against 27.6 unsplit, 64 x 4096 x
// 4096 18.9-19.3 against 23.9, 512 x 2048 x 4096 25.5-25.8 against 28.1;
// 512 x 1024 x 1024 split four ways 18.2-19.0 against 13.0).
inline int prefill_splits(int T, int inner, int outer, int ncu)
{
    const int mtiles = (T + kPrefillBM - 1) / kPrefillBM, ntiles = (outer + kPrefillBN - 1) / kPrefillBN;
    const int tiles = mtiles * ntiles, nblk = inner / 256;
    const int cap = ncu < kPrefillMaxTiles ? ncu : kPrefillMaxTiles;
    if (tiles * 2 > cap || nblk < 8)
        return 1;
    const int s = cap / tiles < nblk / 2 ? cap / tiles : nblk / 2;
    return s > 1 ? s : 1;
}
// Which tile a prefill launch takes: 0 for 64 tokens x 128 rows (split over K
// where that fills idle CUs), 1 or 2 for the wide kernel's 128 tokens x 128 or
// 256 rows.  The line between them is the estimated time of each, in us, from
// its block columns and its tiles per CU u = tiles / CUs (c = u rounded up:
// the busiest CU's tiles).  The coefficients are a least-squares fit of the
// three kernels timed on MI355X at 640 shapes (1 to 2048 tokens, 256 to 14336
// rows, 1024 to 12288 columns; relative rms 7-10 %); over the 326 of them
// without a split the choice is 0.01 % from the fastest on average and never
// over 1 % slower than 64 x 128.  Examples, us (64 x 128 / 128 x 128 /
// 128 x 256): 512 x 4096 x 4096 26.6 / 35.2 / 51.5, 192 x 12288 x 4096 44.5 /
// 34.7 / 51.0, 1024 x 4096 x 4096 48.2 / 39.6 / 52.6, 1024 x 14336 x 4096 154.9
// / 119.6 / 109.9.
constexpr int kPrefillWideBM = 128;
inline double prefill_cost(int tiles, int nblk, int ncu, double fixed, double col, double per_u, double per_c)
{
    const double u = (double)tiles / ncu, c = (double)((tiles + ncu - 1) / ncu);
    return fixed + nblk * (col + per_u * u + per_c * c);
}
struct PrefillCosts {
    double narrow, wide1, wide2; // 64 x 128 (with its splits), 128 x 128, 128 x 256
};
inline PrefillCosts prefill_costs(int T, int inner, int outer, int ncu)
{
    const int nblk = inner / 256, cus = ncu > 0 ? ncu : 1;
    auto tiles = [&](int bm, int bn) { return ((T + bm - 1) / bm) * ((outer + bn - 1) / bn); };
    const int nsplit = prefill_splits(T, inner, outer, ncu);
    PrefillCosts c;
    c.narrow = prefill_cost(tiles(kPrefillBM, kPrefillBN), nblk, cus, 6.6, -0.37, 0.53, 0.99);
    if (nsplit > 1) // the split's share of the columns, then its planes' traffic and the summing launch
        c.narrow = 8.17 + (double)nblk / nsplit * (0.70 + 0.63 * tiles(kPrefillBM, kPrefillBN) * nsplit / cus) +
                   1.07e-6 * T * outer * nsplit;
    c.wide1 = prefill_cost(tiles(kPrefillWideBM, 128), nblk, cus, 4.5, 0.20, 0.63, 1.23);
    c.wide2 = prefill_cost(tiles(kPrefillWideBM, 256), nblk, cus, 6.5, -0.10, 1.13, 2.44);
    return c;
}
inline int prefill_wide_rows(int T, int inner, int outer, int ncu)
{
    if (prefill_splits(T, inner, outer, ncu) > 1)
        return 0; // few tiles of either size: K is shared out instead
    const PrefillCosts c = prefill_costs(T, inner, outer, ncu);
    return c.narrow <= c.wide1 && c.narrow <= c.wide2 ? 0 : c.wide1 <= c.wide2 ? 1 : 2;
}
// Whether it takes the 32-token x 64-row tiles whose waves share K instead
// (k_prefill_q4k_thin): by the same estimate, fitted to 105 shapes of 8 to 1024
// tokens timed in graph replays (relative rms 9 %; the split 64 x 128 tile 5 %).
// Over them the choice is never over 2 % slower than without this kernel,
// 1.13 times as fast on average and 0.2 % from the faster of the two.  That is
// on weights that the memory-side cache holds.  From HBM its gain is smaller,
// and at 1 to 32 tokens some shapes lose (us, the product alone, 64 x 128 / thin;
// held in the cache): 1 x 4096 x 4096 11.1 / 12.1 (11.9 / 11.0), 32 x 3584 x 3584 12.5
// / 15.5 (12.5 / 11.7), 32 x 4096 x 6144 13.9 / 16.1 (14.0 / 12.5), 77 x 2560 x 9728
// 16.3 / 17.4 (16.5 / 15.5); 32 x 2048 x 5632 11.7 / 9.8 (11.7 / 8.4), 128 x 4096 x 4096
// 18.9 / 14.3 (17.8 / 12.4).
constexpr int kPrefillThinBM = 32, kPrefillThinBN = 64;
inline bool prefill_thin(int T, int inner, int outer, int ncu)
{
    const int nblk = inner / 256, cus = ncu > 0 ? ncu : 1;
    const int64_t tiles = ((int64_t)T + kPrefillThinBM - 1) / kPrefillThinBM * (((int64_t)outer + kPrefillThinBN - 1) / kPrefillThinBN);
    if (tiles > 16 * (int64_t)cus)
        return false; // a product of many tiles
    const double thin = prefill_cost((int)tiles, nblk, cus, 3.55, -0.154 + 0.1 * std::min(T, 32) / 32, 0.074, 0.577);
    const int ru = prefill_wide_rows(T, inner, outer, ncu);
    const PrefillCosts c = prefill_costs(T, inner, outer, ncu);
    return thin < (ru == 0 ? c.narrow : ru == 1 ? c.wide1 : c.wide2);
}
hipError_t launch_prefill_q4k(const void *w, const float *X, void *xh, float *Y, int T,
                              int inner, int outer, hipStream_t s);
// Its two halves for rows of more than kPrefillF32MaxK columns: X rounded into
// xh (fp16 rows and one scale exponent per token), then the product from xh
// (which also takes the partial sums of a split over K, leaving the rounded
// rows as they were), so several weights can share one rounding.
hipError_t launch_prefill_convert(const float *X, void *xh, int T, int inner, hipStream_t s);
hipError_t launch_prefill_gemm(const void *w, void *xh, float *Y, int T, int inner, int outer,
                               hipStream_t s);
// Tokens per workgroup tile (64 weight rows) of the product on fp32 operands:
// 32 or 64, whichever needs less time in rounds of one workgroup per CU, a
// 32-token tile taking 0.58-0.62 of a 64-token one's time.  Measured on MI355X
// (us, 32 / 64 tokens): 256 x 2048 x 2048 13.6 / 20.1, 300 x 4096 x 4096 65.2 /
// 71.5, 200 x 4096 x 4096 43.5 / 40.3, 509 x 2048 x 2048 25.9 / 23.6.
constexpr int kPrefillSplitMaxK = 1 << 24; // 64 rows of X or W of this length are within 32-bit byte offsets
inline int prefill_split_tokens(int T, int outer, int ncu)
{
    const int64_t cus = ncu > 0 ? ncu : 1, nt = ((int64_t)outer + 63) / 64;
    const int64_t r32 = (((int64_t)T + 31) / 32 * nt + cus - 1) / cus, r64 = (((int64_t)T + 63) / 64 * nt + cus - 1) / cus;
    return 10 * r32 <= 17 * r64 ? 32 : 64;
}
// ---- copies and LDS reads of k_prefill_q4k_wide, _thin and _split, which
// tests/native/prefill_copy_check.hip walks ----
// A block's 32 chunks of 8 values in a row of Xh: chunk 16 h + 4 g + c at place
// 8 g + 4 h + c.
__host__ __device__ constexpr int pf_chunk_place(int chunk)
{
    return 8 * ((chunk >> 2) & 3) + 4 * (chunk >> 4) + (chunk & 3);
}
// An X stage is 128 bytes (eight 16-byte chunks) of each token, eight tokens a
// copy: lane l of copy i brings token 8 i + l / 8, and its place l % 8 holds chunk
// (l % 8) ^ (token / 2 % 8), so that the 16 lanes of a 128-bit read, one chunk of
// consecutive tokens, hit distinct banks.
__host__ __device__ inline int pf_copy_token(int i, int lane) { return 8 * i + (lane >> 3); }
__host__ __device__ inline int pf_copy_chunk(int token, int lane) { return (lane & 7) ^ ((token >> 1) & 7); }
// Byte of chunk c of token m in a stage of LDS.
__host__ __device__ inline uint32_t pf_stage_at(int m, int c) { return 128u * (uint32_t)m + 16u * (uint32_t)(c ^ ((m >> 1) & 7)); }
// Weight pieces of 16 bytes: whole blocks of `rows` rows (the last piece again
// past them), or the header and 32 quant bytes (pair j) of each.
struct PfPiece {
    int row;
    uint32_t off; // in the row's block
};
__host__ __device__ inline PfPiece pf_block_piece(int i, int lane, int rows)
{
    const int q = min(64 * i + lane, rows * 9 - 1);
    return {q / 9, 16u * (uint32_t)(q - 9 * (q / 9))};
}
__host__ __device__ inline PfPiece pf_pair_piece(int i, int lane, int j)
{
    const int q = 64 * i + lane, row = q / 3, piece = q - 3 * row;
    return {row, piece ? 32u * (uint32_t)j + 16u * (uint32_t)piece : 0u};
}

// The same product on fp32 operands (k_prefill_q4k_split), any inner; needs
// T * outer <= INT32_MAX.
hipError_t launch_prefill_q4k_f32(const void *w, const float *X, float *Y, int T, int inner,
                                  int outer, hipStream_t s);

// kq_q8k.hip
// k_gemv_q8k6: rows of at most kQ86MaxBlocks Q6_K blocks, eight (1680 bytes) an
// item, copied from the 16-byte unit of the item's first byte (phase bytes below
// it) in two copies of 64 lanes; pieces past the item's last byte are the last one
// again.
constexpr int kQ86MaxBlocks = 24, kQ86Waves = 16, kQ86Items = (kQ86MaxBlocks + 7) / 8, kQ86Slot = 2048;
__host__ __device__ inline uint32_t q86_copy_off(int i, int lane, uint32_t phase, int blocks)
{
    return min(1024u * (uint32_t)i + 16u * (uint32_t)lane, (phase + (uint32_t)blocks * 210u - 1u) & ~15u);
}
// Waves to a row: as many of 1, 2 (from 5 blocks on) and 4 (from 17) as one
// round of the chip's waves has for every row.  (Two waves of a row of at most
// eight blocks are one at work, in twice the workgroups.)  Measured on MI355X
// (us, quantizing included, graph replays over weights in HBM, fewer / more
// waves): 256 x 256 3.18 / 3.72, 256 x 512 3.21 / 3.34, 512 x 1024 3.50 / 3.56; 512 x 1280
// 3.56 / 3.68, 512 x 2048 3.77 / 3.71; 512 x 5120 6.29 / 5.20, 1024 x 6144 6.75 / 5.76.
inline int q86_team(int nb, int outer, int ncu)
{
    int tw = 1;
    while (tw < 4 && (int64_t)outer * 2 * tw <= (int64_t)ncu * kQ86Waves && nb > (tw == 1 ? 4 : 16))
        tw *= 2;
    return tw;
}
hipError_t launch_quantize_q8k(const float *x, void *y, int64_t k, hipStream_t s);
hipError_t launch_gemv_q8k(int type, const void *w, const void *q8, float *out, int inner,
                           int outer, hipStream_t s);
// x as fp32, quantized to Q8_K inside the launch where the kernel takes the
// shape (Q4_K / Q5_K, at most 32768 columns; Q6_K of at most 6144 columns and
// one round of rows; 16-byte aligned w and x); q8out
// (optional) receives the Q8_K blocks; otherwise x is quantized into q8out or,
// without it, into q8tmp (inner / 256 blocks) first.  x, out and q8out must
// not overlap: the one launch reads x while it writes the others.
hipError_t launch_gemv_q8k_x(int type, const void *w, const float *x, void *q8out, void *q8tmp,
                             float *out, int inner, int outer, hipStream_t s);

} // namespace ihip
