// kq_prefill.hip -- batched prefill GEMM on gfx950 matrix cores:
//   Y[t, n] = sum_k W[n, k] * X[t, k],  W: N x K Q4_K,  X: T x K fp32.
//
// The reference has no GEMM here: src/ModelCPU.jl:1001-1017 (Inferno.jl)
// runs T independent GEMVs, so the semantics are the Q4_K GEMV applied row
// by row.  On MI355X the T tokens share every weight byte, which makes this
// a dense contraction: X is rounded once to fp16 (the matrix-core operand
// type; fp16 keeps the 1e-4*||w||*||x|| bound where bf16 does not), each
// token row on its own power-of-two scale (k_x_to_f16), and
// v_mfma_f32_32x32x16_f16 accumulates in fp32.  A dot product over fp16
// operands errs by about 2.8e-4 ||w|| ||x|| / sqrt(K) on random data, so short
// rows need more care: rows of at most 512 columns, and the fp32-operand
// entry point, run k_prefill_q4k_split (below); rows of at most 2048 columns
// round each weight once from its exact value (k_prefill_q4k<true>) instead
// of through fp16 sub-block scales.
//
// Tile: 64 tokens x 128 weight rows per workgroup of 8 waves (256
// workgroups at 512 x 4096 x 4096).  Both operands of one Q4_K block column
// (256 k: 32 KB of fp16 activations, 18 KB of weight blocks) stream through
// a three-slot LDS ring filled by direct-to-LDS 128-bit copies: while a wave
// reduces column kb from registers it reads column kb + 1 out of the ring,
// and the copies of columns kb + 2 and kb + 3 are in flight.  Wave (rh, j)
// reduces weight rows 64 rh .. 64 rh + 63 of the tile over sub-block pair j
// of every column, dequantizing its matrix-core operand straight from the
// block bytes into registers (every weight is dequantized once per
// workgroup; the two lane halves decode one row's scales each).  The weights are the A operand, so each
// lane ends with 4 consecutive output rows of one token: the four K-quarter
// partial sums meet in LDS and leave as 16-byte stores.
#include "kq_common.h"
#include "kq_launch.h"

#include <type_traits>

namespace ihip {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int PF_BM = kPrefillBM, PF_BN = kPrefillBN; // workgroup tile: tokens x weight rows

// One token row of X to fp16 (one workgroup per row, 8 values per thread and
// step: two 16-byte loads, one 16-byte store).  The reference multiplies fp32
// activations of any finite size (src/ModelCPU.jl:285-307), while fp16 holds
// magnitudes up to 65504 only and rounds those below 2^-14 to its subnormal
// steps.  So every row is scaled by a power of two 2^s, chosen so that its
// largest magnitude lands in [2^14, 2^15), before the rounding, and s goes to
// xs[t]; the GEMM's epilogue multiplies the row's outputs by 2^-s, which is
// exact.  Every value keeps fp16's 11 significant bits down to 2^-29 of the
// row's maximum.  A row holding NaN or an infinity is converted unscaled
// (s = 0), so the non-finite value reaches its outputs.  Rows of at most
// 8192 values stay in registers between the maximum and the conversion;
// longer rows are read twice.
//
// Order of a row in Xh: its 256-column blocks in order, and inside a block its
// 32 chunks of 8 values (16 bytes) by (stage g, half h, c), chunk 16 h + 4 g +
// c at place 8 g + 4 h + c.  The wide kernel below multiplies a block in four
// stages, lane half h of its matrix products covering columns 128 h + 32 g +
// 8 c ..: with this order a stage of a token row is 128 contiguous bytes.
// element i (a multiple of 8) of a row -> its element offset in Xh's row
__device__ __forceinline__ int pf_x_place(int i) { return (i & ~255) + 8 * pf_chunk_place((i & 255) >> 3); }
constexpr int PF_CVT_REG = 4; // 8-value steps a thread holds: 256 x 8 x 4 = 8192 values
__global__ __launch_bounds__(256) void k_x_to_f16(const float *__restrict__ X,
                                                  _Float16 *__restrict__ Xh, int *__restrict__ xs,
                                                  int K)
{
    __shared__ uint32_t wmax[4];
    const int t = blockIdx.x, tid = threadIdx.x;
    const float *row = X + (size_t)t * K;
    _Float16 *hrow = Xh + (size_t)t * K;
    // |x| bits of eight values: NaN > +Inf > every finite value
    auto absmax8 = [](float4 a, float4 b) {
        const uint32_t m0 = max(__float_as_uint(a.x) & 0x7fffffffu, __float_as_uint(a.y) & 0x7fffffffu);
        const uint32_t m1 = max(__float_as_uint(a.z) & 0x7fffffffu, __float_as_uint(a.w) & 0x7fffffffu);
        const uint32_t m2 = max(__float_as_uint(b.x) & 0x7fffffffu, __float_as_uint(b.y) & 0x7fffffffu);
        const uint32_t m3 = max(__float_as_uint(b.z) & 0x7fffffffu, __float_as_uint(b.w) & 0x7fffffffu);
        return max(max(m0, m1), max(m2, m3));
    };
    const bool in_regs = K <= 256 * 8 * PF_CVT_REG; // workgroup-uniform
    float4 v[PF_CVT_REG][2];
    uint32_t m = 0;
    if (in_regs) {
#pragma unroll
        for (int k = 0; k < PF_CVT_REG; ++k) {
            const int i = 8 * (tid + 256 * k);
            v[k][0] = v[k][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < K) { // K is a multiple of 256: whole 8-value steps
                v[k][0] = *reinterpret_cast<const float4 *>(row + i);
                v[k][1] = *reinterpret_cast<const float4 *>(row + i + 4);
            }
            m = max(m, absmax8(v[k][0], v[k][1]));
        }
    } else {
        for (int i = 8 * tid; i < K; i += 8 * 256)
            m = max(m, absmax8(*reinterpret_cast<const float4 *>(row + i),
                               *reinterpret_cast<const float4 *>(row + i + 4)));
    }
    // the row's maximum: DPP steps within each row of 16 lanes, then the
    // four rows' and the four waves' values through LDS
    m = dpp_max_u32<0xb1, 0xf>(m);
    m = dpp_max_u32<0x4e, 0xf>(m);
    m = dpp_max_u32<0x141, 0xf>(m);
    m = dpp_max_u32<0x140, 0xf>(m);
    {
        const int lane = tid & 63, w = tid >> 6;
        const uint32_t r0 = __builtin_amdgcn_readlane(m, 0), r1 = __builtin_amdgcn_readlane(m, 16);
        const uint32_t r2 = __builtin_amdgcn_readlane(m, 32), r3 = __builtin_amdgcn_readlane(m, 48);
        if (lane == 0)
            wmax[w] = max(max(r0, r1), max(r2, r3));
    }
    __syncthreads();
    m = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    const bool finite = m < 0x7f800000u;
    // m = 0 (an all-zero row): frexp's exponent is 0, any scale keeps the zeros
    const int s = finite ? 15 - __builtin_amdgcn_frexp_expf(__uint_as_float(m)) : 0;
    auto cvt8 = [s](float4 a, float4 b) {
        half8 h;
        h[0] = (_Float16)__builtin_ldexpf(a.x, s); h[1] = (_Float16)__builtin_ldexpf(a.y, s);
        h[2] = (_Float16)__builtin_ldexpf(a.z, s); h[3] = (_Float16)__builtin_ldexpf(a.w, s);
        h[4] = (_Float16)__builtin_ldexpf(b.x, s); h[5] = (_Float16)__builtin_ldexpf(b.y, s);
        h[6] = (_Float16)__builtin_ldexpf(b.z, s); h[7] = (_Float16)__builtin_ldexpf(b.w, s);
        return h;
    };
    if (in_regs) {
#pragma unroll
        for (int k = 0; k < PF_CVT_REG; ++k) {
            const int i = 8 * (tid + 256 * k);
            if (i < K)
                *reinterpret_cast<half8 *>(hrow + pf_x_place(i)) = cvt8(v[k][0], v[k][1]);
        }
    } else {
        for (int i = 8 * tid; i < K; i += 8 * 256)
            *reinterpret_cast<half8 *>(hrow + pf_x_place(i)) =
                cvt8(*reinterpret_cast<const float4 *>(row + i), *reinterpret_cast<const float4 *>(row + i + 4));
    }
    if (tid == 0)
        xs[t] = s;
}

// One ring slot holds block column kb of both operands:
//  * activations, 64 token rows x 512 bytes: row m holds 32 chunks of 16
//    bytes, chunk c at slot c ^ (m & 15), so that the 16 lanes of a 128-bit
//    read (same chunk, consecutive rows) hit distinct banks;
//  * weights, 128 rows x 144 bytes: the rows' Q4_K blocks of column kb.
constexpr int PF_ROW_BYTES = 512;
constexpr int PF_A_STAGE = PF_BM * PF_ROW_BYTES; // 32 KB
constexpr int PF_B_STAGE = PF_BN * 144;          // 18 KB
constexpr int PF_SLOT = PF_A_STAGE + PF_B_STAGE; // 50 KB
constexpr int PF_NSLOT = 3;
constexpr int PF_THREADS = 512;                  // 8 waves
constexpr int PF_B_COPIES = PF_B_STAGE / 1024;   // 18 wave copies of 1 KB

static_assert(PF_B_STAGE % 1024 == 0, "weight stage is whole wave copies");
static_assert(PF_NSLOT * PF_SLOT <= 160 * 1024, "ring fits the 160 KB of LDS");

// One direct-to-LDS copy: lane l's 16 bytes at base + off land at LDS byte
// lds + 16 l.  The base is wave-uniform (scalar registers) and the lane's
// offset a 32-bit register, so a column's copies cost no vector address
// arithmetic.  Written as inline assembly so that the compiler, which would
// otherwise make every later LDS read wait for all copies in flight
// (including those issued ahead for later block columns), leaves the waits to
// the explicit per-wave s_waitcnt of the main loop.
__device__ __forceinline__ void pf_copy16(const void *base, uint32_t off, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(off), "s"(base), "s"(lds)
                 : "memory", "m0");
}

// Per-lane byte offsets of the copies of block column 0 (from Xh and from W);
// column kb adds 512 kb bytes (activations) or 144 kb bytes (weights) to the
// wave-uniform base.  Wave w issues activation
// copies w, w + 8, w + 16, w + 24 (64 chunks each: chunk q = stage row q / 32,
// activation chunk (q % 32) ^ (row & 15)) and weight copies w, w + 8 and, for
// w < 2, w + 16 (chunk q = tile row q / 9, 16-byte piece q % 9): 7 copies for
// waves 0-1, 6 for the others.  Rows past T (tokens) or N (weights) re-read
// the last row.
struct PfSrc {
    uint32_t a0, a1, a2, a3, b0, b1, b2; // plain members: kept in registers
};

__device__ __forceinline__ uint32_t pf_src_a(int m0, int T, int K, int w, int lane, int k)
{
    const int q = (8 * k + w) * 64 + lane;
    const int rp = q >> 5, c = (q & 31) ^ (rp & 15);
    return 2u * ((uint32_t)min(m0 + rp, T - 1) * (uint32_t)K + 8u * (uint32_t)c);
}

__device__ __forceinline__ uint32_t pf_src_b(int n0, int N, uint32_t row_bytes, int lane, int i)
{
    const int q = 64 * min(i, PF_B_COPIES - 1) + lane;
    const int row = q / 9, piece = q - 9 * row;
    return (uint32_t)min(n0 + row, N - 1) * row_bytes + 16u * (uint32_t)piece;
}

// Issue this wave's copies of block column kb into the ring slot at LDS
// address `slot`.
__device__ __forceinline__ void pf_issue(const PfSrc &S, const uint8_t *Xb, const uint8_t *W, int kb,
                                         int w, uint32_t slot)
{
    const uint8_t *xa = Xb + (size_t)kb * 512, *wb = W + (size_t)kb * 144;
    pf_copy16(xa, S.a0, slot + 1024 * w);
    pf_copy16(xa, S.a1, slot + 1024 * (w + 8));
    pf_copy16(xa, S.a2, slot + 1024 * (w + 16));
    pf_copy16(xa, S.a3, slot + 1024 * (w + 24));
    pf_copy16(wb, S.b0, slot + PF_A_STAGE + 1024 * w);
    pf_copy16(wb, S.b1, slot + PF_A_STAGE + 1024 * (w + 8));
    if (w + 16 < PF_B_COPIES) // wave-uniform
        pf_copy16(wb, S.b2, slot + PF_A_STAGE + 1024 * (w + 16));
}

// 8 nibbles (the low or high nibble of 8 bytes) -> 8 fp16 weights
// q * dsc - dmm.  A byte 0000qqqq is the OCP e4m3 encoding of q * 2^-9; the
// scaled convert multiplies by 2^9, giving q exactly in fp16, and one packed
// fp16 FMA per pair applies the sub-block scale and min.
__device__ __forceinline__ half8 pf_dequant8(uint2 bytes, bool high, half2v dsc, half2v dmm)
{
    uint32_t w0 = bytes.x, w1 = bytes.y;
    if (high) {
        w0 >>= 4;
        w1 >>= 4;
    }
    w0 &= 0x0f0f0f0fu;
    w1 &= 0x0f0f0f0fu;
    const half2v q01 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 512.0f, false);
    const half2v q23 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 512.0f, true);
    const half2v q45 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 512.0f, false);
    const half2v q67 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 512.0f, true);
    const half2v r01 = __builtin_elementwise_fma(q01, dsc, dmm);
    const half2v r23 = __builtin_elementwise_fma(q23, dsc, dmm);
    const half2v r45 = __builtin_elementwise_fma(q45, dsc, dmm);
    const half2v r67 = __builtin_elementwise_fma(q67, dsc, dmm);
    half8 r;
    r[0] = r01[0]; r[1] = r01[1]; r[2] = r23[0]; r[3] = r23[1];
    r[4] = r45[0]; r[5] = r45[1]; r[6] = r67[0]; r[7] = r67[1];
    return r;
}

// The same 8 weights rounded once from their exact fp32 values,
// rn16((d sc) q - dmin m): q exact in fp32 from the scaled convert, one fp32
// FMA (d sc q is exact, so the FMA rounds only the difference), then
// v_cvt_pk_f16_f32.  Rounding d sc and dmin m to fp16 first, as
// pf_dequant8 does, puts one shared relative error on all 32 weights of a
// sub-block; this form leaves each weight its own.
__device__ __forceinline__ half8 pf_dequant8_exact(uint2 bytes, bool high, float dsc, float dmm)
{
    typedef float f2v __attribute__((ext_vector_type(2)));
    uint32_t w0 = bytes.x, w1 = bytes.y;
    if (high) {
        w0 >>= 4;
        w1 >>= 4;
    }
    w0 &= 0x0f0f0f0fu;
    w1 &= 0x0f0f0f0fu;
    const f2v q01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w0, 512.0f, false);
    const f2v q23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w0, 512.0f, true);
    const f2v q45 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w1, 512.0f, false);
    const f2v q67 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w1, 512.0f, true);
    const f2v r01 = {fmaf(q01[0], dsc, dmm), fmaf(q01[1], dsc, dmm)};
    const f2v r23 = {fmaf(q23[0], dsc, dmm), fmaf(q23[1], dsc, dmm)};
    const f2v r45 = {fmaf(q45[0], dsc, dmm), fmaf(q45[1], dsc, dmm)};
    const f2v r67 = {fmaf(q67[0], dsc, dmm), fmaf(q67[1], dsc, dmm)};
    const half2v h01 = __builtin_convertvector(r01, half2v), h23 = __builtin_convertvector(r23, half2v);
    const half2v h45 = __builtin_convertvector(r45, half2v), h67 = __builtin_convertvector(r67, half2v);
    half8 r;
    r[0] = h01[0]; r[1] = h01[1]; r[2] = h23[0]; r[3] = h23[1];
    r[4] = h45[0]; r[5] = h45[1]; r[6] = h67[0]; r[7] = h67[1];
    return r;
}

// One column's operands of this lane, read from a ring slot: 2 x 8 quant
// bytes of weight rows `blk0` / `blk1` (rows li and li + 32 of the wave's 64)
// for sub-block pair j, the block header of row li + 32 h only (the two lane
// halves decode one row's scales each and exchange them), and the 16-byte
// fp16 activation chunks of tokens li and li + 32 for the four 16-wide K
// steps (k = 64j + 16s + 8h + (0..7), chunk 8j + 2s + h).
struct PfOps {
    uint4 hd;
    uint2 q0[2], q1[2];
    half8 x[4][2];
};

__device__ __forceinline__ void pf_read(const uint8_t *sa, const uint8_t *blk0, const uint8_t *blk1,
                                        int j, int h, int li, PfOps &o)
{
    o.hd = *reinterpret_cast<const uint4 *>(h ? blk1 : blk0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint8_t *blk = u ? blk1 : blk0;
        o.q0[u] = *reinterpret_cast<const uint2 *>(blk + 16 + 32 * j + 8 * h);
        o.q1[u] = *reinterpret_cast<const uint2 *>(blk + 16 + 32 * j + 16 + 8 * h);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int m = 32 * t + li;
            const int c = 16 * (j & 1) + 8 * (s >> 1) + 4 * (j >> 1) + 2 * (s & 1) + h; // pf_chunk_place(8j + 2s + h)
            o.x[s][t] = *reinterpret_cast<const half8 *>(sa + m * PF_ROW_BYTES + 16 * (c ^ (m & 15)));
        }
}

// Dequantize the column's weights into matrix-core operands and accumulate.
// acc[u][t] is the 32 x 32 tile (weight rows 32u.., tokens 32t..): lane l,
// register r hold token 32t + l % 32, weight row 32u + 8 (r / 4) + 4 (l / 32) + r % 4.
// EXACTW: each weight rounded once from its exact value (pf_dequant8_exact),
// for rows of at most kPrefillExactWMaxK columns, where the shared rounding
// of a sub-block's scale averages over too few sub-blocks.
template <bool EXACTW>
__device__ __forceinline__ void pf_mma(const PfOps &o, int j, float16v (&acc)[2][2])
{
    // Scale d*sc and min -dmin*m of sub-blocks 2j (A) and 2j + 1 (B) for
    // this lane half's row (rounded once to fp16 and packed (A, B), or kept
    // in fp32 when EXACTW) ...
    const float d = h2f(o.hd.x & 0xffffu), dmin = h2f(o.hd.x >> 16);
    float scA, mA, scB, mB;
    k_scale_min_pair(o.hd.y, o.hd.z, o.hd.w, j, scA, mA, scB, mB);
    // ... then exchanged between the lane halves: v_permlane32_swap of a
    // register with itself leaves lanes 0-31's value (row li) in the first
    // result and lanes 32-63's (row li + 32) in the second, in every lane.
    if constexpr (EXACTW) {
        const float dsa = d * scA, dsb = d * scB, dma = -(dmin * mA), dmb = -(dmin * mB);
        const auto xa = __builtin_amdgcn_permlane32_swap(__float_as_uint(dsa), __float_as_uint(dsa), false, false);
        const auto xb = __builtin_amdgcn_permlane32_swap(__float_as_uint(dsb), __float_as_uint(dsb), false, false);
        const auto ya = __builtin_amdgcn_permlane32_swap(__float_as_uint(dma), __float_as_uint(dma), false, false);
        const auto yb = __builtin_amdgcn_permlane32_swap(__float_as_uint(dmb), __float_as_uint(dmb), false, false);
        float dsA[2], dmA[2], dsB[2], dmB[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            dsA[u] = __uint_as_float((uint32_t)xa[u]);
            dsB[u] = __uint_as_float((uint32_t)xb[u]);
            dmA[u] = __uint_as_float((uint32_t)ya[u]);
            dmB[u] = __uint_as_float((uint32_t)yb[u]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const half8 wq = pf_dequant8_exact((s & 1) ? o.q1[u] : o.q0[u], s >= 2,
                                                   s >= 2 ? dsB[u] : dsA[u], s >= 2 ? dmB[u] : dmA[u]);
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, o.x[s][t], acc[u][t], 0, 0, 0);
            }
    } else {
        const half2v ds = {(_Float16)(d * scA), (_Float16)(d * scB)};
        const half2v dm = {(_Float16)(-(dmin * mA)), (_Float16)(-(dmin * mB))};
        const uint32_t dsu = __builtin_bit_cast(uint32_t, ds), dmu = __builtin_bit_cast(uint32_t, dm);
        const auto xs = __builtin_amdgcn_permlane32_swap(dsu, dsu, false, false);
        const auto xm = __builtin_amdgcn_permlane32_swap(dmu, dmu, false, false);
        half2v dsA[2], dmA[2], dsB[2], dmB[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const half2v s2 = __builtin_bit_cast(half2v, (uint32_t)xs[u]);
            const half2v m2 = __builtin_bit_cast(half2v, (uint32_t)xm[u]);
            dsA[u] = half2v{s2[0], s2[0]};
            dmA[u] = half2v{m2[0], m2[0]};
            dsB[u] = half2v{s2[1], s2[1]};
            dmB[u] = half2v{m2[1], m2[1]};
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const half8 wq = pf_dequant8((s & 1) ? o.q1[u] : o.q0[u], s >= 2, s >= 2 ? dsB[u] : dsA[u],
                                             s >= 2 ? dmB[u] : dmA[u]);
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, o.x[s][t], acc[u][t], 0, 0, 0);
            }
    }
}

// Wait for this wave's copies, leaving the last n in flight (n is 0 or one
// or two columns' copy counts, 6 or 7 each), and for its LDS reads: after the
// next barrier no wave still reads a slot that a copy is about to refill.
static_assert(PF_B_COPIES == 18, "copy counts 7 (waves 0-1) and 6");
__device__ __forceinline__ void pf_wait_copies(int n)
{
    switch (n) {
    case 14: __builtin_amdgcn_s_waitcnt(14 | 0x0070); break; // vmcnt(14) lgkmcnt(0)
    case 12: __builtin_amdgcn_s_waitcnt(12 | 0x0070); break;
    case 7: __builtin_amdgcn_s_waitcnt(7 | 0x0070); break;
    case 6: __builtin_amdgcn_s_waitcnt(6 | 0x0070); break;
    default: __builtin_amdgcn_s_waitcnt(0 | 0x0070); break; // vmcnt(0) lgkmcnt(0)
    }
}

// Y[t, n] = sum_k W[n, k] Xh[t, k] for one 64-token x 128-row tile, over
// the block columns of one split of K: split sp of nsplit takes columns
// sp * nblk / nsplit .. (sp + 1) * nblk / nsplit - 1 and writes its sums to
// Y (split 0) or to partial plane sp - 1 of `part` (T x N floats each), which
// k_prefill_splits_sum then adds into Y.  Wave (rh, j) = (wave & 1, wave >> 1)
// accumulates weight rows 64 rh .. +63 over sub-block pair j of every block
// column; at the end wave (rh, j) finishes tile combination c = j (weight
// half u = c >> 1, token half t = c & 1) of its row half from the four
// waves' partial sums.
template <bool EXACTW>
__global__ __launch_bounds__(PF_THREADS) void k_prefill_q4k(const uint8_t *__restrict__ W,
                                                            const _Float16 *__restrict__ Xh,
                                                            const int *__restrict__ xs,
                                                            float *__restrict__ Y,
                                                            float *__restrict__ part, int T, int K,
                                                            int N, int mtiles, int ntiles, int nsplit)
{
    __shared__ __attribute__((aligned(16))) uint8_t ring[PF_NSLOT * PF_SLOT];

    const int tiles = mtiles * ntiles;
    const int lin = prefill_lin((int)blockIdx.x, tiles, nsplit);
    if (lin >= tiles * nsplit)
        return; // whole workgroup

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rh = wave & 1, j = wave >> 1;
    const int h = lane >> 5, li = lane & 31;
    const int nblk = K / 256;
    const size_t row_bytes = (size_t)nblk * 144;
    const PrefillSplit ps = prefill_split_of(lin, mtiles, ntiles, nblk, nsplit);
    const int m0 = ps.mt * PF_BM, n0 = ps.nt * PF_BN;
    const int kb0 = ps.kb0, nk = ps.nk; // this split's block columns (nk >= 1)
    float *const out = ps.sp == 0 ? Y : part + (size_t)(ps.sp - 1) * (size_t)T * (size_t)N;
    const int brow = 64 * rh + li;                        // this lane's first weight row
    const int copies = 4 + (PF_B_COPIES - wave + 7) / 8; // copies this wave issues per column

    float16v acc[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][t][r] = 0.0f;

    // byte offsets below 2^32: the launcher checks T * K * 2 and N * row_bytes
    PfSrc S;
    S.a0 = pf_src_a(m0, T, K, wave, lane, 0);
    S.a1 = pf_src_a(m0, T, K, wave, lane, 1);
    S.a2 = pf_src_a(m0, T, K, wave, lane, 2);
    S.a3 = pf_src_a(m0, T, K, wave, lane, 3);
    S.b0 = pf_src_b(n0, N, (uint32_t)row_bytes, lane, wave);
    S.b1 = pf_src_b(n0, N, (uint32_t)row_bytes, lane, wave + 8);
    S.b2 = pf_src_b(n0, N, (uint32_t)row_bytes, lane, wave + 16);
    // the split's first block column: activations 512 bytes and weight rows
    // 144 bytes per column further on
    const uint8_t *Xb = reinterpret_cast<const uint8_t *>(Xh) + (size_t)kb0 * 512;
    W += (size_t)kb0 * 144;
    const uint32_t ring_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;

    // Column kb lives in slot kb % 3.  A wave reads column kb + 1 into
    // registers while it dequantizes and multiplies column kb, so the LDS
    // reads of the next column overlap this column's matrix-core work; the
    // copies of column kb + 3 go into column kb's slot, which every wave has
    // read (into registers) before the barrier of iteration kb.
    const int nfill = min(nk, PF_NSLOT);
    for (int c = 0; c < nfill; ++c)
        pf_issue(S, Xb, W, c, wave, ring_lds + c * PF_SLOT);
    pf_wait_copies((nfill - 1) * copies);
    lds_barrier();
    const uint8_t *ba = ring + PF_A_STAGE + brow * 144; // this lane's weight rows in slot 0
    PfOps o0, o1;
    pf_read(ring, ba, ba + 32 * 144, j, h, li, o0);

    // Block column kb, which has a successor: wait for the successor's
    // copies, publish it, refill column kb's slot (`slot` = kb % 3), read the
    // successor into `nxt`, then reduce `cur`.  The last column is reduced
    // after the loop, so that no branch inside the loop decides whether a
    // read was issued (the compiler would then wait for every LDS read in
    // flight, the successor's included, before the first matrix product).
    auto step = [&](int kb, int slot, PfOps &cur, PfOps &nxt) {
        pf_wait_copies(kb + 2 < nk ? copies : 0);
        lds_barrier();
        if (kb + 3 < nk)
            pf_issue(S, Xb, W, kb + 3, wave, ring_lds + slot * PF_SLOT);
        const int ns = slot == 2 ? 0 : slot + 1;
        pf_read(ring + ns * PF_SLOT, ba + ns * PF_SLOT, ba + ns * PF_SLOT + 32 * 144, j, h, li, nxt);
        __builtin_amdgcn_sched_barrier(0);
        pf_mma<EXACTW>(cur, j, acc);
    };
    int kb = 0, slot = 0;
    for (; kb + 2 < nk; kb += 2) {
        step(kb, slot, o0, o1);
        slot = slot == 2 ? 0 : slot + 1;
        step(kb + 1, slot, o1, o0);
        slot = slot == 2 ? 0 : slot + 1;
    }
    if (kb + 1 < nk) {
        step(kb, slot, o0, o1);
        pf_mma<EXACTW>(o1, j, acc);
    } else {
        pf_mma<EXACTW>(o0, j, acc);
    }
    __syncthreads(); // every wave is done with the ring

    // partial sums in LDS: float4 P[rh][c][src][q][lane] (128 KB), where
    // q = r / 4 picks 4 consecutive weight rows of one token
    float4 *P = reinterpret_cast<float4 *>(ring);
    auto pidx = [&](int c, int src, int q) { return (((rh * 4 + c) * 4 + src) * 4 + q) * 64 + lane; };
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c == j)
            continue; // wave-uniform
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float16v &a = acc[c >> 1][c & 1];
            P[pidx(c, j, q)] = make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c != j)
            continue; // wave-uniform: this wave finishes combination c
        const int u = c >> 1, t = c & 1;
        float4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            v[q] = make_float4(acc[u][t][4 * q], acc[u][t][4 * q + 1], acc[u][t][4 * q + 2],
                               acc[u][t][4 * q + 3]);
#pragma unroll
        for (int src = 0; src < 4; ++src) {
            if (src == j)
                continue;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 p = P[pidx(c, src, q)];
                v[q].x += p.x;
                v[q].y += p.y;
                v[q].z += p.z;
                v[q].w += p.w;
            }
        }
        const int m = m0 + 32 * t + li;
        if (m >= T)
            break;
        const int sm = -xs[m]; // undo the row's power-of-two scale (exact)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            v[q] = make_float4(__builtin_ldexpf(v[q].x, sm), __builtin_ldexpf(v[q].y, sm),
                               __builtin_ldexpf(v[q].z, sm), __builtin_ldexpf(v[q].w, sm));
        const int nb = n0 + 64 * rh + 32 * u + 4 * h; // + 8 q: 4 consecutive rows
        float *yrow = out + (size_t)m * N;
        if ((N & 3) == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (nb + 8 * q < N)
                    *reinterpret_cast<float4 *>(yrow + nb + 8 * q) = v[q];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = nb + 8 * q;
                if (n < N) yrow[n] = v[q].x;
                if (n + 1 < N) yrow[n + 1] = v[q].y;
                if (n + 2 < N) yrow[n + 2] = v[q].z;
                if (n + 3 < N) yrow[n + 3] = v[q].w;
            }
        }
    }
}

// Wide tiles, for products with enough of them to fill the chip: 128 tokens x
// 128 RU weight rows per workgroup of 4 waves, wave w holding rows 32 RU w ..
// of the tile against all 128 tokens, over all of K.  Against the 64 x 128
// tile above this dequantizes each weight once per 128 tokens instead of 64
// (half the vector work per matrix product), brings 200 KB (RU = 2; RU = 1:
// 330) from L2 per 256 x 256 x 256 product instead of 400, and needs no
// partial sums.
//
// LDS: two X stages of 64 columns (16 KB each) and one column's weight blocks
// of each wave's own rows (9 or 5 KB a wave): 68 KB for RU = 2, two workgroups
// per CU, 52 KB for RU = 1, three.  The workgroups of a CU run at their own
// pace, so one multiplies while another waits at its barrier.
//
// A wave runs K steps of 16 columns: while one step's 4 RU products run, the
// next step's activations are read from LDS and its weights dequantized
// (interleave() keeps the two streams mixed).  A stage is 4 steps.  Before the
// last step's products the wave waits for its copies of the next stage and
// for its LDS reads and meets the others; the stage's buffer is then free, so
// the copies of the stage after next go into it, with a whole stage's time to
// land, and the next stage's first operands are read behind the products.
// The raw weight bytes of a column go to registers (the first half with the
// header during the previous column's last stage), which frees the wave's
// weight buffer for the next column's copies.  Copies past the last stage or
// column repeat the last one, so the loop has no branches and every wait a
// constant count.
//
// Measured on MI355X (us, the product alone; 64 x 128 tiles before):
// 2048 x 12288 x 4096 181-186 against 287-305 (1.11-1.14 PFLOP/s), 512 x 14336 x
// 4096 62-64 against 95, 2048 x 4096 x 4096 69-70 against 98-101, 1024 x 4096 x
// 4096 40-41 (RU = 1) against 50-52.  The matrix cores are busy 58 % of the
// cycles at a clock that power holds at 1.6-1.8 GHz: fewer bytes and vector
// instructions per product raise the clock, reordering does not (priorities,
// another interleave, tile orders: within 1 %; non-temporal stores of Y 10-25 %
// slower).
constexpr int PFW_BM = kPrefillWideBM;
constexpr int PFW_XSTAGE = PFW_BM * 128; // 64 columns of 128 tokens, fp16
// 1 KB copies of a wave's 32 RU rows of one block column: 9, or 5 (the last half used)
__host__ __device__ constexpr int pfw_copies(int ru) { return (32 * ru * 144 + 1023) / 1024; }

template <bool EXACTW, int RU>
__global__ __launch_bounds__(256, RU == 2 ? 2 : 3) void k_prefill_q4k_wide(
    const uint8_t *__restrict__ W, const _Float16 *__restrict__ Xh, const int *__restrict__ xs,
    float *__restrict__ Y, int T, int K, int N, int mtiles, int ntiles)
{
    constexpr int WB = pfw_copies(RU), WREG = WB * 1024, TT = PFW_BM / 32, VPM = EXACTW ? 5 : 4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * PFW_XSTAGE + 4 * WREG];

    const int tiles = mtiles * ntiles;
    const int lin = prefill_lin((int)blockIdx.x, tiles, 1);
    if (lin >= tiles)
        return; // whole workgroup
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, li = lane & 31;
    const int nk = K / 256;
    const uint32_t row_bytes = (uint32_t)nk * 144u;
    const PrefillSplit ps = prefill_split_of(lin, mtiles, ntiles, nk, 1);
    const int m0 = ps.mt * PFW_BM, n0 = ps.nt * (128 * RU) + 32 * RU * wave; // this wave's first row

    // byte offsets of this wave's copies from Xh / W (stage 0, column 0):
    // tokens 32 wave .. +31 of the X stage and the wave's own weight rows.
    // Rows past T or N re-read the last one.
    uint32_t xo[4], wo[WB];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 32 * wave + pf_copy_token(i, lane);
        xo[i] = 2u * (uint32_t)min(m0 + m, T - 1) * (uint32_t)K + 16u * (uint32_t)pf_copy_chunk(m, lane);
    }
#pragma unroll
    for (int i = 0; i < WB; ++i) {
        const PfPiece q = pf_block_piece(i, lane, 32 * RU);
        wo[i] = (uint32_t)min(n0 + q.row, N - 1) * row_bytes + q.off;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t xdst = lds0 + 4096u * wave, wdst = lds0 + 2 * PFW_XSTAGE + (uint32_t)WREG * wave;
    const uint8_t *Xb = reinterpret_cast<const uint8_t *>(Xh);
    auto issue_x = [&](int st, int buf) {
        const uint8_t *b = Xb + (size_t)st * 128;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            pf_copy16(b, xo[i], xdst + PFW_XSTAGE * buf + 1024 * i);
    };
    auto issue_w = [&](int kb) {
        const uint8_t *b = W + (size_t)kb * 144;
#pragma unroll
        for (int i = 0; i < WB; ++i)
            pf_copy16(b, wo[i], wdst + 1024 * i);
    };

    float16v acc[RU][TT];
#pragma unroll
    for (int u = 0; u < RU; ++u)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][t][r] = 0.0f;

    const uint8_t *wl = lds + 2 * PFW_XSTAGE + WREG * wave + 144 * li;
    const uint8_t *xl[4]; // the lane's chunk of K step c in buffer 0, token li
#pragma unroll
    for (int c = 0; c < 4; ++c)
        xl[c] = lds + pf_stage_at(li, 4 * h + c);

    // lane (li, h): rows 32 u + li, columns 128 h .. 128 h + 127 of the block (qs
    // bytes 64 h ..): stage g is sub-block 4 h + g, K step c its bytes 8 c ..
    uint4 rq[RU][4], hdn[RU];
    uint32_t sc4[RU], mn4[RU];
    float d[RU], dmin[RU];
    auto read_w_lo = [&]() {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const uint8_t *b = wl + 32 * 144 * u;
            const uint4 hd = *reinterpret_cast<const uint4 *>(b);
            rq[u][0] = *reinterpret_cast<const uint4 *>(b + 16 + 64 * h);
            rq[u][1] = *reinterpret_cast<const uint4 *>(b + 16 + 64 * h + 16);
            hdn[u] = hd;
        }
    };
    auto decode_w = [&]() {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const uint4 hd = hdn[u];
            d[u] = h2f(hd.x & 0xffffu);
            dmin[u] = -h2f(hd.x >> 16);
            // sub-blocks 4h .. 4h + 3, one per byte (k_scale_min)
            const uint32_t sl = hd.y & 0x3f3f3f3fu, ml = hd.z & 0x3f3f3f3fu;
            const uint32_t sh = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
            const uint32_t mh = ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u);
            sc4[u] = h ? sh : sl;
            mn4[u] = h ? mh : ml;
        }
    };
    auto read_w_hi = [&]() {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const uint8_t *b = wl + 32 * 144 * u + 48 + 64 * h;
            rq[u][2] = *reinterpret_cast<const uint4 *>(b);
            rq[u][3] = *reinterpret_cast<const uint4 *>(b + 16);
        }
    };
    half8 xf[2][TT], wq[2][RU];
    float ds[RU], dm[RU];
    auto read_x = [&](int g, int c) { // into xf[c & 1]
#pragma unroll
        for (int t = 0; t < TT; ++t)
            xf[c & 1][t] = *reinterpret_cast<const half8 *>(xl[c] + PFW_XSTAGE * (g & 1) + 4096 * t);
    };
    auto dequant = [&](int g, int c) { // into wq[c & 1]
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            if (c == 0) {
                ds[u] = d[u] * ubyte_f(sc4[u], g);
                dm[u] = dmin[u] * ubyte_f(mn4[u], g);
            }
            const uint4 r4 = rq[u][2 * (g >> 1) + (c >> 1)];
            const uint2 by = (c & 1) ? make_uint2(r4.z, r4.w) : make_uint2(r4.x, r4.y);
            if constexpr (EXACTW) {
                wq[c & 1][u] = pf_dequant8_exact(by, (g & 1) != 0, ds[u], dm[u]);
            } else {
                const _Float16 s16 = (_Float16)ds[u], m16 = (_Float16)dm[u];
                wq[c & 1][u] = pf_dequant8(by, (g & 1) != 0, half2v{s16, s16}, half2v{m16, m16});
            }
        }
    };
    auto mma = [&](int c) {
#pragma unroll
        for (int u = 0; u < RU; ++u)
#pragma unroll
            for (int t = 0; t < TT; ++t)
                acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq[c & 1][u], xf[c & 1][t], acc[u][t], 0, 0, 0);
    };
    // mixes a step's LDS reads, products and the next step's dequantization
    auto interleave = [&]() {
        __builtin_amdgcn_sched_group_barrier(0x100, TT, 0);
#pragma unroll
        for (int i = 0; i < RU * TT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const int nst = 4 * nk;
    issue_w(0);
    issue_x(0, 0);
    issue_x(1, 1);
    __builtin_amdgcn_s_waitcnt(4 | 0x0070);
    lds_barrier();
    read_w_lo();
    decode_w();
    read_x(0, 0);
    dequant(0, 0);
    for (int kb = 0; kb < nk; ++kb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (g == 0)
                read_w_hi();
            if (g == 3)
                read_w_lo(); // the next column's
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                read_x(g, c + 1);
                mma(c);
                dequant(g, c + 1);
                interleave();
            }
            // the next stage has landed, and every wave holds this one in registers
            if (g == 1)
                __builtin_amdgcn_s_waitcnt(WB | 0x0070);
            else
                __builtin_amdgcn_s_waitcnt(0x0070);
            lds_barrier();
            issue_x(min(4 * kb + g + 2, nst - 1), g & 1);
            if (g == 0)
                issue_w(min(kb + 1, nk - 1));
            __builtin_amdgcn_sched_barrier(0);
            read_x(g + 1, 0);
            mma(3);
            if (g == 3)
                decode_w();
            dequant((g + 1) & 3, 0);
            interleave();
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0070); // the last (unused) copies have landed

#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int m = m0 + 32 * t + li;
        if (m >= T)
            continue;
        const int sm = -xs[m]; // undo the row's power-of-two scale (exact)
        float *yrow = Y + (size_t)m * N;
#pragma unroll
        for (int u = 0; u < RU; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = make_float4(__builtin_ldexpf(acc[u][t][4 * q], sm), __builtin_ldexpf(acc[u][t][4 * q + 1], sm),
                                             __builtin_ldexpf(acc[u][t][4 * q + 2], sm), __builtin_ldexpf(acc[u][t][4 * q + 3], sm));
                const int n = n0 + 32 * u + 8 * q + 4 * h;
                if ((N & 3) == 0) {
                    if (n < N)
                        *reinterpret_cast<float4 *>(yrow + n) = v;
                } else {
                    if (n < N) yrow[n] = v.x;
                    if (n + 1 < N) yrow[n + 1] = v.y;
                    if (n + 2 < N) yrow[n + 2] = v.z;
                    if (n + 3 < N) yrow[n + 3] = v.w;
                }
            }
    }
}

// Small products: 32 tokens x 64 weight rows per workgroup of 8 waves that share
// K.  Wave (half, j) takes sub-block pair j of the block columns 2 i + half and
// accumulates the whole tile, so every activation and every weight byte of
// the tile is read and dequantized by one wave only, each wave copies its own
// operands through LDS and waits for nothing but them, and a weight of few
// rows still has eight waves at work on each tile.  A step's operands go to
// registers before its products, which frees the wave's LDS for the next
// step's copies; two workgroups share a CU (57 KB).  The eight partial tiles
// are added up in LDS in a fixed order: waves w and w + 4, then 0..3.
//
// Bound by the copies (a 48-byte piece of a weight row touches three or four
// cache lines a quad of lanes): wider tiles (64 to 128 tokens, 128 rows) copy
// less but leave CUs idle, and were slower wherever this kernel is taken.
// Measured on MI355X (us, graph replays, the 64 x 128 tile / this): 8 x 1024 x
// 2048 (tokens x columns x rows) 8.9 / 5.3, 256 x 1024 x 2048 10.8 / 6.2, 8 x 2560
// x 9728 11.7 / 7.7, 77 x 2560 x 9728 16.2 / 14.7, 128 x 4096 x 4096 15.4 / 11.8, 512
// x 2048 x 512 11.0 / 8.1.
constexpr int PFT_BM = kPrefillThinBM, PFT_BN = kPrefillThinBN, PFT_RU = PFT_BN / 32;
constexpr int PFT_X = 4096, PFT_WAVE = PFT_X + 48 * PFT_BN; // bytes of a wave's step: 64 columns of X, the rows' pieces
constexpr int PFT_LD = PFT_BN + 4;                          // floats between two tokens of a partial tile
static_assert(PFT_BM == 32 && 8 * PFT_WAVE >= 4 * 4 * PFT_BM * PFT_LD, "four partial tiles fit the waves' LDS");

template <bool EXACTW>
__global__ __launch_bounds__(512, 2) void k_prefill_q4k_thin(const uint8_t *__restrict__ W,
                                                             const _Float16 *__restrict__ Xh,
                                                             const int *__restrict__ xs, float *__restrict__ Y,
                                                             int T, int K, int N, int mtiles, int ntiles)
{
    constexpr int RU = PFT_RU, XC = 4, WC = 3 * PFT_BN / 64; // 1 KB copies of a step
    constexpr int LD = PFT_LD;
    __shared__ __attribute__((aligned(16))) uint8_t lds[8 * PFT_WAVE];

    const int tiles = mtiles * ntiles;
    const int lin = prefill_lin((int)blockIdx.x, tiles, 1);
    if (lin >= tiles)
        return; // whole workgroup
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, li = lane & 31, j = wave & 3, half = wave >> 2;
    const int nk = K / 256;
    const uint32_t row_bytes = (uint32_t)nk * 144u;
    const PrefillSplit ps = prefill_split_of(lin, mtiles, ntiles, nk, 1);
    const int m0 = ps.mt * PFT_BM, n0 = ps.nt * PFT_BN;

    float16v acc[RU];
#pragma unroll
    for (int u = 0; u < RU; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] = 0.0f;

    const int nb = (nk - half + 1) >> 1; // this wave's steps
    if (nb > 0) {
        // copies: the pair's 64 columns of X, and header and 32 quant bytes of
        // every row.  Rows past T or N re-read the last one, steps past the
        // last repeat it.
        uint32_t xo[XC], wo[WC];
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const int m = pf_copy_token(i, lane);
            xo[i] = 2u * (uint32_t)min(m0 + m, T - 1) * (uint32_t)K +
                    16u * (uint32_t)pf_chunk_place(8 * j + pf_copy_chunk(m, lane));
        }
#pragma unroll
        for (int i = 0; i < WC; ++i) {
            const PfPiece q = pf_pair_piece(i, lane, j);
            wo[i] = (uint32_t)min(n0 + q.row, N - 1) * row_bytes + q.off;
        }
        uint8_t *const mine = lds + PFT_WAVE * wave;
        const uint32_t xdst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mine;
        const uint8_t *Xb = reinterpret_cast<const uint8_t *>(Xh) + 512 * half, *Wb = W + 144 * half;
        auto issue = [&](int i) {
            const int st = min(i, nb - 1);
            const uint8_t *x = Xb + (size_t)st * 1024, *w = Wb + (size_t)st * 288;
#pragma unroll
            for (int k = 0; k < WC; ++k)
                pf_copy16(w, wo[k], xdst + PFT_X + 1024 * k);
#pragma unroll
            for (int k = 0; k < XC; ++k)
                pf_copy16(x, xo[k], xdst + 1024 * k);
        };
        const uint8_t *wl = mine + PFT_X + 48 * li;
        issue(0);
        for (int i = 0; i < nb; ++i) {
            __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0): this step's copies
            asm volatile("" ::: "memory");
            half8 x[4];
            uint2 q[RU][2];
            uint4 hd[RU / 2]; // of the row tiles 2 v + h
#pragma unroll
            for (int v = 0; v < RU / 2; ++v)
                hd[v] = *reinterpret_cast<const uint4 *>(wl + 32 * 48 * (2 * v + h));
#pragma unroll
            for (int u = 0; u < RU; ++u)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    q[u][c] = *reinterpret_cast<const uint2 *>(wl + 32 * 48 * u + 16 + 16 * c + 8 * h);
#pragma unroll
            for (int s = 0; s < 4; ++s)
                x[s] = *reinterpret_cast<const half8 *>(mine + pf_stage_at(li, 2 * s + h));
            __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): in registers
            asm volatile("" ::: "memory");
            issue(i + 1);
            // scale and min of sub-blocks 2j, 2j + 1: each lane half decodes its
            // row tiles' and the halves exchange them (pf_mma)
            float dsf[EXACTW ? RU : 1][2], dmf[EXACTW ? RU : 1][2];
            half2v ds[RU], dm[RU];
#pragma unroll
            for (int v = 0; v < RU / 2; ++v) {
                const float d = h2f(hd[v].x & 0xffffu), dmin = h2f(hd[v].x >> 16);
                float scA, mA, scB, mB;
                k_scale_min_pair(hd[v].y, hd[v].z, hd[v].w, j, scA, mA, scB, mB);
                auto both = [](float a) {
                    return __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
                };
                if constexpr (EXACTW) {
                    const auto xa = both(d * scA), xb = both(d * scB), ya = both(-(dmin * mA)), yb = both(-(dmin * mB));
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        dsf[2 * v + k][0] = __uint_as_float((uint32_t)xa[k]);
                        dsf[2 * v + k][1] = __uint_as_float((uint32_t)xb[k]);
                        dmf[2 * v + k][0] = __uint_as_float((uint32_t)ya[k]);
                        dmf[2 * v + k][1] = __uint_as_float((uint32_t)yb[k]);
                    }
                } else {
                    const half2v s2 = {(_Float16)(d * scA), (_Float16)(d * scB)};
                    const half2v m2 = {(_Float16)(-(dmin * mA)), (_Float16)(-(dmin * mB))};
                    const auto xa = both(__builtin_bit_cast(float, s2)), ya = both(__builtin_bit_cast(float, m2));
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        ds[2 * v + k] = __builtin_bit_cast(half2v, (uint32_t)xa[k]);
                        dm[2 * v + k] = __builtin_bit_cast(half2v, (uint32_t)ya[k]);
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int u = 0; u < RU; ++u) {
                    half8 wq;
                    if constexpr (EXACTW)
                        wq = pf_dequant8_exact(q[u][s & 1], s >= 2, dsf[u][s >> 1], dmf[u][s >> 1]);
                    else {
                        const _Float16 a = ds[u][s >> 1], b = dm[u][s >> 1];
                        wq = pf_dequant8(q[u][s & 1], s >= 2, half2v{a, a}, half2v{b, b});
                    }
                    acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, x[s], acc[u], 0, 0, 0);
                }
        }
        __builtin_amdgcn_s_waitcnt(0x0f70); // the last (unused) copies have landed
    }
    __syncthreads();

    // lane (li, h), register 4 q + r of acc[u]: token li, row 32 u + 8 q + 4 h + r
    float *const P = reinterpret_cast<float *>(lds);
    auto place = [&](int w, int u, int q) {
        return reinterpret_cast<float4 *>(P + (PFT_BM * w + li) * LD + 32 * u + 8 * q + 4 * h);
    };
    auto put = [&](int w) {
#pragma unroll
        for (int u = 0; u < RU; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *place(w, u, q) = make_float4(acc[u][4 * q], acc[u][4 * q + 1], acc[u][4 * q + 2], acc[u][4 * q + 3]);
    };
    if (wave >= 4)
        put(wave - 4);
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int u = 0; u < RU; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 p = *place(wave, u, q);
                acc[u][4 * q] += p.x;
                acc[u][4 * q + 1] += p.y;
                acc[u][4 * q + 2] += p.z;
                acc[u][4 * q + 3] += p.w;
            }
        put(wave);
    }
    __syncthreads();
    // 16 threads a token, four rows each
    const int ml = tid >> 4, nl = 4 * (tid & 15), m = m0 + ml, n = n0 + nl;
    if (m >= T || n >= N)
        return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float4 p = *reinterpret_cast<const float4 *>(P + (PFT_BM * w + ml) * LD + nl);
        v.x += p.x;
        v.y += p.y;
        v.z += p.z;
        v.w += p.w;
    }
    const int sm = -xs[m]; // undo the row's power-of-two scale (exact)
    v = make_float4(__builtin_ldexpf(v.x, sm), __builtin_ldexpf(v.y, sm), __builtin_ldexpf(v.z, sm),
                    __builtin_ldexpf(v.w, sm));
    float *y = Y + (size_t)m * N + n;
    if ((N & 3) == 0) {
        *reinterpret_cast<float4 *>(y) = v;
    } else {
        y[0] = v.x;
        if (n + 1 < N) y[1] = v.y;
        if (n + 2 < N) y[2] = v.z;
        if (n + 3 < N) y[3] = v.w;
    }
}

// Y += P[0] + P[1] + ... + P[nparts - 1] (n floats each), in that order, so
// the result does not depend on which split finished first.
template <bool VEC>
__global__ __launch_bounds__(256) void k_prefill_splits_sum(float *__restrict__ Y,
                                                            const float *__restrict__ P, int64_t n,
                                                            int nparts)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    if constexpr (VEC) { // n % 4 == 0: every plane starts 16-byte aligned
        float4 *Y4 = reinterpret_cast<float4 *>(Y);
        const float4 *P4 = reinterpret_cast<const float4 *>(P);
        const int64_t n4 = n >> 2;
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) {
            float4 v = Y4[i];
            for (int q = 0; q < nparts; ++q) {
                const float4 p = P4[q * n4 + i];
                v.x += p.x;
                v.y += p.y;
                v.z += p.z;
                v.w += p.w;
            }
            Y4[i] = v;
        }
    } else {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
            float v = Y[i];
            for (int q = 0; q < nparts; ++q)
                v += P[q * n + i];
            Y[i] = v;
        }
    }
}

// The fp32-operand product: for rows of at most kPrefillF32MaxK columns, and
// at any length for callers that ask for it (launch_prefill_q4k_f32).  With
// fp16 operands a dot product's rounding error, relative to ||w_row|| ||x||,
// shrinks only as 1/sqrt(K): over 512 x 2048 outputs of seeded random data the
// largest error reached 1.7x the row bound 1e-4 ||w_row|| ||x|| at K = 256 and
// 0.97-1.05x at K = 512 (0.73 at 768, 0.70 at 1024, 0.30 at 4096), so short
// rows take this path, whose error is fp32 rounding.
//
// fp32 products run at a sixteenth of the matrix cores' bf16 rate, so the
// operands are written as bf16 without losing a bit:
//  * x = p1 + p2 + p3, its 24 significant bits cut into three bf16 values;
//  * the weights of a sub-block s as d sc q - dmin m
//    = (d sc / 2) (2 q - 15) + (7.5 d sc - dmin m), 2 q - 15 an odd integer
//    of -15 .. 15.  About the middle of the quants' range, so that the two
//    terms do not cancel where the weights centre on zero.
// Every bf16 product is exact.  A sub-block's sum over its 32 columns, three
// v_mfma_f32_32x32x16_bf16 for each 16 of them (smallest parts first),
// accumulates in fp32 from zero and one fp32 FMA per output scales it into the
// row's sum; the second term is an fp32 product (v_mfma_f32_32x32x2_f32) of
// the columns' sums and the mins, two sub-blocks at a time.
//
// Tile: 32 TT tokens x 64 weight rows per workgroup of 8 waves, which share K:
// wave (half, j) takes sub-block pair j of the blocks 2 i + half and
// accumulates the whole tile, so each value of X is cut up by one wave only
// and the waves run at their own pace: every wave copies its operands through
// LDS by itself (two X stages of 32 columns, its 48 bytes of the 64 rows'
// blocks), with no barrier before the eight partial tiles are added up in
// LDS, in wave order.  The vector work of a stage (cutting X 5.5 instructions
// a value, its sums and largest magnitude 1.5, the weights, the scaling) is
// about 1.5 times its matrix time and bounds it; the two waves of a SIMD
// overlap them.
//
// Measured on MI355X (us a call; the fp32 matrix products this replaced):
// 509 x 2048 x 2048 22.0 against 58.0, 512 x 4096 x 4096 80.8 against 186, 700 x
// 4096 x 4096 117 against 262, 100 x 2048 x 2048 12.1 against 55.4, 512 x 256 x
// 4096 13.7 against 14.9; error against 64 bits at 509 x 2048 x 2048 1.1e-7
// against 8.2e-7 (fewer roundings: 64 sums of 32 columns instead of 2048).
//
// The matrix cores take bf16 subnormals as zeros, and sums could overflow
// before a scale is applied or before the two terms cancel.  Each token's
// largest magnitude is found along the way; a tile with a token outside 2^-80 ..
// 2^76 is computed again on tokens scaled by powers of two, which is exact
// (below 2^76 no partial sum reaches 2^127: a scale and a quant are below 2^26,
// a row shorter than 2^24).  A token that holds an infinity has infinite or
// NaN outputs, which only the signs decide: +Inf where every infinity meets a
// weight of its own sign, -Inf where every one meets the other, NaN otherwise.
// A tile with such a token runs once more on the signs of the weights (1, 0,
// -1) and of the infinities (other values 0): its sums, whole numbers, are the
// number of the token's infinities, minus that, or neither.
// Measured (us a call; fp32 matrix products): 509 x 2048 x 2048 24.7 without an
// infinity, 42 with one, 44 with one in every token (62); 512 x 4096 x 4096 83,
// 148, 162 (210); 512 x 256 x 4096 14.5, 23.3, 24.3 (16.9).
constexpr int PFX_WSTAGE = 64 * 48; // header and the pair's 32 quant bytes of 64 rows
constexpr int PFX_LD = 72;          // floats per row of a partial tile
constexpr float kSplitMinX = 0x1p-80f, kSplitMaxX = 0x1p76f;
enum { kSplitPlain, kSplitScaled, kSplitSigns }; // what a pass over the tile multiplies
__host__ __device__ constexpr int pfx_wave_bytes(int tt) { return 2 * 4096 * tt + PFX_WSTAGE; }
static_assert(8 * pfx_wave_bytes(2) <= 160 * 1024 - 512, "the eight waves' stages fit the 160 KB of LDS");
static_assert(PFX_LD * 64 * 4 <= pfx_wave_bytes(2) && PFX_LD * 32 * 4 <= pfx_wave_bytes(1), "and the partial tiles");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// 8 nibbles (the low ones of the 8 bytes, already shifted down) -> 2 q - 15 in
// bf16.  The e4m3 byte whose low four bits are v is v * 2^-9 for every v of 0
// .. 15: v = |2 q - 15|, the sign on top.
__device__ __forceinline__ bf16x8 pfx_quants(uint2 bytes)
{
    auto code = [](uint32_t q) {
        const uint32_t neg = ~q & 0x08080808u;           // q < 8: 2 q - 15 = -(2 (7 - q) + 1)
        const uint32_t flip = neg - (neg >> 3);          // 7 where q < 8
        const uint32_t mag = (q ^ flip) & 0x07070707u;   // q - 8 or 7 - q
        return (mag << 1) | ((neg << 4) | 0x01010101u);
    };
    const uint32_t c0 = code(bytes.x), c1 = code(bytes.y);
    const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c0, 512.0f, false);
    const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c0, 512.0f, true);
    const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c1, 512.0f, false);
    const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c1, 512.0f, true);
    bf16x8 r;
    r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
    r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1];
    return r;
}

// 8 values of x -> their three bf16 parts (each the top half of what the
// parts before it leave, which is exact), their sum and largest magnitude.
__device__ __forceinline__ void pfx_parts(float4 lo, float4 hi, bf16x8 (&p)[3], float &sum, float &big)
{
    float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
    for (int i = 0; i < 8; i += 2)
        big = fmaxf(fmaxf(fabsf(v[i]), fabsf(v[i + 1])), big);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t a = __float_as_uint(v[2 * i]), b = __float_as_uint(v[2 * i + 1]);
            d[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
            v[2 * i] -= __uint_as_float(a & 0xffff0000u);
            v[2 * i + 1] -= __uint_as_float(b & 0xffff0000u);
        }
        p[k] = __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3]));
    }
}

// Signs of the weights d1 q - m1 of the same nibbles (NaN for NaN) in bf16.
// d1 q and m1 are exact in fp32, so the difference has the sign of the weight.
__device__ __forceinline__ bf16x8 pfx_signs(uint2 bytes, float d1, float m1)
{
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t s[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t q = ((i < 2 ? bytes.x : bytes.y) >> (16 * (i & 1) + 8 * k)) & 15u;
            const float v = d1 * (float)q - m1;
            s[k] = __float_as_uint(v > 0.0f ? 1.0f : v < 0.0f ? -1.0f : v);
        }
        d[i] = __builtin_amdgcn_perm(s[1], s[0], 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3]));
}

// 8 values of x -> 1 or -1 for the infinities among them, NaN for NaN, 0 for
// the rest; counts the infinities.
__device__ __forceinline__ bf16x8 pfx_infinities(float4 lo, float4 hi, int &count)
{
    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t s[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float x = v[2 * i + k];
            const bool inf = fabsf(x) == __builtin_inff();
            count += inf ? 1 : 0;
            s[k] = __float_as_uint(inf ? copysignf(1.0f, x) : x != x ? __builtin_nanf("") : 0.0f);
        }
        d[i] = __builtin_amdgcn_perm(s[1], s[0], 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3]));
}

// FAR: rows past kPrefillSplitMaxK columns, whose bytes 64 rows (32 tokens)
// away need 64-bit offsets.
template <int TT, bool FAR>
__global__ __launch_bounds__(512, 2) void k_prefill_q4k_split(const uint8_t *__restrict__ W,
                                                              const float *__restrict__ X,
                                                              float *__restrict__ Y, int T, int K, int N,
                                                              int mtiles, int ntiles)
{
    constexpr int XC = 4 * TT, XST = 4096 * TT, WAVE = pfx_wave_bytes(TT); // 1 KB copies and bytes of an X stage
    __shared__ __attribute__((aligned(16))) uint8_t lds[8 * WAVE];
    __shared__ uint32_t tokmax[32 * TT]; // the tokens' largest |x| (bits)
    __shared__ int tokinf[32 * TT];      // and their infinities
    using Offset = std::conditional_t<FAR, size_t, uint32_t>;
    auto copy16 = [](const uint8_t *base, Offset off, uint32_t dst) {
        if constexpr (FAR)
            lds_copy16(base + off, dst);
        else
            pf_copy16(base, off, dst);
    };

    const int tiles = mtiles * ntiles;
    const int lin = prefill_lin((int)blockIdx.x, tiles, 1);
    if (lin >= tiles)
        return; // whole workgroup
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, li = lane & 31, j = wave & 3, half = wave >> 2;
    const int nk = K / 256;
    const size_t row_bytes = (size_t)nk * 144;
    const PrefillSplit ps = prefill_split_of(lin, mtiles, ntiles, nk, 1);
    const int m0 = ps.mt * (32 * TT), n0 = ps.nt * 64;
    if (tid < 32 * TT) {
        tokmax[tid] = 0u;
        tokinf[tid] = 0;
    }
    __syncthreads();

    float16v acc[TT][2];
    float big[TT];
    int shift[TT], infs[TT];
    const int nb = (nk - half + 1) >> 1, ns = 2 * nb; // this wave's blocks and stages
    auto product = [&](auto mode) { // scaled: of the tokens times 2^shift
        constexpr bool SCALED = decltype(mode)::value == kSplitScaled, SIGNS = decltype(mode)::value == kSplitSigns;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            big[t] = 0.0f;
            infs[t] = 0;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.0f;
        }
        if (nb <= 0)
            return;
        // copies: 32 columns of X a stage, and 64 rows x 3 pieces of the blocks.
        // 32-bit offsets suffice: the launcher bounds K.  Rows past T or N
        // re-read the last one, stages past the last repeat it.
        Offset xo[XC], wo[3];
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const int m = pf_copy_token(i, lane);
            xo[i] = (Offset)min(m, T - 1 - m0) * ((Offset)K * 4u) + 16u * (uint32_t)pf_copy_chunk(m, lane);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const PfPiece q = pf_pair_piece(i, lane, j);
            wo[i] = (Offset)min(q.row, N - 1 - n0) * (Offset)row_bytes + q.off;
        }
        const uint8_t *Xb = reinterpret_cast<const uint8_t *>(X + (size_t)m0 * K + 256 * half + 64 * j);
        const uint8_t *Wb = W + (size_t)n0 * row_bytes + 144 * half;
        uint8_t *const mine = lds + WAVE * wave;
        const uint32_t xdst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mine;
        const uint32_t wdst = xdst + 2 * XST;
        auto issue_x = [&](int n) {
            const int st = min(n, ns - 1);
            const uint8_t *b = Xb + (size_t)(st >> 1) * 2048 + 128 * (st & 1);
#pragma unroll
            for (int i = 0; i < XC; ++i)
                copy16(b, xo[i], xdst + XST * (n & 1) + 1024 * i);
        };
        auto issue_w = [&](int i) {
            const uint8_t *b = Wb + (size_t)min(i, nb - 1) * 288;
#pragma unroll
            for (int k = 0; k < 3; ++k)
                copy16(b, wo[k], wdst + 1024 * k);
        };
        const uint8_t *wl = mine + 2 * XST + 48 * li;

        float4 xr[TT][2][2];
        uint2 qs[2][2];
        float ds[2][2], ndm[2], xsum[2][TT]; // [row tile or sub-block][..]
        float m1[SIGNS ? 2 : 1][2];
        auto read_x = [&](int s) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        xr[t][c][e] = *reinterpret_cast<const float4 *>(mine + XST * s + 4096 * t +
                                                                       pf_stage_at(li, 4 * c + 2 * h + e));
        };
        auto stage = [&](int s) {
            bf16x8 wq[2][2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const uint2 b = s ? make_uint2(qs[u][c].x >> 4, qs[u][c].y >> 4) : qs[u][c];
                    if constexpr (SIGNS)
                        wq[u][c] = pfx_signs(b, 2.0f * ds[u][s], m1[u][s]);
                    else
                        wq[u][c] = pfx_quants(b);
                }
            if constexpr (SIGNS) {
#pragma unroll
                for (int t = 0; t < TT; ++t)
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const bf16x8 p = pfx_infinities(xr[t][c][0], xr[t][c][1], infs[t]);
#pragma unroll
                        for (int u = 0; u < 2; ++u)
                            acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p, wq[u][c], acc[t][u], 0, 0, 0);
                    }
                return;
            }
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                bf16x8 p[2][3];
                xsum[s][t] = 0.0f;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if constexpr (SCALED) {
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            float4 &v = xr[t][c][e];
                            v = make_float4(__builtin_ldexpf(v.x, shift[t]), __builtin_ldexpf(v.y, shift[t]),
                                            __builtin_ldexpf(v.z, shift[t]), __builtin_ldexpf(v.w, shift[t]));
                        }
                    }
                    pfx_parts(xr[t][c][0], xr[t][c][1], p[c], xsum[s][t], big[t]);
                }
                float16v sub[2];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sub[u][r] = 0.0f;
#pragma unroll
                for (int k = 2; k >= 0; --k)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int u = 0; u < 2; ++u)
                            sub[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[c][k], wq[u][c], sub[u], 0, 0, 0);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[t][u][r] = fmaf(sub[u][r], ds[u][s], acc[t][u][r]);
            }
        };

        issue_w(0);
        issue_x(0);
        issue_x(1);
        for (int i = 0; i < nb; ++i) {
            __builtin_amdgcn_s_waitcnt(XC | 0x0f70); // all but the next stage's copies have landed
            asm volatile("" ::: "memory");
            uint4 hd[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                hd[u] = *reinterpret_cast<const uint4 *>(wl + 32 * 48 * u);
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    qs[u][c] = *reinterpret_cast<const uint2 *>(wl + 32 * 48 * u + 16 + 16 * c + 8 * h);
            }
            read_x(0);
            __builtin_amdgcn_s_waitcnt(0xc07f); // and are in registers: their place is free
            asm volatile("" ::: "memory");
            issue_x(2 * i + 2);
            issue_w(i + 1);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const float d = h2f(hd[u].x & 0xffffu), dmin = h2f(hd[u].x >> 16);
                float scA, mA, scB, mB;
                k_scale_min_pair(hd[u].y, hd[u].z, hd[u].w, j, scA, mA, scB, mB);
                ds[u][0] = 0.5f * d * scA;
                ds[u][1] = 0.5f * d * scB;
                // this lane half's sub-block of the pair
                ndm[u] = fmaf(15.0f, h ? ds[u][1] : ds[u][0], -(dmin * (h ? mB : mA)));
                if constexpr (SIGNS) {
                    m1[u][0] = dmin * mA;
                    m1[u][1] = dmin * mB;
                }
            }
            stage(0);
            __builtin_amdgcn_s_waitcnt((XC + 3) | 0x0f70);
            asm volatile("" ::: "memory");
            read_x(1);
            __builtin_amdgcn_s_waitcnt(0xc07f);
            asm volatile("" ::: "memory");
            issue_x(2 * i + 3);
            stage(1);
            if constexpr (SIGNS)
                continue;
            // lane (li, h): token li's sum over the pair's sub-block h
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const auto x2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(xsum[0][t]),
                                                                 __float_as_uint(xsum[1][t]), false, false);
                const float both = __uint_as_float((uint32_t)x2[0]) + __uint_as_float((uint32_t)x2[1]);
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(both, ndm[u], acc[t][u], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0070); // the last (unused) copies have landed
    };
    product(std::integral_constant<int, kSplitPlain>{});
#pragma unroll
    for (int t = 0; t < TT; ++t)
        atomicMax(&tokmax[32 * t + li], __float_as_uint(big[t]));
    __syncthreads();
    // a token's power of two: its largest magnitude to [0.5, 1)
    auto shift_of = [&](int m) {
        const float b = __uint_as_float(tokmax[m]);
        return b > 0.0f && b < __builtin_inff() ? -__builtin_amdgcn_frexp_expf(b) : 0;
    };
    bool out_of_range = false, infinite = false;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const float b = __uint_as_float(tokmax[32 * t + li]);
        infinite |= b == __builtin_inff();
        out_of_range |= (b > 0.0f && b < kSplitMinX) || (b >= kSplitMaxX && b < __builtin_inff());
        shift[t] = shift_of(32 * t + li);
    }
    const bool again = __ballot(out_of_range) != 0; // the same in every wave
    if (again) {
        product(std::integral_constant<int, kSplitScaled>{});
        __syncthreads();
    }
    // Y of the tokens with (inf) or without an infinity from the waves' partial
    // tiles.  Lane (li, h), register r of acc[t][u]: token 32 t + 8 (r / 4) + 4 h
    // + r % 4, row 32 u + li.
    float *const P = reinterpret_cast<float *>(lds);
    auto write = [&](bool inf) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    P[(32 * TT * wave + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3)) * PFX_LD + 32 * u + li] = acc[t][u][r];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < TT; ++p) {
            const int ml = 32 * p + (tid >> 4), nl = 4 * (tid & 15), m = m0 + ml, n = n0 + nl;
            if (m >= T || n >= N || (tokmax[ml] == 0x7f800000u) != inf)
                continue;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < 8; ++w) {
                const float4 q = *reinterpret_cast<const float4 *>(P + (32 * TT * w + ml) * PFX_LD + nl);
                v.x += q.x;
                v.y += q.y;
                v.z += q.z;
                v.w += q.w;
            }
            if (inf) {
                const float k = (float)tokinf[ml];
                auto sign = [&](float a) { return a == k ? __builtin_inff() : a == -k ? -__builtin_inff() : __builtin_nanf(""); };
                v = make_float4(sign(v.x), sign(v.y), sign(v.z), sign(v.w));
            } else {
                const int sm = again ? -shift_of(ml) : 0;
                v = make_float4(__builtin_ldexpf(v.x, sm), __builtin_ldexpf(v.y, sm), __builtin_ldexpf(v.z, sm),
                                __builtin_ldexpf(v.w, sm));
            }
            float *y = Y + (size_t)m * (size_t)N + n;
            if ((N & 3) == 0) {
                *reinterpret_cast<float4 *>(y) = v;
            } else {
                y[0] = v.x;
                if (n + 1 < N) y[1] = v.y;
                if (n + 2 < N) y[2] = v.z;
                if (n + 3 < N) y[3] = v.w;
            }
        }
    };
    write(false);
    if (__ballot(infinite) != 0) { // the same in every wave
        __syncthreads();
        product(std::integral_constant<int, kSplitSigns>{});
#pragma unroll
        for (int t = 0; t < TT; ++t)
            atomicAdd(&tokinf[32 * t + li], infs[t]);
        __syncthreads();
        write(true);
    }
}

hipError_t launch_prefill_q4k_f32(const void *w, const float *X, float *Y, int T, int inner,
                                  int outer, hipStream_t s)
{
    if (T <= 0 || outer <= 0 || inner <= 0 || inner % 256 || (int64_t)T * outer > (int64_t)INT32_MAX)
        return hipErrorInvalidValue;
    const int tt = inner > kPrefillSplitMaxK ? 1 : prefill_split_tokens(T, outer, device_cus()) / 32;
    const int mtiles = (T + 32 * tt - 1) / (32 * tt), ntiles = (outer + 63) / 64;
    const dim3 grid(prefill_grid(mtiles * ntiles, 1)), block(512);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, (const uint8_t *)w, X, Y, T, inner, outer, mtiles, ntiles);
    };
    if (inner > kPrefillSplitMaxK)
        launch(k_prefill_q4k_split<1, true>);
    else if (tt == 1)
        launch(k_prefill_q4k_split<1, false>);
    else
        launch(k_prefill_q4k_split<2, false>);
    return hipGetLastError();
}

hipError_t launch_prefill_convert(const float *X, void *xh, int T, int inner, hipStream_t s)
{
    if (T <= 0 || inner <= 0 || inner % 256)
        return hipErrorInvalidValue;
    int *xs = reinterpret_cast<int *>(static_cast<uint8_t *>(xh) + prefill_scale_offset(T, inner));
    hipLaunchKernelGGL(k_x_to_f16, dim3((unsigned)T), dim3(256), 0, s, X, (_Float16 *)xh, xs, inner);
    return hipGetLastError();
}

hipError_t launch_prefill_q4k(const void *w, const float *X, void *xh, float *Y, int T,
                              int inner, int outer, hipStream_t s)
{
    if (T <= 0 || inner % 256 || !prefill_fits(T, inner, outer))
        return hipErrorInvalidValue;
    if (inner <= kPrefillF32MaxK)
        return launch_prefill_q4k_f32(w, X, Y, T, inner, outer, s);
    const hipError_t e = launch_prefill_convert(X, xh, T, inner, s);
    if (e != hipSuccess)
        return e;
    return launch_prefill_gemm(w, xh, Y, T, inner, outer, s);
}

template <int RU>
static void launch_prefill_wide(const void *w, const void *xh, const int *xs, float *Y, int T, int inner,
                                int outer, hipStream_t s)
{
    const int mtiles = (T + kPrefillWideBM - 1) / kPrefillWideBM;
    const int ntiles = (outer + 128 * RU - 1) / (128 * RU);
    const dim3 grid(prefill_grid(mtiles * ntiles, 1)), block(256);
    if (inner <= kPrefillExactWMaxK)
        hipLaunchKernelGGL((k_prefill_q4k_wide<true, RU>), grid, block, 0, s, (const uint8_t *)w,
                           (const _Float16 *)xh, xs, Y, T, inner, outer, mtiles, ntiles);
    else
        hipLaunchKernelGGL((k_prefill_q4k_wide<false, RU>), grid, block, 0, s, (const uint8_t *)w,
                           (const _Float16 *)xh, xs, Y, T, inner, outer, mtiles, ntiles);
}

hipError_t launch_prefill_gemm(const void *w, void *xh, float *Y, int T, int inner, int outer,
                               hipStream_t s)
{
    if (T <= 0 || inner <= kPrefillF32MaxK || inner % 256 || !prefill_fits(T, inner, outer))
        return hipErrorInvalidValue;
    int *xs = reinterpret_cast<int *>(static_cast<uint8_t *>(xh) + prefill_scale_offset(T, inner));
    float *P = reinterpret_cast<float *>(static_cast<uint8_t *>(xh) + prefill_part_offset(T, inner));
    if (prefill_thin(T, inner, outer, device_cus())) {
        const int mt = (T + PFT_BM - 1) / PFT_BM, nt = (outer + PFT_BN - 1) / PFT_BN;
        const dim3 grid(prefill_grid(mt * nt, 1)), block(512);
        if (inner <= kPrefillExactWMaxK)
            hipLaunchKernelGGL(k_prefill_q4k_thin<true>, grid, block, 0, s, (const uint8_t *)w, (const _Float16 *)xh,
                               (const int *)xs, Y, T, inner, outer, mt, nt);
        else
            hipLaunchKernelGGL(k_prefill_q4k_thin<false>, grid, block, 0, s, (const uint8_t *)w, (const _Float16 *)xh,
                               (const int *)xs, Y, T, inner, outer, mt, nt);
        return hipGetLastError();
    }
    const int ru = prefill_wide_rows(T, inner, outer, device_cus());
    if (ru) {
        if (ru == 2)
            launch_prefill_wide<2>(w, xh, xs, Y, T, inner, outer, s);
        else
            launch_prefill_wide<1>(w, xh, xs, Y, T, inner, outer, s);
        return hipGetLastError();
    }
    const int mtiles = (T + PF_BM - 1) / PF_BM, ntiles = (outer + PF_BN - 1) / PF_BN;
    const int nsplit = prefill_splits(T, inner, outer, device_cus());
    const dim3 grid(prefill_grid(mtiles * ntiles, nsplit));
    if (inner <= kPrefillExactWMaxK)
        hipLaunchKernelGGL(k_prefill_q4k<true>, grid, dim3(PF_THREADS), 0, s, (const uint8_t *)w,
                           (const _Float16 *)xh, (const int *)xs, Y, P, T, inner, outer, mtiles, ntiles, nsplit);
    else
        hipLaunchKernelGGL(k_prefill_q4k<false>, grid, dim3(PF_THREADS), 0, s, (const uint8_t *)w,
                           (const _Float16 *)xh, (const int *)xs, Y, P, T, inner, outer, mtiles, ntiles, nsplit);
    if (nsplit > 1) {
        const int64_t n = (int64_t)T * outer;
        const int64_t units = (n & 3) == 0 ? n >> 2 : n;
        const unsigned grid = (unsigned)std::min<int64_t>((units + 255) / 256, 2048);
        if ((n & 3) == 0)
            hipLaunchKernelGGL(k_prefill_splits_sum<true>, dim3(grid), dim3(256), 0, s, Y,
                               (const float *)P, n, nsplit - 1);
        else
            hipLaunchKernelGGL(k_prefill_splits_sum<false>, dim3(grid), dim3(256), 0, s, Y,
                               (const float *)P, n, nsplit - 1);
    }
    return hipGetLastError();
}

} // namespace ihip
