// prefill_copy_check.hip -- host-side check of the direct-to-LDS copies of three
// prefill kernels (k_prefill_q4k_wide, _thin and _split in
// inferno.jl_amd/csrc/kq_prefill.hip).
//
// Test infrastructure, run on the CPU only: it launches nothing.  It forms the
// copies' offsets and the LDS reads with the kernels' functions (kq_launch.h) and
// asserts, for the first, a middle and the last tile each way, every wave, the
// first and the last stages, every copy and lane, that
//   * each copy reads 16 bytes inside the activations or W, 16-byte aligned;
//   * it lands inside the wave's own part of LDS;
//   * what a lane then reads is the token's or row's bytes that its step of the
//     product stands for (rows past the last: the last one's).
//
// Built by inferno_hip.build into tests/native/_build/libsdig_check.so; called
// from tests/test_prefill_plan.py through ctypes.
#include "kq_launch.h"

#include <cstdarg>
#include <cstdio>
#include <set>
#include <vector>

using namespace ihip;

namespace {

struct CReport {
    char *msg;
    int cap;
    long long n = 0;
    void fail(const char *fmt, ...)
    {
        if (n++ == 0 && msg && cap > 0) {
            va_list ap;
            va_start(ap, fmt);
            vsnprintf(msg, (size_t)cap, fmt, ap);
            va_end(ap);
        }
    }
};

// LDS bytes -> the byte of the operand they hold
struct Image {
    std::vector<int64_t> at;
    explicit Image(int bytes) : at((size_t)bytes, -1) {}
    void copy(CReport &R, const char *what, int64_t src, int64_t end, uint32_t dst)
    {
        if (src < 0 || src % 16 || src + 16 > end)
            R.fail("%s: bytes %lld.. of %lld", what, (long long)src, (long long)end);
        if (dst % 16 || dst + 16 > at.size()) {
            R.fail("%s: lands at %u of %zu", what, dst, at.size());
            return;
        }
        for (int b = 0; b < 16; ++b) at[dst + b] = src + b;
    }
    void expect(CReport &R, const char *what, uint32_t lds, int64_t want, int bytes)
    {
        for (int b = 0; b < bytes; ++b)
            if (lds + b >= at.size() || at[lds + b] != want + b) {
                R.fail("%s: LDS byte %u holds %lld, not %lld", what, lds + b,
                       lds + b < at.size() ? (long long)at[lds + b] : -2LL, (long long)(want + b));
                return;
            }
    }
};

std::set<int> some(int n) { return {0, n / 2, n - 1}; }

} // namespace

// kind: 0 the wide kernel (size: RU), 1 the thin one, 2 the split one (size: TT).
// Returns the number of violations; msg receives the first.
extern "C" long long prefill_copy_check(int kind, int size, int T, int K, int N, char *msg, int cap)
{
    CReport R{msg, cap};
    if (msg && cap > 0)
        msg[0] = 0;
    const int64_t nk = K / 256, row_bytes = nk * 144, w_end = N * row_bytes;
    if (kind == 0) {
        const int RU = size, WB = (32 * RU * 144 + 1023) / 1024, BM = kPrefillWideBM;
        for (int mt : some((T + BM - 1) / BM))
            for (int nt : some((N + 128 * RU - 1) / (128 * RU))) {
                const int m0 = mt * BM;
                for (int64_t kb : {(int64_t)0, nk - 1})
                    for (int g = 0; g < 4; ++g) {
                        const int64_t st = 4 * kb + g;
                        Image x(BM * 128); // the workgroup's stage
                        for (int wave = 0; wave < 4; ++wave)
                            for (int i = 0; i < 4; ++i)
                                for (int l = 0; l < 64; ++l) {
                                    const int m = 32 * wave + pf_copy_token(i, l);
                                    x.copy(R, "wide X", st * 128 + 2 * (int64_t)std::min(m0 + m, T - 1) * K + 16 * pf_copy_chunk(m, l),
                                           2 * (int64_t)T * K, 4096u * wave + 1024u * i + 16u * l);
                                }
                        for (int l = 0; l < 64; ++l)
                            for (int t = 0; t < BM / 32; ++t)
                                for (int c = 0; c < 4; ++c) {
                                    const int li = l & 31, h = l >> 5;
                                    x.expect(R, "wide X", pf_stage_at(li, 4 * h + c) + 4096u * t,
                                             2 * (int64_t)std::min(m0 + 32 * t + li, T - 1) * K + 512 * kb +
                                                 16 * pf_chunk_place(16 * h + 4 * g + c), 16);
                                }
                    }
                for (int wave = 0; wave < 4; ++wave)
                    for (int64_t kb : {(int64_t)0, nk - 1}) {
                        const int n0 = nt * 128 * RU + 32 * RU * wave;
                        Image w(1024 * WB);
                        for (int i = 0; i < WB; ++i)
                            for (int l = 0; l < 64; ++l) {
                                const PfPiece q = pf_block_piece(i, l, 32 * RU);
                                w.copy(R, "wide W", kb * 144 + std::min(n0 + q.row, N - 1) * row_bytes + q.off, w_end,
                                       1024u * i + 16u * l);
                            }
                        for (int r = 0; r < 32 * RU; ++r)
                            w.expect(R, "wide W", 144u * r, std::min(n0 + r, N - 1) * row_bytes + kb * 144, 144);
                    }
            }
        return R.n;
    }
    // thin: 32 tokens x 64 rows; split: 32 TT tokens x 64 rows, fp32
    const int BM = kind == 1 ? kPrefillThinBM : 32 * size, XC = BM / 8, elem = kind == 1 ? 2 : 4;
    for (int mt : some((T + BM - 1) / BM))
        for (int nt : some((N + 63) / 64))
            for (int wave = 0; wave < 8; ++wave) {
                const int j = wave & 3, half = wave >> 2, m0 = mt * BM, n0 = nt * 64;
                const int64_t nb = (nk - half + 1) >> 1;
                for (int64_t i : {(int64_t)0, nb - 1}) {
                    if (nb <= 0)
                        continue;
                    const int64_t kb = 2 * i + half;
                    Image w(48 * 64);
                    for (int k = 0; k < 3; ++k)
                        for (int l = 0; l < 64; ++l) {
                            const PfPiece q = pf_pair_piece(k, l, j);
                            w.copy(R, "pair W", 144 * half + 288 * i + std::min(n0 + q.row, N - 1) * row_bytes + q.off, w_end,
                                   1024u * k + 16u * l);
                        }
                    for (int r = 0; r < 64; ++r) {
                        const int64_t blk = std::min(n0 + r, N - 1) * row_bytes + 144 * kb;
                        w.expect(R, "pair header", 48u * r, blk, 16);
                        w.expect(R, "pair quants", 48u * r + 16u, blk + 16 + 32 * j, 32);
                    }
                    for (int s = 0; s < (kind == 1 ? 1 : 2); ++s) { // stages
                        Image x(BM * 128);
                        for (int c = 0; c < XC; ++c)
                            for (int l = 0; l < 64; ++l) {
                                const int m = pf_copy_token(c, l), e = pf_copy_chunk(m, l);
                                const int64_t row = (int64_t)std::min(m0 + m, T - 1) * K * elem;
                                x.copy(R, "X", row + (kind == 1 ? 512 * half + 1024 * i + 16 * pf_chunk_place(8 * j + e)
                                                                : 4 * (256 * half + 64 * j) + 2048 * i + 128 * s + 16 * e),
                                       (int64_t)T * K * elem, 1024u * c + 16u * l);
                            }
                        for (int l = 0; l < 64; ++l)
                            for (int t = 0; t < BM / 32; ++t)
                                for (int c = 0; c < (kind == 1 ? 4 : 2); ++c)
                                    for (int e = 0; e < (kind == 1 ? 1 : 2); ++e) {
                                        const int li = l & 31, h = l >> 5;
                                        const int64_t row = (int64_t)std::min(m0 + 32 * t + li, T - 1) * K * elem;
                                        if (kind == 1)
                                            x.expect(R, "thin X", pf_stage_at(li, 2 * c + h),
                                                     row + 512 * kb + 16 * pf_chunk_place(8 * j + 2 * c + h), 16);
                                        else
                                            x.expect(R, "split X", 4096u * t + pf_stage_at(li, 4 * c + 2 * h + e),
                                                     row + 4 * (256 * kb + 64 * j + 32 * s + 16 * c + 8 * h + 4 * e), 16);
                                    }
                    }
                }
            }
    return R.n;
}
