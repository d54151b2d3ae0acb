// mdig_check.hip -- host-side bounds and coverage check of the matrix-core
// GEMV launch (k_gemv_mdig in inferno.jl_amd/csrc/kq_gemv.hip).
//
// Test infrastructure, run on the CPU only: it launches nothing.  It includes
// the header the launcher and the kernel take the launch and the copies' offsets
// from (kq_gemv_plan.h) and walks workgroups of a launch (all of a small one, the
// first, middle and last ones of a large one), every wave, unit, copy and lane,
// asserting that
//   * every (row group, matrix, step) is one unit of one workgroup, its place
//     among the row sums inside the array, and the divisions by nstep exact;
//   * the copies of x cover the row and stay inside it, and with the units
//     issued ahead of them stay in different slots of the wave's ring;
//   * every weight copy reads whole 16-byte units inside W or the unit holding
//     its last byte, lands in its slot, and the bytes of every block that a lane
//     uses lie in the slot where the lane reads them;
//   * what a lane reads beyond its block stays inside the wave's ring;
//   * the vmcnt waits allow no more copies in flight than were issued after the
//     ones they guard, and fit the instruction's four low bits.
//
// Built by inferno_hip.build into tests/native/_build/libsdig_check.so; called
// from tests/test_gemv_plan.py through ctypes.
#include "kq_gemv_plan.h"
#include "kq_launch.h"

#include <cstdarg>
#include <cstdio>
#include <vector>

using namespace ihip;

namespace {

struct MReport {
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

template <int FMT>
void walk(MReport &R, int nblk, int outer, bool gateup, bool norm, int ncu, uint64_t w_at, long long *stats)
{
    using F = MdFmt<FMT>;
    constexpr int BPS = F::BLOCKS, LP = F::PITCH, PP = F::PIECES, NC = F::COPIES, SLOT = 1024 * NC;
    const int inner = nblk * (1024 / BPS), nstep = (nblk + BPS - 1) / BPS, NM = gateup ? 2 : 1;
    const int ngroups = (outer + 3) / 4, gpw = mdig_groups(outer, nstep * NM, ncu), grid = (ngroups + gpw - 1) / gpw;
    const MdPlan p = mdig_plan(FMT, nstep, gpw);
    const int NWV = p.nw, D = p.d, NT = NWV * 64;
    const uint32_t inv = md_inv(nstep);
    const uint64_t row_bytes = (uint64_t)nblk * F::BYTES, w_end = (w_at + (uint64_t)outer * row_bytes + 15) / 16 * 16;
    stats[0] = grid;
    stats[1] = gpw;
    stats[2] = NWV;
    stats[3] = D;
    if (nstep > p.maxs || nstep > kMdMaxSteps)
        R.fail("%d steps, the instantiation takes %d", nstep, p.maxs);
    if (gpw < 1 || gpw * NM * nstep > kMdUnits)
        R.fail("%d groups x %d x %d steps are more units than %d", gpw, NM, nstep, kMdUnits);
    if (4 * LP > 64 * NC || D > 3 || 3 * NC > 15)
        R.fail("a slot or a wait does not fit");
    for (int a = 0; a <= 16; ++a)
        if (md_div(a, inv) != a / nstep)
            R.fail("%d / %d gives %d", a, nstep, md_div(a, inv));
    const int NX = (p.maxs * 256 + NT - 1) / NT, XC = md_x_chunk(NX, D, NC, norm);
    // x: every 16 bytes of the row by the thread that converts them
    for (int w = 0; w < NWV; ++w) {
        const int nx = md_x_copies(inner, w, NT);
        if (nx < 0 || nx > NX)
            R.fail("wave %d: %d copies of x, %d converted", w, nx, NX);
        for (int k = 0; k < nx; ++k)
            for (int l = 0; l < 64; ++l) {
                const int tid = 64 * w + l;
                const long long at = 16LL * NT * k + md_x_off(inner, tid, NT, k);
                if (at < 0 || at % 16 || at + 16 > 4LL * inner)
                    R.fail("wave %d copy %d lane %d: bytes %lld.. of %d columns", w, k, l, at, inner);
                if (4LL * (tid + (long long)NT * k) < inner && at != 16LL * (tid + (long long)NT * k))
                    R.fail("wave %d copy %d lane %d: not its own values", w, k, l);
            }
        for (int f = w * 64; f < inner / 4; f += NT) // the wave's float4s are within its copies
            if ((f - w * 64) / NT >= nx)
                R.fail("wave %d: values %d.. are not copied", w, 4 * f);
    }
    std::vector<int> seen((size_t)ngroups * NM * nstep, 0);
    for (int bid = 0; bid < grid && R.n < 20; ++bid) {
        const int G0 = bid * gpw, ng = std::min(gpw, ngroups - G0), units = ng * NM * nstep;
        for (int w = 0; w < NWV; ++w) { // which units
            const int n = md_wave_units(units, w, NWV), qn = md_div(NWV, inv), rn = NWV - qn * nstep;
            int vg = md_div(w, inv), s = w - vg * nstep;
            for (int i = 0; i < n; ++i) {
                const int u = w + NWV * i;
                if (u != vg * nstep + s || s >= nstep || vg >= ng * NM)
                    R.fail("wg %d wave %d unit %d: cursor at %d, step %d", bid, w, i, vg, s);
                else
                    seen[((size_t)(G0 + vg / NM) * NM + vg % NM) * nstep + s]++;
                vg += qn;
                s += rn;
                if (s >= nstep) {
                    s -= nstep;
                    ++vg;
                }
            }
        }
        if (grid > 48 && bid >= 16 && bid < grid - 16 && (bid < grid / 2 || bid >= grid / 2 + 8))
            continue; // the copies: first, middle and last workgroups
        for (int w = 0; w < NWV; ++w) {
            const int n = md_wave_units(units, w, NWV);
            const int nx = md_x_copies(inner, w, NT), xc = std::min(nx, XC), raw = md_raw_slots(xc, norm, NC);
            const int pre = std::max(0, std::min(n, D - raw));
            if (raw > D || ((norm ? 2 : 1) * xc) * 1024 > raw * SLOT)
                R.fail("wave %d: %d copies of x in %d of %d slots", w, xc, raw, D);
            if (nx > xc && pre > 0)
                R.fail("wave %d: x comes in parts over slots that hold weights", w);
            if (pre > 2)
                R.fail("wave %d: %d units ahead of x", w, pre); // slots 0 .. pre - 1, the raw ones are the last
            for (int i = 0; i < n; ++i) {
                const int later = std::min(D, n - i) - 1, issued = std::min(n, i + D) - 1 - i;
                if (later > issued)
                    R.fail("wave %d unit %d: waits for all but %d units, %d issued after it", w, i, later, issued);
                const int u = w + NWV * i, vg = u / nstep, s = u % nstep, row0 = 4 * (G0 + vg / NM);
                // the kernel's issue()
                const uint64_t base0 = w_at + (uint64_t)row0 * row_bytes + (uint64_t)s * (BPS * F::BYTES);
                const uint32_t rmax = (uint32_t)(std::min(outer - row0, 4) - 1) * (uint32_t)row_bytes;
                const uint32_t nbytes = (uint32_t)std::min(nblk - BPS * s, BPS) * F::BYTES;
                const uint32_t phase = F::PHASED ? (uint32_t)base0 & 15u : 0u;
                if (!F::PHASED && (base0 & 15u))
                    R.fail("wg %d wave %d: step at byte phase %u", bid, w, (unsigned)(base0 & 15u));
                std::vector<int64_t> image(SLOT, -1);
                for (int c = 0; c < NC; ++c)
                    for (int l = 0; l < 64; ++l) {
                        const int q = 64 * c + l, row = md_piece_row(q, LP);
                        const uint32_t o = md_copy_off<F::PHASED>(std::min((uint32_t)row * (uint32_t)row_bytes, rmax),
                                                                  md_piece_off(q, row, LP, PP), nbytes, phase);
                        const uint64_t src = base0 - phase + o;
                        if (src % 16 || src < w_at || src + 16 > w_end)
                            R.fail("wg %d wave %d unit %d copy %d lane %d: W bytes %lld.. of %lld", bid, w, i, c, l,
                                   (long long)(src - w_at), (long long)(w_end - w_at));
                        for (int b = 0; b < 16; ++b) image[1024 * c + 16 * l + b] = (int64_t)src + b;
                        stats[4]++;
                    }
                for (int l = 0; l < 64; ++l) { // the kernel's reads: lane 4 b + r
                    const int b = l >> 2, r = l & 3, first = BPS == 32 ? 2 * b : b >> 2;
                    const int row = row0 + std::min(r, outer - 1 - row0);
                    const uint64_t step = w_at + (uint64_t)row * row_bytes + (uint64_t)s * (BPS * F::BYTES);
                    const uint32_t slot_row = (uint32_t)r * (LP * 16), ph = F::PHASED ? (uint32_t)step & 15u : 0u;
                    for (int k = 0; k < (BPS == 32 ? 2 : 1); ++k) {
                        const int blk = first + k;
                        const uint32_t at = slot_row + ph + (uint32_t)blk * F::BYTES;
                        // past the block's last byte: up to a dword of the next
                        if (at + F::BYTES + 4 > (uint32_t)SLOT)
                            R.fail("lane %d block %d: reads to byte %u of a slot of %d", l, blk, at + F::BYTES + 4, SLOT);
                        if (BPS * s + blk >= nblk)
                            continue; // not part of the row: unused
                        for (int x = 0; x < F::BYTES; ++x)
                            if (image[at + x] != (int64_t)(step + (uint64_t)blk * F::BYTES + x)) {
                                R.fail("wg %d wave %d unit %d row %d block %d byte %d: not in the slot", bid, w, i, row, blk, x);
                                break;
                            }
                    }
                }
            }
        }
    }
    for (size_t i = 0; i < seen.size(); ++i)
        if (seen[i] != 1) {
            R.fail("unit %zu is computed %d times", i, seen[i]);
            break;
        }
}

} // namespace

// Returns the number of violations (0: the launch is clean); msg receives the
// first.  stats: workgroups,
// groups per workgroup, waves, ring slots, copies checked.
extern "C" long long mdig_check(int type, int nblk, int outer, int gateup, int norm, int ncu, char *msg, int cap,
                                long long *stats)
{
    MReport R{msg, cap};
    if (msg && cap > 0)
        msg[0] = 0;
    if (nblk < 1 || outer < 1) {
        R.fail("bad shape");
        return R.n;
    }
    const uint64_t at = 1u << 20;
    switch (type) {
    case kQ4_K: walk<kQ4_K>(R, nblk, outer, gateup, norm, ncu, at, stats); break;
    case kQ5_K: walk<kQ5_K>(R, nblk, outer, gateup, norm, ncu, at, stats); break;
    case kQ6_K: walk<kQ6_K>(R, nblk, outer, gateup, norm, ncu, at, stats); break;
    case kQ8_0: walk<kQ8_0>(R, nblk, outer, gateup, norm, ncu, at, stats); break;
    case kIQ4_NL: walk<kIQ4_NL>(R, nblk, outer, gateup, norm, ncu, at, stats); break;
    default: R.fail("unknown type %d", type);
    }
    return R.n;
}

// k_gemv_q8k6 (kq_q8k.hip): every row has a team and every item of a row one of
// its waves, the copies read whole units inside W or the unit holding its last
// byte, the bytes of each block lie in the slot where the lanes read them, and a
// lane's dwords past its block stay in the slot.
extern "C" long long q8k6_check(int nb, int outer, int ncu, char *msg, int cap)
{
    MReport R{msg, cap};
    if (msg && cap > 0)
        msg[0] = 0;
    const int tw = q86_team(nb, outer, ncu), teams = kQ86Waves / tw, grid = (outer + teams - 1) / teams, ni = (nb + 7) / 8;
    if (nb < 1 || nb > kQ86MaxBlocks || outer < 1 || outer > ncu * kQ86Waves || grid > ncu)
        R.fail("%d rows of %d blocks: %d workgroups", outer, nb, grid);
    std::vector<int> items((size_t)ni, 0);
    for (int rank = 0; rank < tw; ++rank) {
        const int n = (ni - rank + tw - 1) / tw;
        if (n > kQ86Items)
            R.fail("%d items for a wave", n);
        for (int i = 0; i < n; ++i)
            if (rank + tw * i >= ni)
                R.fail("item %d of %d", rank + tw * i, ni);
            else
                items[(size_t)(rank + tw * i)]++;
    }
    for (int i = 0; i < ni; ++i)
        if (items[(size_t)i] != 1)
            R.fail("item %d is computed %d times", i, items[(size_t)i]);
    const int64_t row_bytes = (int64_t)nb * 210, w_end = ((int64_t)outer * row_bytes + 15) / 16 * 16;
    for (int row = 0; row < outer && R.n < 20; ++row)
        for (int it = 0; it < ni; ++it) {
            const int64_t at = row * row_bytes + it * 1680; // W itself is 16-byte aligned
            const uint32_t phase = (uint32_t)(at & 15);
            const int blocks = std::min(8, nb - 8 * it);
            if (phase != (uint32_t)(row * row_bytes & 15))
                R.fail("row %d item %d: not at its row's phase", row, it);
            std::vector<int64_t> image(kQ86Slot, -1);
            for (int i = 0; i < 2; ++i)
                for (int l = 0; l < 64; ++l) {
                    const int64_t src = at - phase + q86_copy_off(i, l, phase, blocks);
                    if (src < 0 || src % 16 || src + 16 > w_end)
                        R.fail("row %d item %d: bytes %lld.. of %lld", row, it, (long long)src, (long long)w_end);
                    for (int b = 0; b < 16; ++b) image[(size_t)(1024 * i + 16 * l + b)] = src + b;
                }
            if (phase + 7 * 210 + 4 * 54 > (uint32_t)kQ86Slot)
                R.fail("the last block's dwords leave the slot");
            for (int s = 0; s < blocks; ++s)
                for (int b = 0; b < 210; ++b)
                    if (image[phase + 210u * (uint32_t)s + (uint32_t)b] != at + 210 * s + b)
                        R.fail("row %d item %d block %d byte %d: not in the slot", row, it, s, b);
        }
    return R.n;
}
