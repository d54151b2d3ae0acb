"""Which kernel takes a GEMV (kq_gemv_plan.h, through tests/native/
gemv_plan_check.hip, on the CPU): the faster one at shapes where the two were
timed 4 % apart or more, and on the GPU both kernels' results at the edges of
the rules.  And every copy, slot and wait of k_gemv_mdig's launches, walked on
the CPU through the kernel's own index functions (tests/native/mdig_check.hip).
"""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest

import oracle
from inferno_hip import synth

LIB = Path(__file__).resolve().parent / "native" / "_build" / "libsdig_check.so"
Q4_K, Q5_K, Q6_K = synth.Q4_K, synth.Q5_K, synth.Q6_K


@pytest.fixture(scope="module")
def plan():
    if not LIB.exists():
        from inferno_hip import build
        build.build_checks()
    return C.CDLL(str(LIB))


# (type, rows, columns, wide us, k_gemv_mdig us): graph replays, weights in HBM
NORM_TIMES = (
    (Q4_K, 256, 1536, 2.71, 3.01), (Q4_K, 1024, 2560, 3.04, 3.37), (Q4_K, 1024, 4096, 3.41, 3.82),
    (Q4_K, 2048, 2048, 3.05, 3.34), (Q4_K, 2048, 4096, 4.08, 4.47), (Q4_K, 2304, 1024, 3.59, 3.20),
    (Q4_K, 3072, 2304, 3.78, 4.12), (Q4_K, 4096, 3328, 4.34, 4.99), (Q4_K, 4096, 4096, 4.49, 5.14),
    (Q4_K, 6144, 1536, 5.17, 4.14), (Q4_K, 6144, 4096, 6.45, 5.80), (Q4_K, 8192, 3584, 5.51, 6.25),
    (Q4_K, 12288, 2560, 6.68, 6.20), (Q4_K, 12288, 4096, 7.22, 8.12), (Q4_K, 16384, 1024, 7.46, 4.74),
    (Q5_K, 512, 3584, 3.54, 3.88), (Q5_K, 1024, 1024, 3.30, 3.10), (Q5_K, 1536, 2560, 3.46, 3.79),
    (Q5_K, 1024, 4096, 3.78, 4.01), (Q5_K, 2304, 3072, 4.60, 4.33), (Q5_K, 4096, 3328, 4.93, 5.22),
    (Q5_K, 6144, 4096, 7.27, 6.38), (Q5_K, 8192, 2304, 6.33, 5.72), (Q5_K, 12288, 3584, 8.29, 8.79),
    (Q5_K, 16384, 4096, 10.71, 11.44))


@pytest.mark.parametrize("t,outer,inner,wide,mdig", NORM_TIMES)
def test_folded_norm_takes_the_faster_kernel(plan, t, outer, inner, wide, mdig):
    assert bool(plan.norm_takes_wide_of(t, inner // 256, outer, 256)) == (wide < mdig)


# either side of every line of the rule: 8 and 16 rows per CU, the persistent
# form's 8192 rows, 4, 8 and 12 blocks
@pytest.mark.gpu
@pytest.mark.parametrize("t", (Q4_K, Q5_K))
@pytest.mark.parametrize("outer,inner", [(1, 1280), (7, 2304), (2047, 1024), (2048, 2304), (2049, 2048), (2049, 2304), (4096, 3328),
                                         (4095, 3072), (4097, 4096), (8191, 3584), (8192, 3328), (8197, 3072), (8203, 4096)])
def test_folded_norm_rows(t, outer, inner):
    import torch
    from inferno_hip import device as D
    print(f"folded norm type {t} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x6E0 + outer)
    w, x = synth.weight(rng, t, outer, inner), synth.activations(rng, inner)
    nw = rng.uniform(0.5, 1.5, inner).astype(np.float32)
    y = D.gemv_norm(D.DeviceWeight(torch.from_numpy(w).cuda(), t, inner, outer), torch.from_numpy(nw).cuda(), 1e-6,
                    torch.from_numpy(x).cuda()).cpu().numpy()
    n = oracle.rmsnorm_f64(x, nw, 1e-6)
    # the row bound, and the fp32 norm's few roundings
    tol = 1.01e-4 * oracle.row_norms(t, w, inner, outer) * np.linalg.norm(n)
    ratio = np.max(np.abs(y.astype(np.float64) - oracle.gemv_f64(t, w, n, inner, outer)) / tol)
    print(f"max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0


# (rows, columns, waves): timed with 8 and with 12
@pytest.mark.parametrize("outer,inner,waves", [(12288, 4096, 12), (4096, 4096, 12), (8192, 3328, 12), (32768, 3840, 12),
                                               (2048, 4096, 8), (1024, 4096, 8), (4096, 2560, 8), (512, 3328, 8)])
def test_q6_k_rows_of_four_steps(plan, outer, inner, waves):
    out = (C.c_int * 4)()
    plan.mdig_plan_of(Q6_K, outer, -(-inner // 1024), 256, out)
    assert out[0] == waves


@pytest.mark.gpu
@pytest.mark.parametrize("outer,inner", [(3073, 4096), (3072, 3328), (4099, 3840), (12301, 4096), (32771, 3328)])
def test_q6_k_rows_on_twelve_waves(outer, inner):
    """Against float64, and the bits of the same rows in a launch of 8 waves."""
    import torch
    from inferno_hip import device as D
    print(f"Q6_K {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x6E1 + outer)
    w, x = synth.weight(rng, Q6_K, outer, inner), synth.activations(rng, inner)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    y = D.gemv(D.DeviceWeight(wd, Q6_K, inner, outer), xd).cpu().numpy()
    tol = oracle.tolerance(oracle.row_norms(Q6_K, w, inner, outer), x)
    ratio = np.max(np.abs(y.astype(np.float64) - oracle.gemv_f64(Q6_K, w, x, inner, outer)) / tol)
    print(f"max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0
    k = 1021
    few = D.gemv(D.DeviceWeight(wd[: k * (len(w) // outer)], Q6_K, inner, k), xd).cpu().numpy()
    assert np.array_equal(few.view(np.uint32), y[:k].view(np.uint32))


GATE_UP_TIMES = (
    (Q4_K, 1024, 3328, 3.61, 3.95), (Q4_K, 1024, 2048, 3.46, 3.25), (Q4_K, 1024, 2816, 3.69, 3.45), (Q4_K, 1536, 2304, 3.61, 3.91), (Q4_K, 2048, 2816, 3.83, 4.14),
    (Q4_K, 1536, 3584, 3.90, 4.65), (Q4_K, 2304, 2560, 5.09, 4.56), (Q4_K, 9728, 3584, 10.62, 9.88), (Q4_K, 1408, 5120, 5.38, 4.86),
    (Q5_K, 512, 2560, 4.01, 3.70), (Q5_K, 1024, 3584, 4.40, 4.01), (Q5_K, 1536, 3328, 4.54, 4.85), (Q5_K, 2048, 3584, 4.85, 5.11),
    (Q5_K, 1408, 4096, 4.64, 4.83), (Q5_K, 1536, 3072, 4.52, 4.31), (Q5_K, 2304, 4096, 6.84, 5.98), (Q5_K, 14336, 4096, 18.28, 17.58))


@pytest.mark.parametrize("t,outer,inner,wide,mdig", GATE_UP_TIMES)
def test_gate_up_takes_the_faster_kernel(plan, t, outer, inner, wide, mdig):
    assert bool(plan.gate_up_takes_wide_of(t, inner // 256, outer, 256)) == (wide < mdig)


# either side of every line of the rule, with the folded norm and without
@pytest.mark.gpu
@pytest.mark.parametrize("t", (Q4_K, Q5_K))
@pytest.mark.parametrize("outer,inner", [(1, 2304), (2047, 2048), (2048, 2304), (2049, 2304), (1024, 2560), (1025, 2560), (1024, 3328), (1025, 3328),
                                         (2041, 4096), (2049, 3584), (1025, 3072)])
def test_gate_up_rows(t, outer, inner):
    import torch
    from inferno_hip import device as D
    print(f"gate/up type {t} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x6E2 + outer + inner)
    ws = [synth.weight(rng, t, outer, inner) for _ in range(2)]
    x, nw = synth.activations(rng, inner), rng.uniform(0.5, 1.5, inner).astype(np.float32)
    dws = [D.DeviceWeight(torch.from_numpy(w).cuda(), t, inner, outer) for w in ws]
    xd = torch.from_numpy(x).cuda()
    mats = [oracle.dequant(t, w, outer * inner).reshape(outer, inner).astype(np.float64) for w in ws]

    def check(h, n, what):
        g, u = (m @ n for m in mats)
        ng, nu = (np.linalg.norm(m, axis=1) * 1.01e-4 * np.linalg.norm(n) for m in mats)
        with np.errstate(over="ignore"):
            s = 1 / (1 + np.exp(-g))
        # silu's slope is below 1.1; fp32 roundings of the last two products
        tol = 1.1 * ng * (np.abs(u) + nu) + np.abs(g * s) * nu + 1e-6 * np.abs(g * s * u)
        assert np.all(np.abs(h - g * s * u) <= tol), what

    check(D.gate_up_swiglu(*dws, xd).cpu().numpy().astype(np.float64), x.astype(np.float64), "plain")
    wd = synth.weight(rng, Q4_K, inner, 256 * -(-outer // 256))
    if outer % 256 == 0:  # the norm's form is the FFN block's
        h = torch.empty(outer + inner, device="cuda")
        D.ffn_block(*dws, D.DeviceWeight(torch.from_numpy(wd).cuda(), Q4_K, outer, inner), torch.from_numpy(nw).cuda(),
                    1e-6, xd, h)
        check(h[:outer].cpu().numpy().astype(np.float64), oracle.rmsnorm_f64(x, nw, 1e-6), "norm")


# by length only: the rows of an engine's projections decide
@pytest.mark.parametrize("inner,wide,mdig", [(3328, 4.81, 5.21), (3584, 4.86, 5.25), (4096, 5.0, 5.4), (3072, 4.72, 4.44),
                                             (2560, 4.61, 4.34), (5120, 7.39, 5.62)])
def test_iq4_nl_of_4096_rows_takes_the_faster_kernel(plan, inner, wide, mdig):
    assert bool(plan.b32_takes_wide_of(synth.IQ4_NL, inner)) == (wide < mdig)


@pytest.mark.gpu
@pytest.mark.parametrize("outer,inner", [(1, 3328), (2049, 3328), (515, 3584), (8195, 3328), (9, 3360), (30, 3072)])
def test_iq4_nl_rows(outer, inner):
    import torch
    from inferno_hip import device as D
    print(f"IQ4_NL {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x6E3 + outer)
    w, x = synth.weight(rng, synth.IQ4_NL, outer, inner), synth.activations(rng, inner)
    y = D.gemv(D.DeviceWeight(torch.from_numpy(w).cuda(), synth.IQ4_NL, inner, outer), torch.from_numpy(x).cuda()).cpu().numpy()
    tol = oracle.tolerance(oracle.row_norms(synth.IQ4_NL, w, inner, outer), x)
    ratio = np.max(np.abs(y.astype(np.float64) - oracle.gemv_f64(synth.IQ4_NL, w, x, inner, outer)) / tol)
    print(f"max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0


def _mdig_walk(plan, t, outer, inner, gateup=False, norm=False, ncu=256):
    msg, st = C.create_string_buffer(512), (C.c_longlong * 8)()
    plan.mdig_check.restype = C.c_longlong
    n = plan.mdig_check(t, inner // (256 if t in (Q4_K, Q5_K, Q6_K) else 32), outer, int(gateup), int(norm), ncu, msg, 512, st)
    assert n == 0, f"type {t} {outer}x{inner} gate/up {gateup} norm {norm}: {n} violations, first: {msg.value.decode()}"
    return list(st)


# every number of steps, whole and partial last steps, ragged row groups
@pytest.mark.parametrize("t", (Q4_K, Q5_K, Q6_K, synth.Q8_0, synth.IQ4_NL))
def test_matrix_core_launches_stay_in_bounds(plan, t):
    unit = 256 if t in (Q4_K, Q5_K, Q6_K) else 32
    for nstep in range(1, 17):
        for inner in sorted({1024 * nstep, 1024 * nstep - unit, 1024 * (nstep - 1) + unit}):
            for outer in (1, 6, 1027, 4100):
                _mdig_walk(plan, t, outer, inner)
    for outer, inner in ((12288, 4096), (151936, 2560), (32771, 3328), (5, 16384)):
        _mdig_walk(plan, t, outer, inner)


@pytest.mark.parametrize("t", (Q4_K, Q5_K))
def test_matrix_core_gate_up_and_norm_launches_stay_in_bounds(plan, t):
    for nstep in range(1, 17):
        for inner in (1024 * nstep, 1024 * nstep - 768):
            for outer in (3, 1030, 2049):
                for norm in (False, True):
                    _mdig_walk(plan, t, outer, inner, gateup=True, norm=norm)
                if nstep <= 4:
                    _mdig_walk(plan, t, outer, inner, norm=True)
    _mdig_walk(plan, t, 13824, 5120, gateup=True, norm=True)


@pytest.mark.parametrize("ncu", (1, 7, 80, 304))
def test_matrix_core_launches_on_other_devices(plan, ncu):
    for t, outer, inner in ((Q6_K, 4099, 3840), (synth.Q8_0, 1031, 16352), (Q4_K, 2050, 8448), (Q5_K, 31, 256)):
        st = _mdig_walk(plan, t, outer, inner, ncu=ncu)
        assert st[1] * (-(-inner // 1024)) <= 512


@pytest.mark.parametrize("nb", range(1, 25))
def test_int8_q6_k_launches_stay_in_bounds(plan, nb):
    plan.q8k6_check.restype = C.c_longlong
    msg = C.create_string_buffer(512)
    for outer in (1, 15, 17, 257, 1030):
        for ncu in (80, 256):
            assert plan.q8k6_check(nb, outer, ncu, msg, 512) == 0, f"{outer} rows: {msg.value.decode()}"
