"""The four-row matrix-core GEMV (k_gemv_mdig) at the edges of what it takes:
groups of one to four rows, steps of one to four blocks, rows at every length
where the launch changes, Q6_K rows at every byte phase, and activations at
the ends of fp32's range.  Against the float64 sums, and row for row the same
whatever the launch.
"""
import numpy as np
import pytest

import oracle
from inferno_hip import synth

pytestmark = pytest.mark.gpu

TYPES = (synth.Q4_K, synth.Q5_K, synth.Q6_K, synth.Q8_0, synth.IQ4_NL)


def _gemv(t, w, x, outer, inner, resid=None):
    import torch
    from inferno_hip import device as D
    dw = D.DeviceWeight(torch.from_numpy(w).cuda(), t, inner, outer)
    xd = torch.from_numpy(x).cuda()
    if resid is None:
        return D.gemv(dw, xd).cpu().numpy()
    return D.gemv_add(dw, xd, torch.from_numpy(resid).cuda()).cpu().numpy()


def _check(t, w, x, y, outer, inner, floor=0.0):
    ref = oracle.gemv_f64(t, w, x, inner, outer)
    tol = oracle.tolerance(oracle.row_norms(t, w, inner, outer), x) + floor
    ratio = np.max(np.abs(y.astype(np.float64) - ref) / tol)
    print(f"type {t} {outer}x{inner}: max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("outer,inner", [(1, 256), (3, 768), (5, 1024), (6, 1280), (1027, 3072), (9, 4096), (1029, 4352),
                                         (2, 12288), (1030, 12544), (7, 16384), (4100, 5120), (65, 16128)])
def test_gemv_edges(t, outer, inner):
    print(f"gemv type {t} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x4D16 + outer)
    w = synth.weight(rng, t, outer, inner)
    x = synth.activations(rng, inner)
    y = _gemv(t, w, x, outer, inner)
    _check(t, w, x, y, outer, inner)
    # the first rows alone, in another launch: the same bits; the residual is
    # one fp32 addition after the sum
    k = max(1, outer // 3)
    rows = w[: k * (len(w) // outer)]
    assert np.array_equal(_gemv(t, rows, x, k, inner).view(np.uint32), y[:k].view(np.uint32))
    r = rng.standard_normal(outer).astype(np.float32)
    assert np.array_equal(_gemv(t, w, x, outer, inner, r).view(np.uint32), (r + y).view(np.uint32))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("scale", [2.0 ** -140, 2.0 ** -126, 2.0 ** 110])
def test_gemv_ends_of_the_range(t, scale):
    print(f"gemv type {t} scale {scale}", flush=True)
    rng = synth.rng_for(0x4D17)
    outer, inner = 70, 4352
    w = synth.weight(rng, t, outer, inner)
    x = (rng.uniform(-1, 1, inner) * scale).astype(np.float32)
    x[64:96] = 0.0
    # results near fp32's smallest step: half of it for each of the 136 sub-block terms
    _check(t, w, x, _gemv(t, w, x, outer, inner), outer, inner, 136 * 2.0 ** -150)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_gemv_non_finite(t, bad):
    rng = synth.rng_for(0x4D18)
    outer, inner = 33, 4352
    x = synth.activations(rng, inner)
    x[4300] = bad
    assert np.isnan(_gemv(t, synth.weight(rng, t, outer, inner), x, outer, inner)).all()


@pytest.mark.parametrize("t", TYPES[:2])
@pytest.mark.parametrize("hidden,inter", [(3584, 768), (768, 1024), (4352, 256), (9472, 256), (16384, 256)])
def test_ffn_block_norm(t, hidden, inter):
    """x and the norm's weights through the ring, in one piece and in two."""
    import torch
    from inferno_hip import device as D
    print(f"ffn block type {t} {hidden}x{inter}", flush=True)
    rng = synth.rng_for(0x4D1A + hidden)
    wg, wu = synth.weight(rng, t, inter, hidden), synth.weight(rng, t, inter, hidden)
    wd = synth.weight(rng, t, hidden, inter)
    x, nw = synth.activations(rng, hidden), rng.uniform(0.5, 1.5, hidden).astype(np.float32)
    h = torch.empty(inter + hidden, device="cuda")
    dw = [D.DeviceWeight(torch.from_numpy(a).cuda(), t, k, o) for a, k, o in
          ((wg, hidden, inter), (wu, hidden, inter), (wd, inter, hidden))]
    D.ffn_block(*dw, torch.from_numpy(nw).cuda(), 1e-6, torch.from_numpy(x).cuda(), h)
    got = h[:inter].cpu().numpy().astype(np.float64)
    n = oracle.rmsnorm_f64(x, nw, 1e-6)
    mats = [oracle.dequant(t, a, inter * hidden).reshape(inter, hidden).astype(np.float64) for a in (wg, wu)]
    g, u = (m @ n for m in mats)
    ng, nu = (np.linalg.norm(m, axis=1) * 1.01e-4 * np.linalg.norm(n) for m in mats)
    with np.errstate(over="ignore"):
        s = 1 / (1 + np.exp(-g))
    assert np.all(np.abs(got - g * s * u) <= 1.1 * ng * (np.abs(u) + nu) + np.abs(g * s) * nu + 1e-6 * np.abs(g * s * u))
