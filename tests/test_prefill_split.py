"""The product on fp32 operands (k_prefill_q4k_split: X cut into three bf16
parts, K shared by the eight waves of a workgroup) against float64 at the edges
of its tiles and of its share of K, and with values at the ends of fp32's range.
"""
import numpy as np
import pytest

import oracle
from inferno_hip import synth

pytestmark = pytest.mark.gpu


def _product(w, X, outer, inner):
    import torch
    from inferno_hip import device as D
    Y = D.prefill_q4_k_f32(D.DeviceWeight(torch.from_numpy(w).cuda(), synth.Q4_K, inner, outer),
                           torch.from_numpy(X).cuda())
    return Y.cpu().numpy().astype(np.float64)


def _check(w, X, outer, inner, what):
    wf = oracle.dequant(synth.Q4_K, w, inner * outer).reshape(outer, inner).astype(np.float64)
    xf = X.astype(np.float64)
    # fp32 rounding stays under a tenth of the row bound 1e-4 ||w_row|| ||x||
    # (K terms of 2^-24 each, random signs: 2^-24 sqrt(K) / sqrt(K) of the norms
    # times the six roundings of a sub-block); one step of fp32's
    # subnormals for results below its range
    tol = 1e-5 * np.linalg.norm(wf, axis=1)[None, :] * np.linalg.norm(xf, axis=1)[:, None] + 2.0 ** -149
    ratio = np.max(np.abs(_product(w, X, outer, inner) - xf @ wf.T) / tol)
    print(f"{what}: max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0


# tokens around the 32- and 64-token tiles, rows around 64 and off 4 (scalar
# stores), one to nine block columns (the wave halves' uneven shares, none for one)
@pytest.mark.parametrize("T,outer,inner", [(1, 1, 256), (31, 63, 512), (33, 65, 768), (32, 4096, 256),
                                           (63, 130, 2304), (65, 8193, 512), (129, 4095, 1280), (257, 4100, 256)])
def test_tile_edges(T, outer, inner):
    print(f"split prefill T={T} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x5B17 + T)
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    X = (rng.standard_normal((T, inner)) * np.exp2(rng.integers(-20, 21, T))[:, None]).astype(np.float32)
    _check(w, X, outer, inner, f"{T}x{outer}x{inner}")


@pytest.mark.parametrize("scale", [2.0 ** -140, 2.0 ** -120, 2.0 ** -100, 2.0 ** 100, 2.0 ** 116, 2.0 ** 119])
def test_ends_of_the_range(scale):
    """Tokens whose bf16 parts would be subnormal or whose sub-block sums would
    overflow (their tiles are computed on scaled tokens)."""
    print(f"split prefill scale={scale}", flush=True)
    rng = synth.rng_for(0x5B18)
    T, outer, inner = 40, 70, 512
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    X = (rng.uniform(-1, 1, (T, inner)) * scale).astype(np.float32)
    X[3] = rng.standard_normal(inner)  # an ordinary token in the same tile
    _check(w, X, outer, inner, f"scale {scale}")


def test_non_finite_activations_reach_their_tokens_only():
    rng = synth.rng_for(0x5B19)
    T, outer, inner = 70, 64, 512
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    X = rng.standard_normal((T, inner)).astype(np.float32)
    bad = X.copy()
    bad[5, 100], bad[66, 300] = np.nan, np.inf
    bad.view(np.uint32)[7, 9] = 0x7F800001  # a NaN whose upper half is an infinity's
    Y, Z = _product(w, X, outer, inner), _product(w, bad, outer, inner)
    wf = oracle.dequant(synth.Q4_K, w, inner * outer).reshape(outer, inner)
    assert np.isnan(Z[5]).all() and np.isnan(Z[7]).all()
    col = wf[:, 300]
    assert np.array_equal(np.isposinf(Z[66]), col > 0) and np.array_equal(np.isneginf(Z[66]), col < 0)
    keep = [t for t in range(T) if t not in (5, 7, 66)]
    np.testing.assert_allclose(Z[keep], Y[keep], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("bias", [0.0, 3.0])
def test_error_is_no_larger_than_fp32_products_in_order(bias):
    """Against the fp32 sum of fp32 products in column order, activations with
    and without a common offset."""
    rng = synth.rng_for(0x5B1A)
    T, outer, inner = 64, 256, 2048
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    X = (rng.standard_normal((T, inner)) + bias).astype(np.float32)
    wf = oracle.dequant(synth.Q4_K, w, inner * outer).reshape(outer, inner).astype(np.float32)
    exact = X.astype(np.float64) @ wf.T.astype(np.float64)
    serial = np.zeros((T, outer), np.float32)
    for k in range(inner):
        serial += X[:, k:k + 1] * wf[None, :, k]
    here = np.linalg.norm(_product(w, X, outer, inner) - exact)
    there = np.linalg.norm(serial - exact)
    print(f"bias {bias}: {here / np.linalg.norm(exact):.2e}, fp32 in order {there / np.linalg.norm(exact):.2e}", flush=True)
    assert here <= there


@pytest.mark.parametrize("top", [2.0 ** 75, 2.0 ** 90, 2.0 ** 117])
def test_terms_that_cancel_do_not_overflow(top):
    """Weights of zero beside a large scale (quants 0, scale 63, d = 1): the two
    terms they are split into are 472 times the activations and cancel."""
    print(f"split prefill cancelling terms, x to {top}", flush=True)
    rng = synth.rng_for(0x5B1B)
    T, outer, inner = 33, 65, 512
    w = np.zeros((outer, inner // 256, 144), np.uint8)
    w[:, :, 0:2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)  # d = 1, dmin = 0
    w[:, :, 4:8], w[:, :, 12:16] = 0xFF, 0x0F  # the eight scales 63, the mins 0
    w[:, :, 8:12] = 0
    w[:, :, 16::32] = 1  # one weight of 63 in each 64
    w = w.reshape(-1)
    X = (rng.uniform(0.5, 1, (T, inner)) * top).astype(np.float32)
    _check(w, X, outer, inner, f"cancelling terms, x to {top}")


# a tile of 64 tokens, one of 32; K shared unevenly by the wave halves
@pytest.mark.parametrize("T,outer,inner", [(600, 2050, 768), (70, 66, 2304), (5, 3, 256)])
def test_infinities_in_many_tokens(T, outer, inner):
    """Infinities of one sign, of both and beside a NaN, on weights of either
    sign and of zero, in tokens of ordinary and of extreme size: every output is
    what IEEE sums give."""
    print(f"split prefill with infinities T={T} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x5B1C + T)
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    blocks = w.reshape(outer, inner // 256, 144)
    zero = np.arange(outer) % 3 == 1
    blocks[zero, 0, 4:16] = 0  # rows whose first block has scales and mins of zero
    X = rng.standard_normal((T, inner)).astype(np.float32)
    X[1::5] *= np.float32(2.0) ** rng.integers(-140, 120, X[1::5].shape[0])[:, None].astype(np.float32)
    kinds = np.arange(T) % 5  # 0 finite, 1 one infinity, 2 several of one sign, 3 of both, 4 beside a NaN
    for t in range(T):
        n = (0, 1, 4, 4, 2)[kinds[t]]
        at = rng.integers(0, inner, n)
        X[t, at] = np.inf if t % 2 else -np.inf
        if kinds[t] == 2:  # where a row's weights have one sign, it is the result's
            X[t, at[1:]] = X[t, at[0]]
        if kinds[t] == 3:
            X[t, at[1::2]] = -X[t, at[0]]
        if kinds[t] == 4:
            X[t, (at[1] + 1) % inner] = np.nan
    wf = oracle.dequant(synth.Q4_K, w, inner * outer).reshape(outer, inner).astype(np.float64)
    got = _product(w, X, outer, inner)
    seen = set()
    with np.errstate(invalid="ignore"):
        for t in range(T):
            if kinds[t] == 0:
                continue
            bad = np.flatnonzero(~np.isfinite(X[t]))
            want = (X[t, bad].astype(np.float64)[None, :] * wf[:, bad]).sum(axis=1)
            assert np.array_equal(got[t], want, equal_nan=True), t
            seen |= {str(v) for v in np.unique(want[np.isfinite(want) == 0])}
    assert {"inf", "-inf", "nan"} <= seen
    fin = kinds == 0
    tol = 1e-5 * np.linalg.norm(wf, axis=1)[None, :] * np.linalg.norm(X[fin].astype(np.float64), axis=1)[:, None] + 2.0 ** -149
    assert np.all(np.abs(got[fin] - X[fin].astype(np.float64) @ wf.T) <= tol)


def test_rows_past_32_bit_offsets():
    """Rows of 2^24 + 256 columns: tokens and weight rows addressed by 64 bits."""
    rng = synth.rng_for(0x5B1D)
    T, outer, inner = 33, 3, (1 << 24) + 256
    print(f"split prefill T={T} {outer}x{inner}", flush=True)
    row = synth.weight(rng, synth.Q4_K, outer, 4096).reshape(outer, 16, 144)
    w = np.concatenate([np.tile(row, (1, inner // 4096, 1)), row[:, :1]], axis=1)  # 4097 x 16 + 1 blocks
    x = rng.standard_normal(4096).astype(np.float32)
    import torch
    from inferno_hip import device as D
    dw = D.DeviceWeight(torch.from_numpy(np.ascontiguousarray(w).reshape(-1)).cuda(), synth.Q4_K, inner, outer)
    X = torch.zeros(T, inner, device="cuda")
    xd = torch.from_numpy(x).cuda()
    scales = 1.0 + torch.arange(T, device="cuda") / 8
    X[:, : inner - 256].view(T, -1, 4096).copy_(xd * scales[:, None, None])
    X[:, inner - 256:] = xd[:256] * scales[:, None]
    got = D.prefill_q4_k_f32(dw, X).cpu().numpy().astype(np.float64)
    wf = oracle.dequant(synth.Q4_K, row.reshape(-1), 4096 * outer).reshape(outer, 4096).astype(np.float64)
    n = inner // 4096
    x8 = (x[None, :] * scales.cpu().numpy()[:, None]).astype(np.float64)
    want = n * (x8 @ wf.T) + x8[:, :256] @ wf[:, :256].T
    norms = np.sqrt(n) * np.linalg.norm(wf, axis=1)[None, :] * np.sqrt(n) * np.linalg.norm(x8, axis=1)[:, None]
    # the row bound: a wave adds 65538 sub-block sums in order, each rounding
    # 2^-24 of a running sum of about a 64th of the norms' product (the cosine of
    # 4096 random values): 6e-5 if every rounding went the same way
    assert np.max(np.abs(got - want) / norms) <= 1e-4
