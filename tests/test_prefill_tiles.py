"""Tile choice of the prefill GEMM: the wide kernel's 128-token tiles for products
with enough of them to fill the chip (prefill_wide_rows,
inferno.jl_amd/csrc/kq_launch.h), 32-token x 64-row tiles whose waves share K
for small ones (prefill_thin), 64 tokens x 128 rows otherwise, and both kernels
against a float64 product at the edges of their tiles.
"""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest

import oracle
from inferno_hip import synth

LIB = Path(__file__).resolve().parent / "native" / "_build" / "libsdig_check.so"


@pytest.fixture(scope="module")
def wide_rows():
    from inferno_hip import build
    if not LIB.exists():
        build.build_checks()
    f = C.CDLL(str(LIB)).prefill_wide_rows_of
    f.argtypes, f.restype = [C.c_int] * 4, C.c_int
    return lambda T, outer, inner, ncu=256: f(T, inner, outer, ncu)


@pytest.fixture(scope="module")
def thin(wide_rows):
    f = C.CDLL(str(LIB)).prefill_thin_of
    f.argtypes, f.restype = [C.c_int] * 4, C.c_int
    return lambda T, outer, inner, ncu=256: bool(f(T, inner, outer, ncu))


def test_thin_choice(thin):
    assert thin(8, 9728, 2560) and thin(77, 9728, 2560) and thin(128, 4096, 4096) and thin(512, 2048, 1024)
    assert not thin(512, 4096, 4096)       # one 64 x 128 tile per CU
    assert not thin(2048, 12288, 4096)
    assert not thin(64, 4096, 12288)       # long rows: split over workgroups
    assert not thin(1, 1 << 24, 1024)
    assert isinstance(thin(8, 512, 1024, 1), bool)


def test_tile_choice(wide_rows):
    assert wide_rows(512, 4096, 4096) == 0       # one 64 x 128 tile per CU
    assert wide_rows(64, 4096, 4096) == 0        # split over K
    assert wide_rows(1024, 4096, 4096) == 1
    assert wide_rows(2048, 12288, 4096) == 2
    assert wide_rows(1, 1 << 20, 1024) in (0, 1, 2)
    assert wide_rows(2048, 12288, 4096, ncu=1) == 2


# (tokens, rows, columns, rows per wave / 32): a last token tile of one token,
# of one short of full, a last row tile of one row; rows off 4 (scalar stores);
# columns of one more than kPrefillF32MaxK's blocks, of the exact-weight
# limit and past it; one and many row tiles
WIDE = ((641, 8193, 768, 1), (1151, 4099, 1024, 1), (1000, 4096, 2048, 1), (193, 12289, 2304, 1),
        (1025, 14081, 1024, 2), (1537, 8193, 1536, 2), (1279, 12290, 2304, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("T,outer,inner,ru", WIDE)
def test_wide_tiles_match_float64(wide_rows, T, outer, inner, ru):
    """Within 1e-4 * ||w_row|| * ||x|| of the float64 product, as every prefill
    launch on seeded random data."""
    assert wide_rows(T, outer, inner) == ru
    _match_float64("wide", T, outer, inner)


# one token and one row, tiles one short and one over, rows off 4; 3 to 16
# block columns (uneven shares of the wave halves), both weight roundings
THIN = ((1, 1, 768), (31, 63, 1024), (33, 65, 1280), (65, 4097, 2048), (32, 4096, 2304), (95, 4098, 2816), (300, 1030, 4096))


@pytest.mark.gpu
@pytest.mark.parametrize("T,outer,inner", THIN)
def test_thin_tiles_match_float64(thin, T, outer, inner):
    assert thin(T, outer, inner)
    _match_float64("thin", T, outer, inner)


def _match_float64(what, T, outer, inner):
    import torch
    from inferno_hip import device as D
    print(f"{what} prefill T={T} {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x71DE + T)
    w = synth.weight(rng, synth.Q4_K, outer, inner)
    X = (rng.standard_normal((T, inner)) * np.exp2(rng.integers(-20, 21, T))[:, None]).astype(np.float32)
    Y = D.prefill_q4_k(D.DeviceWeight(torch.from_numpy(w).cuda(), synth.Q4_K, inner, outer),
                       torch.from_numpy(X).cuda())
    wf = torch.from_numpy(oracle.dequant(synth.Q4_K, w, inner * outer).reshape(outer, inner)).cuda().double()
    xf = torch.from_numpy(X).cuda().double()
    ref = xf @ wf.t().contiguous()
    tol = 1e-4 * xf.norm(dim=1)[:, None] * wf.norm(dim=1)[None, :]
    ratio = ((Y.double() - ref).abs() / tol).max().item()
    print(f"{what} prefill max err/tol = {ratio:.3e}", flush=True)
    assert ratio <= 1.0
