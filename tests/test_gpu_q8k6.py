"""The streamed Q6_K kernel of the int8-activation variant (k_gemv_q8k6),
bit for bit against the oracle: rows of one block to the longest it takes and
one more, block counts around its items of eight (every byte phase of a row),
rows around its 16 waves and up to one round of the chip's and past it, x quantized in the
launch or before it.
"""
import numpy as np
import pytest

import oracle
from inferno_hip import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("outer,nb", [(1, 1), (3, 7), (15, 8), (17, 9), (33, 24), (5, 25), (4096, 3), (4099, 1), (257, 13), (1030, 20)])
def test_q6_k_rows_bit_exact(outer, nb):
    import torch
    from inferno_hip import device as D
    inner = 256 * nb
    print(f"q8k6 {outer}x{inner}", flush=True)
    rng = synth.rng_for(0x0860 + nb)
    w = synth.weight(rng, synth.Q6_K, outer, inner)
    x = synth.activations(rng, inner)
    x[:256] = 0.0 if nb > 1 else x[:256]  # a block of scale 0
    want = oracle.gemv_q8k(synth.Q6_K, w, x, inner, outer)
    dw = D.DeviceWeight(torch.from_numpy(w).cuda(), synth.Q6_K, inner, outer)
    xd = torch.from_numpy(x).cuda()
    q8 = torch.empty(nb * 292, dtype=torch.uint8, device="cuda")
    got = D.gemv_q8k_x(dw, xd, None, q8).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(q8.cpu().numpy(), oracle.quantize_row_q8k(x))
    again = D.gemv_q8k(dw, q8).cpu().numpy()
    assert np.array_equal(again.view(np.uint32), want.view(np.uint32))
