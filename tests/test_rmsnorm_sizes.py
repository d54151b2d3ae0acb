"""k_rmsnorm at the lengths where its form changes (values in registers, two
or eight a thread, or read again), in place and not, against the fp64 oracle."""
import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 1023, 1025, 2048, 2049, 8191, 8192, 8193, 20000])
def test_rmsnorm_sizes(n):
    import torch
    from inferno_hip import device as D
    print(f"rmsnorm n={n}", flush=True)
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 3).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    ref = oracle.rmsnorm_f64(x, w, 1e-6)
    # the sum of squares, the root and the quotient, and two products: 4 ulps
    tol = 4 * np.spacing(np.abs(ref).astype(np.float32)) + 1e-30
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    assert np.all(np.abs(D.rmsnorm(xd, wd, 1e-6).cpu().numpy() - ref) <= tol)
    D.rmsnorm(xd, wd, 1e-6, out=xd)
    assert np.all(np.abs(xd.cpu().numpy() - ref) <= tol)
