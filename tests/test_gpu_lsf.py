"""The LSF contraction at the edges of its tiles (16 rows, 16 outputs in
groups of 64, four taps a step) and on both sides of the widest region it
takes (904 wavelengths), against the circular convolution of the same profiles in 64 bits.  Taps
of either sign without symmetry; a region without LSF stays as it is.
"""
import numpy as np
import pytest

from firtez_dz_amd import atmos, gpu, lines

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2,ncol", [(1, 2, 1), (3, 4, 3), (15, 16, 4), (17, 63, 5), (64, 65, 9), (100, 31, 17),
                                        (130, 1, 2), (860, 5, 5), (861, 4, 5), (904, 2, 5), (905, 3, 5),
                                        (1000, 3, 3)])
@pytest.mark.parametrize("valid", [(1, 1), (0, 1), (1, 0)])
def test_lsf_against_convolution(gpu_ctx, n1, n2, ncol, valid):
    import torch
    ls = lines.setup([((4,), n1, -300.0, 600.0 / n1), ((5,), n2, -300.0, 600.0 / n2)])
    atm, z = atmos.seeded(ncol, 1, 32, dz_km=30.0, seed=n1)
    gpu_ctx.configure(ls, z)
    gpu_ctx.gain_hsra()
    d = torch.from_numpy(atm).cuda()
    assert int(gpu_ctx.hydrostatic_torch(d).max()) == 0
    st0, jac0, _ = gpu_ctx.forward_torch(d.clone(), gpu.RF_SPHERICAL if n1 < 200 else gpu.RF_NONE)
    rng = np.random.default_rng(n1)
    taps = [rng.normal(0, 1, n) for n in (n1, n2)]
    kern = np.concatenate([t / np.abs(t).sum() / t.size for t in taps])     # the rows see n * kern
    gpu_ctx.set_lsf(kern, np.array(valid, np.int32))
    try:
        st1, jac1, _ = gpu_ctx.forward_torch(d.clone(), gpu.RF_SPHERICAL if n1 < 200 else gpu.RF_NONE)
    finally:
        gpu_ctx.set_lsf(None)
    for a, b in ((st0, st1), (jac0, jac1)):
        if a is None:
            continue
        x = a.cpu().numpy().astype(np.float64).reshape(-1, n1 + n2)
        y = b.cpu().numpy().astype(np.float64).reshape(-1, n1 + n2)
        for p0, n, v in ((0, n1, valid[0]), (n1, n2, valid[1])):
            xr, yr = x[:, p0:p0 + n], y[:, p0:p0 + n]
            if not v:
                assert np.array_equal(xr, yr)
                continue
            t = (kern[p0:p0 + n] * n).astype(np.float32).astype(np.float64)
            c = t[(np.arange(n)[:, None] - np.arange(n)[None, :]) % n]      # c[i, k] = tap (i - k) mod n
            # n products and sums in 32 bits: at most n + 1 roundings of the sum of magnitudes
            bound = (n + 1) * 2.0 ** -24 * (np.abs(xr) @ np.abs(c).T) + 1e-37
            assert np.all(np.abs(xr @ c.T - yr) <= bound), (p0, n)
