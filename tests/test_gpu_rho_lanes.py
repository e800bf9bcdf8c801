"""The fixed point's lanes per column (64, 32 or 16 by the columns of a tile):
every group size sums the elements by the same tree, so a column's equation of
state, hydrostatic integration and Stokes vector are the same bits whatever
tile it is launched in, on both sides of each limit, and follow the oracle."""
import numpy as np
import pytest

from firtez_dz_amd import atmos, gpu, lines

pytestmark = pytest.mark.gpu

NZ = 12


@pytest.fixture(scope="module")
def cube(gpu_ctx):
    import torch
    atm, z = atmos.seeded(61, 52, NZ, dz_km=80.0, seed=4)          # 3172 columns: 16 lanes
    gpu_ctx.configure(lines.fe6301_6302(nwave=9, start=-200.0, step=50.0), z)
    t = torch.from_numpy(atm).cuda()
    he = t.clone()
    s0 = gpu_ctx.hydrostatic_torch(he)
    fw = he.clone()
    st, _, s1 = gpu_ctx.forward_torch(fw, gpu.RF_NONE)
    torch.cuda.synchronize()
    assert int(s0.max()) == 0 and int(s1.max()) == 0
    return t, he, fw, st, z


@pytest.mark.parametrize("n", [1, 3, 63, 1024, 1025, 3072, 3073])
def test_lanes_per_column_same_bits(gpu_ctx, cube, n):
    import torch
    t, he, fw, st, z = cube
    for c0 in {0, t.shape[2] - n}:
        sub = t[:, :, c0:c0 + n].contiguous()
        gpu_ctx.hydrostatic_torch(sub)
        assert torch.equal(sub, he[:, :, c0:c0 + n])
        st2, _, status = gpu_ctx.forward_torch(sub, gpu.RF_NONE)
        torch.cuda.synchronize()
        assert int(status.max()) == 0
        assert torch.equal(sub, fw[:, :, c0:c0 + n]) and torch.equal(st2, st[c0:c0 + n])


def test_hydrostatic_vs_oracle(cube, cpu):
    """REAL(4) results of FP64 sums: a unit in the last place (6e-8), and one
    more iteration at most changes n_e by half the stopping test (5e-5) where a
    rounding decides it, which moves Pg by far less than 1e-6."""
    t, he, _, _, z = cube
    a, h = t.cpu().numpy(), he.cpu().numpy()
    for c in (0, 1, 1500, 3171):
        pg, rho, _, _, _ = cpu.he(a[0, :, c], float(a[1, -1, c]), z)
        assert np.max(np.abs(h[1, :, c] - pg) / pg) <= 1e-6
        assert np.max(np.abs(h[2, :, c] - rho) / rho) <= 1e-6
