"""The transfer's launch forms against each other and against the general path.

  * teams of waves (few columns, or no response functions) give the bits of one
    wave per 64 lanes (many columns, or per-pixel windows): the same columns
    synthesised alone, in a small and in a large cube, heights beside multiples
    of the team's size;
  * the node contraction within the transfer against the per-height
    Cartesian responses contracted on the host in 64 bits, for one node up to
    one per height, subsets of parameters and of Stokes parameters.
"""
import numpy as np
import pytest

from firtez_dz_amd import atmos, gpu, lines

pytestmark = pytest.mark.gpu


def cube(gpu_ctx, ls, ncol, nz, seed=5, he=False):
    import torch
    atm, z = atmos.seeded(ncol, 1, nz, dz_km=1200.0 / nz, seed=seed)
    gpu_ctx.configure(ls, z)
    gpu_ctx.gain_hsra()
    gpu_ctx.set_hydrostatic(False)
    d = torch.from_numpy(atm).cuda()
    assert int(gpu_ctx.hydrostatic_torch(d).max()) == 0
    gpu_ctx.set_hydrostatic(he)
    return d


@pytest.mark.parametrize("nz", [2, 7, 9, 33])
@pytest.mark.parametrize("mode,he", [(gpu.RF_NONE, False), (gpu.RF_SPHERICAL, False), (gpu.RF_CARTESIAN, True),
                                     (gpu.RF_CARTESIAN_P0, False), (gpu.RF_CARTESIAN_P0, True)])
def test_teams_give_the_bits_of_one_wave(gpu_ctx, nz, mode, he):
    import torch
    ls = lines.setup([((4, 5), 100, -624.0, 22.0), ((2,), 29, -300.0, 20.0)])
    try:
        d = cube(gpu_ctx, ls, 700, nz, he=he)
        # with response functions 1094 + 318 packed waves are no teams; a packed
        # synthesis always is one, per-pixel windows (here of every wavelength) are not
        if mode == gpu.RF_NONE:
            gpu_ctx.set_windows(np.tile(np.array([[0, 100], [0, 29]], np.int32), (700, 1, 1)))
        st, jac, status = gpu_ctx.forward_torch(d.clone(), mode)
        gpu_ctx.set_windows(None)
        st = st.reshape(700, 4, 129)
        assert int(status.max()) == 0 and bool(torch.isfinite(st).all())
        for n in (1, 5, 300) + ((700,) if mode == gpu.RF_NONE else ()):     # 8, 8 and 4 waves
            s1, j1, _ = gpu_ctx.forward_torch(d[:, :, :n].contiguous(), mode)
            assert torch.equal(s1, st[:n]), n
            if jac is not None:
                assert torch.equal(j1, jac[:n]), (n, [int((j1[:, p] != jac[:n, p]).sum()) for p in range(j1.shape[1])])
    finally:
        gpu_ctx.set_hydrostatic(False)


@pytest.mark.parametrize("nz", [2, 7, 33])
def test_teams_contract_to_the_bits_of_one_wave(gpu_ctx, nz):
    import torch
    ls = lines.setup([((4, 5), 100, -624.0, 22.0)])
    d = cube(gpu_ctx, ls, 700, nz)
    gpu_ctx.set_inversion(gpu.inversion({"T": min(4, nz), "Bx": 1, "By": 2, "Bz": nz, "vz": 2}))
    st, eqv, _ = gpu_ctx.forward_nodes_torch(d.clone())
    for n in (1, 130, 300):
        s1, e1, _ = gpu_ctx.forward_nodes_torch(d[:, :, :n].contiguous())
        assert torch.equal(s1, st[:n]) and torch.equal(e1, eqv[:n]), n


@pytest.mark.parametrize("nodes,invstk", [({"T": 1}, (1, 1, 1, 1)), ({"T": 3, "Bz": 1, "vz": 5}, (1, 0, 0, 1)),
                                          ({"Bx": 2, "By": 33}, (0, 1, 1, 0)),
                                          ({"T": 8, "Bx": 3, "By": 3, "Bz": 2, "vz": 4}, (1, 1, 1, 1))])
@pytest.mark.parametrize("ncol", [3, 700])
def test_contraction_against_general_path(gpu_ctx, cpu, nodes, invstk, ncol):
    nz = 33
    ls = lines.setup([((4, 5), 100, -624.0, 22.0)])
    d = cube(gpu_ctx, ls, ncol, nz)
    np_, nfreq = gpu_ctx.set_inversion(gpu.inversion(nodes, invstk=invstk))
    _, eqv, _ = gpu_ctx.forward_nodes_torch(d.clone())
    _, jac, _ = gpu_ctx.forward_torch(d.clone(), gpu.RF_CARTESIAN)
    eqv = eqv.cpu().numpy().astype(np.float64).reshape(ncol, np_, sum(invstk), gpu_ctx.numw)
    jac = jac.cpu().numpy().astype(np.float64)[:, :, :, [s for s in range(4) if invstk[s]]]
    names = gpu.PARAM_NAMES[gpu.RF_CARTESIAN]
    j0 = 0
    for name in [n for n in gpu.INV_PARAMS if n in nodes]:
        cf = np.array(cpu.int_coefs(nz, nodes[name]))              # [nz][nodes]
        J = jac[:, names.index(name)]                              # [ncol][nz][stk][numw]
        for j in range(nodes[name]):
            ref = np.einsum("k,cksw->csw", cf[:, j], J)
            mag = np.einsum("k,cksw->csw", np.abs(cf[:, j]), np.abs(J))
            # the responses themselves are 32-bit results of the same formulas (2e-6 of
            # the profile's largest), the sums are in 64 bits
            tol = 2e-6 * mag.max(axis=-1, keepdims=True) + 2.0 ** -23 * np.abs(ref) + 1e-35
            assert np.all(np.abs(eqv[:, j0 + j] - ref) <= tol), (name, j)
        j0 += nodes[name]
    assert j0 == np_


@pytest.mark.parametrize("ncol,mode", [(3, gpu.RF_NONE), (3, gpu.RF_SPHERICAL), (40, gpu.RF_CARTESIAN),
                                       (120, gpu.RF_SPHERICAL)])
def test_column_that_fails_in_one_region(gpu_ctx, ncol, mode):
    """A column whose profiles overflow in one region only (1e9 G, a line without Zeeman
    splitting in the other) is flagged.  Workgroups of its other region that start later than
    that return NaN, the others the region's own result, a whole team either way; the
    other columns, some of whose lanes share its waves, keep their bits."""
    import torch
    ls = lines.setup([((4,), 150, -600.0, 8.0), ((5,), 150, -600.0, 8.0)])
    for k, v in dict(sl=2.0, ll=3.0, jl=1.0, su=2.0, lu=2.0, ju=0.0).items():     # 5F1 - 5D0: g = 0
        setattr(ls.lines[ls.regions[0].lines[0]], k, v)
    one = lines.LineSetup([ls.lines[ls.regions[0].lines[0]]], [lines.Region([0], 150, -600.0, 8.0)])
    d = cube(gpu_ctx, ls, ncol, 33)
    d[7, :, 1] = 1e9
    good = [i for i in range(ncol) if i != 1]
    st, jac, status = gpu_ctx.forward_torch(d.clone(), mode)
    sg, jg, s0 = gpu_ctx.forward_torch(d[:, :, good].contiguous(), mode)
    torch.cuda.synchronize()
    assert int(s0.max()) == 0 and status.tolist() == [2 if i == 1 else 0 for i in range(ncol)]
    assert torch.equal(st[good], sg) and (jac is None or torch.equal(jac[good], jg))
    assert bool(torch.isnan(st[1, :, 150:]).all())
    gain = gpu_ctx.gain_hsra()
    gpu_ctx.configure(one, np.arange(33) * (1200.0 / 33))
    gpu_ctx.set_gain(gain[:, :150])
    s1, _, st1 = gpu_ctx.forward_torch(d[:, :, 1:2].contiguous(), gpu.RF_NONE)
    assert int(st1.max()) == 0
    got, ref = st[1, :, :150], s1[0]
    nan = torch.isnan(got)
    assert torch.equal(got[~nan], ref[~nan])
    assert torch.equal(nan, nan[:1].expand_as(nan))       # all four Stokes parameters of a wavelength
