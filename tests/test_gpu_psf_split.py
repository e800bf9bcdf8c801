"""PSF convolution (psf[x][y] here) on the matrix cores against the 64-bit circular sum: tap
counts on both sides of the narrowest it takes and of its two strip widths, maps
beside multiples of the 32 x (64 or 128) tiles and narrower than one (several
turns of the periodic wrap), PSFs of one row; inputs and taps outside the range
of the split, which take the vector units tile by tile or as a whole.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(psf, maps, adjoint):
    py, px = psf.shape[1] // 2, psf.shape[0] // 2
    out = np.zeros(maps.shape)
    mag = np.zeros(maps.shape)
    for dx in range(-px, px + 1):
        for dy in range(-py, py + 1):
            w = float(np.float32(psf[px + dx, py + dy]))
            sh = (-dx, -dy) if adjoint else (dx, dy)
            r = np.roll(maps, sh, axis=(1, 2))
            out += w * r
            mag += abs(w) * np.abs(r)
    return out, mag


def run(ctx, psf, maps, adjoint):
    import torch
    nm, nx, ny = maps.shape
    ctx.set_psf(psf.T.copy())      # [y][x]
    try:
        t = torch.from_numpy(maps.reshape(nm, nx * ny).astype(np.float32)).cuda()
        return ctx.psf_convolve_torch(t, nx, ny, adjoint=adjoint).cpu().numpy().astype(np.float64).reshape(maps.shape)
    finally:
        ctx.set_psf(None)


@pytest.mark.parametrize("sx,sy,nx,ny", [(15, 15, 40, 70), (17, 17, 17, 17), (17, 1, 33, 65), (31, 31, 31, 64),
                                         (31, 3, 65, 128), (33, 33, 33, 129), (33, 5, 96, 40), (43, 21, 50, 200),
                                         (51, 7, 60, 100), (55, 3, 55, 257), (63, 63, 63, 63), (63, 1, 64, 300)])
@pytest.mark.parametrize("adjoint", [False, True])
def test_convolution_at_tile_edges(gpu_ctx, sx, sy, nx, ny, adjoint):
    rng = np.random.default_rng(sx * ny)
    psf = rng.normal(size=(sx, sy))
    maps = rng.normal(size=(3, nx, ny)).astype(np.float32).astype(np.float64)
    maps[1] *= 1e-9
    maps[2, : nx // 2] = 0.0
    got = run(gpu_ctx, psf, maps, adjoint)
    ref, mag = reference(psf, maps, adjoint)
    # products to 2^-24 (parts left out), FP32 sums of sx sy terms in six parts
    assert np.all(np.abs(got - ref) <= (sx * sy + 8) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38, 1e-35])
def test_inputs_outside_the_split(gpu_ctx, value):
    rng = np.random.default_rng(2)
    psf = rng.uniform(0.1, 1.0, (31, 9))
    nx, ny = 128, 300
    maps = rng.normal(size=(2, nx, ny)).astype(np.float32).astype(np.float64)
    if abs(value) < 1:
        maps[1] = value * rng.uniform(0.5, 1.0, (nx, ny)).astype(np.float32)
        maps = maps.astype(np.float32).astype(np.float64)
    else:
        maps[1, 40, 70] = np.float32(value)
    got = run(gpu_ctx, psf, maps, False)
    clean = maps.copy()
    if abs(value) < 1e30:
        ref, mag = reference(psf, clean, False)
        assert np.all(np.abs(got - ref) <= (31 * 9 + 8) * 2.0 ** -24 * mag + 2.0 ** -149 * 31 * 9)
        return
    clean[1, 40, 70] = 0.0
    ref, mag = reference(psf, clean, False)
    ok = np.abs(got - ref) <= (31 * 9 + 8) * 2.0 ** -24 * mag
    assert ok[0].all()
    hit = np.zeros((nx, ny), bool)
    hit[40 - 15:40 + 16, 70 - 4:70 + 5] = True
    if np.isfinite(value):
        big, _ = reference(psf, maps, False)
        assert np.all(np.abs(got[1][hit] - big[1][hit]) <= 1e-5 * np.abs(big[1][hit]))
        assert ok[1][~hit].all()
        return
    # a PSF of 31 is padded to 32 taps: 0 x inf reaches one row further
    pad = np.zeros((nx, ny), bool)
    pad[40 - 16:40 + 17, 70 - 4:70 + 5] = True
    assert ok[1][~pad].all()
    if np.isinf(value):
        assert np.all(got[1][hit] == value)
    else:
        assert np.isnan(got[1][hit]).all()


@pytest.mark.parametrize("sx", [17, 31, 33, 41, 55, 63])
@pytest.mark.parametrize("ny", [40, 70, 130, 200])
def test_tiles_outside_the_split(gpu_ctx, sx, ny):
    """Tiles of inputs below the split's range beside ordinary ones, for every tap
    count and tile height that is launched, last tiles partly and wholly past the map."""
    rng = np.random.default_rng(sx + ny)
    psf = rng.uniform(0.1, 1.0, (sx, 5))
    nx = 100
    maps = rng.normal(size=(2, nx, ny)).astype(np.float32).astype(np.float64)
    maps[0] *= 1e-33
    maps[1, 20, ny - 1] = 1e-33
    maps = maps.astype(np.float32).astype(np.float64)
    for adjoint in (False, True):
        got = run(gpu_ctx, psf, maps, adjoint)
        ref, mag = reference(psf, maps, adjoint)
        assert np.all(np.abs(got - ref) <= (sx * 5 + 8) * 2.0 ** -24 * mag + 2.0 ** -149 * sx * 5)


def test_taps_outside_the_split(gpu_ctx):
    rng = np.random.default_rng(3)
    psf = rng.uniform(0.5, 1.0, (21, 7))
    psf[0, 0] = 1e-33
    maps = rng.normal(size=(2, 70, 70)).astype(np.float32).astype(np.float64)
    got = run(gpu_ctx, psf, maps, False)
    ref, mag = reference(psf, maps, False)
    assert np.all(np.abs(got - ref) <= (21 * 7 + 8) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("ein,etap", [(-98, 0), (-90, -30), (-60, -60), (-95, -45), (-98, -98)])
def test_small_products(gpu_ctx, ein, etap):
    """Operands inside the split's range whose products, or the products of
    their parts, are subnormal: as exact as sums of FP32 products."""
    rng = np.random.default_rng(4)
    psf = rng.uniform(0.6, 1.0, (31, 9)) * 2.0 ** etap
    maps = (rng.uniform(0.6, 1.0, (2, 64, 70)) * rng.choice([-1.0, 1.0], (2, 64, 70)) * 2.0 ** ein)
    maps = maps.astype(np.float32).astype(np.float64)
    got = run(gpu_ctx, psf, maps, False)
    ref, mag = reference(psf, maps, False)
    # the bound of ordinary operands, and a rounding at the subnormal spacing for each of six products a tap
    assert np.all(np.abs(got - ref) <= (31 * 9 + 8) * 2.0 ** -24 * mag + 6 * 31 * 9 * 2.0 ** -149)
