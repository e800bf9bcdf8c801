"""Network kernels at the edges of their tiles: widths and batches beside
multiples of 16, 32 and 64, one hidden unit, the widest layer that the
one-launch forward takes and one beyond it, and batches on both sides of the
sizes at which its rows per workgroup change.

Tolerances: an activation or a gradient whose FP32 sum lies beside a BF16 rounding
boundary may round the other way (2^-8 of it), in every layer, which bounds
the relative change of results whose terms do not cancel; biases' and
weights' own sums are FP32.
"""
import numpy as np
import pytest

from oracle import mlp as omlp
from firtez_dz_amd import lines

pytestmark = pytest.mark.gpu


def make(gpu_ctx, nin, nh, nl, nodes):
    gpu_ctx.configure(lines.fe6301_6302(nwave=max(1, nin // 4)), np.arange(32) * 30.0)
    gpu_ctx.mlp_create(nin, nh, nl, nodes, 3)
    nout = 5 * nodes
    rng = np.random.default_rng(nin + nh)
    p = gpu_ctx.mlp_params().astype(np.float64)
    npar = len(p) - 2 * (nin + nout)
    p[:npar] += rng.normal(0, 0.02, npar)
    p[npar:npar + nin] = rng.normal(0.3, 0.2, nin)
    p[npar + nin:npar + 2 * nin] = rng.uniform(0.05, 0.2, nin)
    p[npar + 2 * nin:npar + 2 * nin + nout] = rng.normal(0, 1, nout)
    p[npar + 2 * nin + nout:] = rng.uniform(0.5, 2.0, nout)
    p = p.astype(np.float32)
    gpu_ctx.mlp_set_params(p)
    return p.astype(np.float64), nout, rng


SHAPES = [(1, 1, 1, 1), (4, 16, 1, 2), (33, 17, 2, 1), (100, 31, 1, 3), (96, 200, 2, 5), (64, 513, 1, 3),
          (448, 512, 3, 4), (31, 129, 6, 8)]


@pytest.mark.parametrize("nin,nh,nl,nodes", SHAPES)
@pytest.mark.parametrize("n", [1, 33, 100])
def test_forward_and_gradient(gpu_ctx, nin, nh, nl, nodes, n):
    import torch
    p, nout, rng = make(gpu_ctx, nin, nh, nl, nodes)
    x = rng.normal(0.3, 0.15, (2 * n, nin)).astype(np.float32)
    t = rng.normal(0, 1, (2 * n, nout)).astype(np.float32)
    idx = rng.permutation(2 * n)[:n].astype(np.int32)
    y = gpu_ctx.mlp_forward_torch(torch.from_numpy(x).cuda()).cpu().numpy()
    ref, _ = omlp.forward(p, x, nin, nh, nl, nout, emulate=True)
    tol = (nl + 1) * 2.0 ** -8
    assert np.max(np.abs(y - ref)) <= tol * np.abs(ref).max()
    loss, g = gpu_ctx.mlp_gradient_torch(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(),
                                         torch.from_numpy(idx).cuda())
    rl, rg = omlp.loss_and_grad(p, x[idx], t[idx], nin, nh, nl, nout, emulate=True)
    assert abs(float(loss.item()) - rl) <= 2 * tol * rl
    g = g.cpu().numpy()
    dims = [nin] + [nh] * nl + [nout]
    o = 0
    for i, k in zip(dims[:-1], dims[1:]):
        for sl in (slice(o, o + i * k), slice(o + i * k, o + i * k + k)):
            assert np.max(np.abs(g[sl] - rg[sl])) <= tol * max(np.abs(rg[sl]).max(), 1e-30)
        o += i * k + k


@pytest.mark.parametrize("nin,nh", [(100, 200), (448, 512), (64, 513)])
def test_rows_do_not_depend_on_the_batch(gpu_ctx, nin, nh):
    """A row's result is the same bits in every batch, and in the initial model: the sums over
    a layer's inputs run in one order."""
    import torch
    p, nout, rng = make(gpu_ctx, nin, nh, 2, 4)
    x = torch.from_numpy(rng.normal(0.3, 0.15, (8200, nin)).astype(np.float32)).cuda()
    y = gpu_ctx.mlp_forward_torch(x)
    for n in (1, 17, 4096, 4097, 8192):
        assert torch.equal(gpu_ctx.mlp_forward_torch(x[:n]), y[:n]), n
    atm = torch.zeros((12, 32, 8200), device="cuda")
    gpu_ctx.learned_init_torch(x.double(), atm)
    for n in (1, 4097):
        a = torch.zeros((12, 32, n), device="cuda")
        gpu_ctx.learned_init_torch(x[:n].double().contiguous(), a)
        assert torch.equal(a, atm[:, :, :n]), n


def test_training_after_larger_and_smaller_batches(gpu_ctx):
    """Buffers of a larger batch hold nothing that a smaller one reads."""
    import torch
    p, nout, rng = make(gpu_ctx, 100, 72, 2, 2)
    x = torch.from_numpy(rng.normal(0.3, 0.15, (300, 100)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.normal(0, 1, (300, nout)).astype(np.float32)).cuda()
    l0, g0 = gpu_ctx.mlp_gradient_torch(x[:45].contiguous(), t[:45].contiguous())
    l0, g0 = l0.clone(), g0.clone()
    big = x.clone()
    big[45:] = float("nan")
    gpu_ctx.mlp_gradient_torch(big, t)
    l1, g1 = gpu_ctx.mlp_gradient_torch(x[:45].contiguous(), t[:45].contiguous())
    npar = g0.numel() - 2 * (100 + nout)
    assert torch.equal(l0, l1) and torch.equal(g0[:npar], g1[:npar])


def test_gradient_of_large_tiles(gpu_ctx):
    """A batch whose hidden layers take 64 x 64 tiles, forward and backward."""
    check_gradient(gpu_ctx, 64, 513, 2, 2, 4100)


@pytest.mark.parametrize("indexed", [False, True])
def test_gradient_in_parts(gpu_ctx, indexed):
    """More rows than one pass takes (2^20): loss and gradient of all of them."""
    check_gradient(gpu_ctx, 5, 17, 1, 1, (1 << 20) + 37, indexed)


def check_gradient(gpu_ctx, nin, nh, nl, nodes, n, indexed=True):
    import torch
    p, nout, rng = make(gpu_ctx, nin, nh, nl, nodes)
    x = rng.normal(0.3, 0.15, (n + 9, nin)).astype(np.float32)
    t = rng.normal(0, 1, (n + 9, nout)).astype(np.float32)
    idx = rng.permutation(n + 9)[:n].astype(np.int32) if indexed else np.arange(n)
    loss, g = gpu_ctx.mlp_gradient_torch(*(torch.from_numpy(v if indexed else v[:n]).cuda() for v in (x, t)),
                                         torch.from_numpy(idx).cuda() if indexed else None)
    rl, rg = omlp.loss_and_grad(p, x[idx], t[idx], nin, nh, nl, nout, emulate=True)
    tol = (nl + 1) * 2.0 ** -8
    assert abs(float(loss.item()) - rl) <= 2 * tol * rl
    g = g.cpu().numpy()
    dims = [nin] + [nh] * nl + [nout]
    o = 0
    for i, k in zip(dims[:-1], dims[1:]):
        for sl in (slice(o, o + i * k), slice(o + i * k, o + i * k + k)):
            assert np.max(np.abs(g[sl] - rg[sl])) <= tol * max(np.abs(rg[sl]).max(), 1e-30)
        o += i * k + k


@pytest.mark.parametrize("nin", [100, 448])
def test_outputs_in_the_place_of_inputs(gpu_ctx, nin):
    """The forward pass with its output at the start of its input gives the
    bits of one apart from it."""
    import ctypes
    import torch
    p, nout, rng = make(gpu_ctx, nin, 200, 2, 4)
    x = torch.from_numpy(rng.normal(0.3, 0.15, (5000, nin)).astype(np.float32)).cuda()
    ref = gpu_ctx.mlp_forward_torch(x)
    q = ctypes.c_void_p(x.data_ptr())
    assert gpu_ctx.lib.fz_mlp_forward_dev(gpu_ctx.h, 5000, q, None, q, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(x.reshape(-1)[:5000 * nout].reshape(5000, nout), ref)
