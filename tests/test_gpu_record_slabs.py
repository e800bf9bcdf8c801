"""Maps whose per-height records do not fit the memory that is left are worked
through in slabs of columns: the same bits as with all records at once."""
import numpy as np
import pytest

from firtez_dz_amd import atmos, gpu, lines

pytestmark = pytest.mark.gpu

NZ, NCOL = 96, 12000
CALLS = ("synthesis", "responses", "nodes", "pressure", "line_tau")


def run(call, ls, z, gain, start):
    import torch
    ctx = gpu.Context(0)
    try:
        ctx.configure(ls, z)
        ctx.set_gain(gain)
        model = start.clone()
        if call in ("nodes", "pressure"):
            ctx.set_inversion(gpu.inversion({"T": 4, "Bz": 2} if call == "nodes" else {"T": 2, "Pg": 1}))
            out = ctx.forward_nodes_torch(model)
        elif call == "line_tau":
            out = ctx.line_tau_torch(model)
        else:
            out = ctx.forward_torch(model, gpu.RF_SPHERICAL if call == "responses" else gpu.RF_NONE)
        torch.cuda.synchronize()
        return [model.cpu()] + [t.cpu() for t in (out if isinstance(out, tuple) else (out,)) if t is not None]
    finally:
        ctx.close()


def test_slabs_give_the_same_bits(gpu_ctx):
    import torch
    # 32 line slots: 3.3 KB a record, 3.8 GB in all
    ls = lines.setup([((4, 5, 4, 5), 2, -100.0 * r, 900.0) for r in range(8)])
    nrec = 4 * NZ * NCOL * (1 + 24 + 8 * (4 + 4 * 24))
    atm, z = atmos.seeded(120, NCOL // 120, NZ, seed=6)
    gpu_ctx.configure(ls, z)
    gain = gpu_ctx.gain_hsra()
    start = torch.from_numpy(atm).cuda()
    assert int(gpu_ctx.hydrostatic_torch(start).max()) == 0
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] // 3 > nrec
    whole = {c: run(c, ls, z, gain, start) for c in CALLS}
    # 7 GB left, of which the records may take a third, outputs and work arrays the rest
    torch.cuda.empty_cache()
    hold = torch.empty(torch.cuda.mem_get_info()[0] - (7 << 30), dtype=torch.uint8, device="cuda")
    try:
        for c in CALLS:
            assert torch.cuda.mem_get_info()[0] // 3 < nrec
            for a, b in zip(whole[c], run(c, ls, z, gain, start)):
                assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b), c
            torch.cuda.empty_cache()
    finally:
        del hold
        torch.cuda.empty_cache()
