"""Host code of the library on a machine without a GPU (tests/hostdouble): what
it launches and holds after allocations fail, and with maps at the limits of
the card.  Each case runs in an interpreter of its own."""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "firtez_dz_amd", "libfirtez_gpu.so")


def psf_launches(d):
    d.watch["psf_"] = lambda x: (("operands" if "operand" in x.name else "split" if "split" in x.name else "vector"),
                                 x.arg(1, ctypes.c_void_p).value if "split" in x.name else None)

    def convolve(ctx, nx, ny, _buf=[]):
        if not _buf:
            _buf.append((d.malloc(1 << 24), d.malloc(1 << 24)))
        return ctx.lib.fz_psf_convolve_dev(ctx.h, nx, ny, 2, _buf[0][0], _buf[0][1], 0, None)
    return convolve


def case_psf_failed_operands():
    """A failed allocation while the taps are cut leaves no state that a
    later convolution would launch with missing operands."""
    import numpy as np
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    convolve = psf_launches(d)
    ctx.set_psf(np.full((17, 17), 1.0 / 289.0))
    assert convolve(ctx, 64, 64) == 0
    ctx.set_psf(np.full((31, 31), 1.0 / 961.0))
    d.seen.clear()
    for fail in range(2):           # the tables, nothing
        d.lib.double_fail_after(fail)
        rc = convolve(ctx, 64, 64)
        assert (rc != 0) == (fail < 1) and len(d.seen) == 2 * fail, (fail, rc)
    d.lib.double_fail_after(-1)
    for n in (64, 70, 64):
        assert convolve(ctx, n, n) == 0
    assert [k for k, _ in d.seen] == ["operands"] + 4 * ["split"] and all(f for k, f in d.seen if k == "split"), d.seen


def case_psf_tables_of_a_psf():
    """The tables are made once for a PSF, whatever maps it is applied to, and
    again for another one; maps narrower than the PSF are refused."""
    import numpy as np
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    convolve = psf_launches(d)
    for side, kind in ((31, "split"), (15, "vector"), (43, "split"), (63, "split"), (17, "split")):
        ctx.set_psf(np.full((side, side), 1.0 / side ** 2))
        d.seen.clear()
        assert convolve(ctx, side, side) == 0
        n = d.lib.double_mallocs()
        for nx, ny in ((64, 70), (200, 63), (63, 200), (64, 70)):
            assert convolve(ctx, nx, ny) == 0
            assert convolve(ctx, side - 1, ny) != 0 and convolve(ctx, nx, side - 1) != 0
        assert d.lib.double_mallocs() == n
        assert [k for k, _ in d.seen] == (["operands"] if kind == "split" else []) + 5 * [kind], d.seen
    ctx.set_psf(None)
    assert convolve(ctx, 64, 64) != 0


def case_network_buffers_only_grow():
    """Training batches between forward passes of a large map allocate
    nothing once both sizes have been seen, in either order."""
    import numpy as np
    from firtez_dz_amd import lines
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    ctx.configure(lines.fe6301_6302(nwave=16), np.arange(32) * 30.0)
    x = d.malloc(1 << 30)
    for sizes in ((5000, 100), (100, 5000), (70000, 70000)):
        ctx.mlp_create(64, 513, 2, 3)
        def both():
            assert ctx.lib.fz_mlp_forward_dev(ctx.h, sizes[0], x, None, x, None) == 0
            assert ctx.lib.fz_mlp_gradient_dev(ctx.h, sizes[1], x, x, None, x, x, None) == 0
        both()
        n, held = d.lib.double_mallocs(), d.lib.double_held()
        for _ in range(3):
            both()
        assert (d.lib.double_mallocs(), d.lib.double_held()) == (n, held), sizes


class RtArgs(ctypes.Structure):     # the first members of the transfer's argument
    _fields_ = [(n, ctypes.c_int) for n in ("ncol", "col0", "ntile", "rcol0", "rncol")]


class MicroTile(ctypes.Structure):  # and of the microphysics'
    _fields_ = ([(n, ctypes.c_int) for n in ("ncol", "col0", "ntile", "der", "rcol0", "rncol")] +
                [("atm", ctypes.c_void_p), ("micro", ctypes.c_void_p)])


def case_transfer_indices_in_32_bits():
    """A transfer launch numbers its lanes in 32 bits and its work-items fit
    the launch, whatever tile is set; the launches cover the map once."""
    import numpy as np
    from firtez_dz_amd import gpu, lines
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    d.watch["rt_kernel"] = lambda x: (x.arg(0, RtArgs), x.grid * x.block)
    for widths, ncol, nodes in (((8192,), 262144, False), ((1024,) * 8, 262145, False), ((1,), 4000000, False),
                                ((8192,), 262144, True)):
        ctx.configure(lines.setup([((4,), n, -1.0 * n, 2.0) for n in widths]), np.arange(2) * 30.0)
        ctx._check(ctx.lib.fz_set_tile(ctx.h, 1 << 24, 64), "tile")
        atm, stokes = d.malloc(12 * 2 * 4 * ncol), d.malloc(16 * ctx.numw * ncol)
        d.seen.clear()
        if nodes:
            ctx.set_inversion(gpu.inversion({"T": 1}))
            assert ctx.lib.fz_forward_nodes_dev(ctx.h, ncol, atm, stokes, stokes, None, None) == 0
        else:
            assert ctx.lib.fz_forward_dev(ctx.h, ncol, atm, gpu.RF_NONE, stokes, None, None, None) == 0
        d.free(atm)
        d.free(stokes)
        col = 0
        for a, items in d.seen:
            assert a.col0 == col and a.ntile > 0 and a.ntile * max(widths) + 64 < 2 ** 31 and items < 2 ** 32
            col += a.ntile
        assert col == ncol


def case_maps_whose_records_exceed_the_memory():
    """Twelve million columns of 96 heights: model, profiles and the rest fit
    the card, the records of all columns (355 GB) do not.  Every column's
    records are written before they are read, inside their buffer."""
    import numpy as np
    from firtez_dz_amd import gpu, lines
    d = hostdouble.load()
    nz, ncol = 96, 12000000
    ctx = d.gpu.Context(0)
    d.watch = {"opac_kernel": lambda x: ("w", x.arg(0, MicroTile)), "tau_kernel": lambda x: ("w", x.arg(0, MicroTile)),
               "rt_kernel": lambda x: ("r", x.arg(0, RtArgs)), "taulin": lambda x: ("r", x.arg(0, RtArgs))}
    atm = d.malloc(12 * nz * 4 * ncol)
    for call in ("synthesis", "nodes", "pressure", "line_tau", "small"):
        if call == "small":
            ncol = 300
        ctx.configure(lines.fe6301_6302(nwave=2 if call == "line_tau" else 56), np.arange(nz) * 15.0)
        out = d.malloc(4 * ncol * (nz * 2 if call == "line_tau" else 4 * 56))
        eqv = d.malloc(4 * ncol * 4 * 56) if call in ("nodes", "pressure") else None
        d.seen.clear()
        if eqv:
            ctx.set_inversion(gpu.inversion({"T": 1} if call == "nodes" else {"Pg": 1}))
            rc = ctx.lib.fz_forward_nodes_dev(ctx.h, ncol, atm, out, eqv, None, None)
            d.free(eqv)
        elif call == "line_tau":
            rc = ctx.lib.fz_line_tau_dev(ctx.h, ncol, atm, out, None, None)
        else:
            rc = ctx.lib.fz_forward_dev(ctx.h, ncol, atm, gpu.RF_NONE, out, None, None, None)
        assert rc == 0, (call, ctx.lib.fz_last_error(ctx.h))
        d.free(out)
        held, done, written = (0, 0), 0, 0      # held: the columns now in the records
        for kind, a in d.seen:
            lo, hi = a.rcol0, a.rcol0 + a.rncol
            assert a.ncol == ncol and lo <= a.col0 and a.col0 + a.ntile <= hi
            if kind == "w":
                assert d.lib.double_size(a.micro) >= 77 * 4 * nz * a.rncol
                held = (min(held[0], a.col0) if held[0] >= lo else a.col0, a.col0 + a.ntile)
                written = max(written, a.col0 + a.ntile)
            else:
                assert held[0] <= a.col0 and a.col0 + a.ntile <= held[1] and a.col0 == done, call
                done += a.ntile
        assert done == written == ncol, call


def case_inversion_that_was_not_set():
    """After a refused or failed fz_set_inversion nothing is launched from
    what it left half set; the next one that succeeds holds again."""
    import numpy as np
    from firtez_dz_amd import gpu, lines
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    ctx.configure(lines.fe6301_6302(nwave=16), np.arange(32) * 30.0)
    atm, out, eqv = (d.malloc(1 << 24) for _ in range(3))
    good = gpu.inversion({"T": 4, "Bz": 2, "vz": 1})
    d.watch["rt_kernel"] = lambda x: x.name

    def forward():
        return ctx.lib.fz_forward_nodes_dev(ctx.h, 10, atm, out, eqv, None, None)

    for bad in (gpu.inversion({"T": 4, "vz": 33}), gpu.inversion({"T": 4}, invstk=(0, 0, 0, 0)),
                gpu.inversion({"T": 4}, solver=9), None):
        ctx.set_inversion(good)
        assert forward() == 0
        n = len(d.seen)
        if bad is None:     # no memory for larger tables
            d.lib.double_fail_after(0)
        try:
            ctx.set_inversion(bad or gpu.inversion({p: 16 for p in ("T", "Bx", "By", "Bz", "vz")}))
            raise AssertionError("accepted")
        except gpu.FzError:
            pass
        d.lib.double_fail_after(-1)
        assert forward() != 0 and len(d.seen) == n
    ctx.set_inversion(good)
    assert forward() == 0
    # the tables' buffer is kept
    n = d.lib.double_mallocs()
    for _ in range(3):
        ctx.set_inversion(good)
        ctx.set_inversion(gpu.inversion({"T": 3}))
    ctx.set_inversion(good)
    assert d.lib.double_mallocs() == n
    # the tables are those of one height and wavelength grid
    for nwave, nz, same in ((16, 40, False), (17, 32, False), (16, 32, True)):
        ctx.configure(lines.fe6301_6302(nwave=nwave), np.arange(nz) * 30.0)
        n = len(d.seen)
        assert (forward() == 0) == same and (len(d.seen) > n) == same


def case_network_gradient_of_many_rows():
    """The gradient of twenty million rows fits the card beside its data, as
    sums over parts of the batch."""
    import numpy as np
    from firtez_dz_amd import lines
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    ctx.configure(lines.fe6301_6302(), np.arange(64) * 15.0)
    ctx.mlp_create(448, 512, 3, 4)
    n = 20000000
    x, t = d.malloc(4 * 448 * n), d.malloc(4 * 20 * n)
    d.watch["mlp_input"] = lambda a: ("x", a.arg(0, ctypes.c_int).value, a.arg(2, ctypes.c_void_p).value)
    d.watch["mlp_dw"] = lambda a: ("dw",)
    ctx._check(ctx.lib.fz_mlp_gradient_dev(ctx.h, n, x, t, None, None, None, None), "gradient")
    row = 0
    for k in d.seen:
        if k[0] == "x":
            assert k[2] == x + 4 * 448 * row
            row += k[1]
    assert row == n and sum(k[0] == "dw" for k in d.seen) == sum(k[0] == "x" for k in d.seen)


def case_network_outputs_over_its_inputs():
    """The forward pass of all layers in one launch is not taken where its
    outputs would overwrite inputs that other workgroups have yet to read."""
    import numpy as np
    from firtez_dz_amd import lines
    d = hostdouble.load()
    ctx = d.gpu.Context(0)
    ctx.configure(lines.fe6301_6302(nwave=16), np.arange(32) * 30.0)
    ctx.mlp_create(64, 100, 2, 3)
    d.watch["mlp_"] = lambda x: "infer" in x.name
    n, p = 1000, d.malloc(1 << 22)
    base = p + (1 << 20)
    for x, xd, nx in ((base, None, 4 * 64 * n), (None, base, 8 * 64 * n)):
        for y, one in ((base, False), (base + 4, False), (base + nx - 4, False), (base + nx, True),
                       (base - 4 * 15 * n, True), (base - 4 * 15 * n + 4, False)):
            d.seen.clear()
            assert ctx.lib.fz_mlp_forward_dev(ctx.h, n, x, xd, y, None) == 0
            assert d.seen == [True] if one else not any(d.seen), (y - base, d.seen)


CASES = [n[5:] for n in list(globals()) if n.startswith("case_")]


@pytest.mark.parametrize("case", CASES)
def test_host(case):
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path[:0] = [ROOT, os.path.join(ROOT, "tests")]
    import hostdouble
    globals()["case_" + sys.argv[1]]()
