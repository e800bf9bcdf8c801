"""Algorithmic work of the radiative-transfer kernel (rt_kernel in
csrc/fz_gpu.hip), counted from its source per (height, wavelength) and summed
to a per-(column, wavelength) figure used for the roofline.

Convention: add, sub, mul = 1; FMA = 2; div, sqrt, exp, log, sin, cos and a
hardware reciprocal = 1 each.  Loads/stores, selects, comparisons and integer
index arithmetic are not counted.  The counts are per non-boundary layer.
They were tallied by hand from the source of each device function (the
names below follow csrc/fz_rt.hpp and rt_kernel); change them together with
the kernel.  The evolution operator is counted in its series form, which nearly
all layers take.
"""
from __future__ import annotations

# per Zeeman component
VOIGT = 36           # u^2 (1); numerator 6 + 4, denominator 6 + 5 + 1, |den|^2 (3), reciprocal (1), H (4), F (5)
COMP_FWD = 2 + VOIGT + 4              # u, 2 accumulations (absorb)
COMP_DER = 2 + VOIGT + 12             # u, 6 moments (absorb_der)
# per component type (sigma_r, pi, sigma_b) of a line
TYPE_FWD = 2 + 4                      # u of the type's centre, 2 accumulations
TYPE_SUM = 32                         # dH/du, dH/da and their products with u and the shift from the moments
TYPE_SUM_ONE = 11                     # the same of a type with one component
TYPE_ACC = 24                         # value, T, v, |B| of absorption and dispersion
TYPE_ACC_PR = 16                      # Pg and rho
# per line
LINE_FWD = 5                          # kappa_l dz, shift, Doppler scale, field scale
LINE_DER = 14
LINE_DER_PR = 6
# per layer
MIX = 15 + 2                          # the five elements from the types' sums, with the continuum
SOURCE = 6                            # c2/T, exp, departure, -1, reciprocal, x c1
SOURCE_DER = 10                       # the same and dS/dT = S (ex/(ex-1)) (c2/T) / T
TURN = 6                              # into the layer's frame or back
EVOL_BUILD = 107                      # evol_build (series form): invariants, exp, four series, coefficients
EVOL_BUILD_DER = 103                  # their derivatives
PIECES = 40                           # evol_pieces
APPLY = 20                            # evol_apply
FORMAL = 1 + 2 * TURN + PIECES + APPLY + 9   # I_k = S + O (I_(k-1) - S)
GRAD = 218                            # evol_grad
GRAD_DOT = 36
AZIMUTH = 36
INCLINATION = 3 + MIX - 2 + GRAD_DOT
SOURCE_TERM = 18                      # (1-O) e0 dS/dT
CHAIN = 52                            # (|B|, inclination, azimuth) -> (Bx, By, Bz)
EXTEND = 28 + 4 * (2 * TURN + 28 + 8) # ACC in the frame, ACC <- ACC . O_k
PROPAGATE_PER_PARAM = 28              # ACC . local response


def per_layer(nlines: int, ncomp: int, nparam: int, ntriplet: int = 0) -> dict:
    """ntriplet: how many of the lines have one component per type."""
    ntype = 3 * nlines
    # a one-component type takes its centre's u
    ncu = ncomp - 3 * ntriplet
    fwd = (SOURCE + nlines * LINE_FWD + ncomp * COMP_FWD + ntype * TYPE_FWD + MIX + EVOL_BUILD + FORMAL)
    der = 0
    if nparam:
        pr = nparam == 7
        der = (SOURCE_DER + nlines * (LINE_DER + (LINE_DER_PR if pr else 0))
               + ncomp * VOIGT + ncu * (COMP_DER - VOIGT)
               + ntype * (2 + TYPE_ACC + (TYPE_ACC_PR if pr else 0))
               + 3 * (nlines - ntriplet) * TYPE_SUM + 3 * ntriplet * TYPE_SUM_ONE
               + MIX + EVOL_BUILD + EVOL_BUILD_DER + 1 + TURN + PIECES + GRAD
               + (3 + (2 if pr else 0)) * (MIX + GRAD_DOT) + AZIMUTH + INCLINATION
               + SOURCE_TERM + (CHAIN if pr else 0) + EXTEND + nparam * PROPAGATE_PER_PARAM)
    return {"pass1": fwd, "pass2": der, "total": fwd + der}


def per_column_lambda(nz: int, nlines: int, ncomp: int, nparam: int, ntriplet: int = 0) -> float:
    """FLOPs per (column, wavelength) over nz layers (boundary layer excluded)."""
    return (nz - 1) * per_layer(nlines, ncomp, nparam, ntriplet)["total"]


# bytes that must cross HBM per (column, wavelength): the Jacobian and Stokes
# written once, plus the per-height inputs amortised over the wavelengths
def bytes_per_column_lambda(nz: int, numw: int, nparam: int, nfield: int) -> float:
    out = 4 * 4 + nparam * nz * 4 * 4
    inp = (12 + nfield) * nz * 4 / numw
    return out + inp


# HBM traffic of rt_kernel<1> per column of the forward + Jacobian workload
# (nz = 96, 112 wavelengths, spherical Jacobian), from the FETCH_SIZE and
# WRITE_SIZE counters of one 32768-column launch (each scaled by its reading
# for a device copy of known size: FETCH_SIZE x2, WRITE_SIZE x1):
# (5.676e6 KiB x 2 + 3.309e7 KiB) x 1024 / 32768 columns
RT_HBM_BYTES_PER_COLUMN = 1.3887e6
RT_HBM_SOURCE = ("rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE of rt_kernel<1>, a 32768-column launch of this "
                 "workload, scaled per column (profiles/rt_kernel_fwd_jacobian_288x288x96.md)")
