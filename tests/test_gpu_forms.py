"""The stencil kernels on extents that cut rows and leave lanes idle, against the CPU oracle.

A 64-site group of consecutive sites cuts x-rows unless NX divides 64, needs x-neighbours outside
itself then, and the last one has idle lanes unless V is a multiple of 64; small lattices run a form
of their own (at most 160 groups in FP64, 256 in FP32).  The extents below lie on both sides of each
of these, with rows shorter and longer than a group.
"""
import numpy as np
import pytest

import lattice_tools as lt

pytestmark = pytest.mark.gpu

gen = lt.gen
COEFF = 3.0

DIMS = [
    (5, 3, 2, 1),      # 30 sites: one group, most lanes idle, a direction of one site
    (16, 10, 8, 8),    # 160 groups of whole rows: the last small FP64 lattice
    (24, 11, 5, 9),    # 186 groups, rows cut, lanes idle
    (16, 16, 8, 6),    # 192 groups of whole rows
    (66, 4, 9, 8),     # 297 groups, rows longer than a group
    (131, 3, 7, 6),    # the same with an odd row and idle lanes
    (18, 10, 10, 10),  # 282 groups, rows cut, idle lanes
]


def maxdiff(a, b):
    return float(np.abs(np.asarray(a) - np.asarray(b)).max())


# FP64: the bar of the other parity tests, relative 1e-12.  FP32: the float forces of float-rounded
# links, 2e-6 (plain) and 2e-5 (stout, two levels here) of the largest, as in the FP32 parity tests.
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("dims", DIMS)
def test_force_flow_and_stout_forms(gf, oracle, dims, precision):
    print(f"[forms] {dims} {precision}", flush=True)
    bar, sbar = (1e-12, 1e-12) if precision == "f64" else (2e-6, 2e-5)
    U = gen.cold_links(dims)
    oracle.exp_update(dims, U, gen.algebra_coefficients(dims, 0.3, 71), 1.0)
    P = gen.gaussian_momenta(dims, 72)
    with gf.Lattice(dims, precision=precision) as L:
        L.upload_links(U)
        L.upload_momenta(P)
        U, P = L.download_links(), L.download_momenta()
        F = oracle.force(dims, U, COEFF)
        L.force(COEFF)
        assert maxdiff(L.download_force(), F) < bar * np.abs(F).max()
        D = oracle.dsdu(dims, U, COEFF)
        assert maxdiff(L.dsdu(COEFF), D) < bar * np.abs(D).max()
        # kick and link update of every link, and of no lane past the last site
        L.md_update(COEFF, 0.02, 0.03)
        oracle.kick(dims, P, F, 0.02)
        assert maxdiff(L.download_momenta(), P) < bar * np.abs(P).max()
        U1 = U.copy()
        oracle.exp_update(dims, U1, P, 0.03)
        assert maxdiff(L.download_links(), U1) < max(bar, 1e-12)
        L.upload_links(U)
        L.stout_config(2, 0.1, "store")
        F = oracle.stout_force(dims, U, 2, 0.1, COEFF)
        for mode in ("store", "recompute"):
            L.stout_config(2, 0.1, mode)
            L.force(COEFF)
            assert maxdiff(L.download_force(), F) < sbar * np.abs(F).max()
        L.stout_config(0, 0.0)
        E = L.flow(0.02, 2, 1)
        Eref = oracle.flow(dims, U.copy(), 0.02, 2, 1)
        assert np.all(np.abs(E - Eref) < bar * np.abs(Eref))
