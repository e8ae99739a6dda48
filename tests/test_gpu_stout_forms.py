"""The stout kernels in the forms that lattices beyond the smallest take, against the CPU oracle.

Extents: one small lattice (at most 160 groups of 64 sites in FP64, 256 in FP32), whole rows (NX divides 64, V a multiple
of 64) and rows cut by the groups with idle lanes, above both limits.
"""
import ctypes

import numpy as np
import pytest

import lattice_tools as lt

pytestmark = pytest.mark.gpu

gen = lt.gen
SMALL, ROWS, CUT = (8, 8, 8, 8), (16, 16, 16, 6), (18, 10, 10, 10)


def links(oracle, dims, seed, spread=0.3):
    U = gen.cold_links(dims)
    oracle.exp_update(dims, U, gen.algebra_coefficients(dims, spread, seed), 1.0)
    return U


# One FP32 level at rho = 1, where the error of Q outweighs the rounding of the stored link (1e-8): RMS of rows 0 and 1
# against the FP64 level of the same float links.  A numpy emulation of the kernel's products on such links (float FMAs
# for the staples, the product with U, the TA projection and the sum in double) gives 5.0e-8, with the products, TA and
# the sum in float as well 7.7e-8; the bar lies 1.2 above the first.
@pytest.mark.parametrize("dims", [SMALL, ROWS, CUT])
def test_fp32_level_forms_q_in_double(gf, oracle, dims):
    print(f"[stout] FP32 level {dims}", flush=True)
    with gf.Lattice(dims, precision="f32") as L:
        L.upload_links(links(oracle, dims, 71))
        U = L.download_links()
        L.stout_config(1, 1.0, "store")
        S = L.stout_smear()
    d = (S - oracle.stout_smear(dims, U, 1, 1.0)).reshape(4, -1, 3, 3)[..., :2]  # [.., j, i]: column-major
    assert np.sqrt(np.mean(np.abs(d) ** 2)) < 1.2 * 5.03e-8


def backward(oracle, dims, U, nlev, rho, D):
    for l in range(nlev, 0, -1):
        D = oracle.stout_backward(dims, oracle.stout_smear(dims, U, l - 1, rho) if l > 1 else U, rho, D)
    return D


# The explicit backward pass above the small lattices' limits: the top level's site-local step, the staple part with and
# without the next level's step behind it, and Q kept by the smearing, formed again (recompute), and formed again because
# the Hamiltonian has smeared the links anew.  FP64: 1e-13 a level, as at 4^4; FP32: 2e-5 of the largest element, the bar of
# the three-level force.
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("dims", [SMALL, ROWS, CUT, (131, 3, 7, 6)])
@pytest.mark.parametrize("nlev,rho", [(1, 0.5), (3, 0.12)])
def test_explicit_backward(gf, oracle, dims, precision, nlev, rho):
    print(f"[stout] backward {dims} {precision} {nlev}", flush=True)
    D = gen.hot_start_links(dims, 43)
    with gf.Lattice(dims, precision=precision) as L:
        L.upload_links(links(oracle, dims, 42))
        U = L.download_links()
        ref = backward(oracle, dims, U, nlev, rho, D)
        bar = nlev * 1e-13 if precision == "f64" else 2e-5 * np.abs(ref).max()
        L.stout_config(nlev, rho, "store")
        L.stout_smear(download=False)
        assert np.abs(L.stout_backward(D) - ref).max() < bar
        L.hamiltonian(3.0)
        assert np.abs(L.stout_backward(D) - ref).max() < bar
        L.stout_config(nlev, rho, "recompute")
        L.stout_smear(download=False)
        assert np.abs(L.stout_backward(D) - ref).max() < bar


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_backward_pass_of_links_changed_since_the_smearing(gf, oracle, precision):
    """One level needs nothing of the smearing but the links it started from: back_prop then belongs to the links as they
    are, also where Q has been kept from earlier ones"""
    print(f"[stout] backward of changed links {precision}", flush=True)
    dims, rho = ROWS, 0.2
    D = gen.hot_start_links(dims, 43)
    with gf.Lattice(dims, precision=precision) as L:
        A, B = links(oracle, dims, 42), links(oracle, dims, 44)
        L.upload_links(A)
        L.gaussian_momenta(5)
        L.save_links()
        L.stout_config(1, rho, "store")
        changes = {
            "upload": lambda: L.upload_links(B),
            "cold": L.set_cold,
            "hot": lambda: L.hot_start(3),
            "links from algebra": lambda: L.links_from_algebra(gen.algebra_coefficients(dims, 0.3, 46)),
            "exp update": lambda: L.exp_update(0.1),
            "md update": lambda: L.md_update(3.0, 0.1, 0.1),
            "trajectory": lambda: L.md_trajectory(3.0, 2, 0.1),
            "restore": L.restore_links,
            "heatbath": lambda: L.heatbath(5.5, 1, 2),
            "overrelaxation": lambda: L.overrelaxation(1, 2),
            "flow": lambda: L.flow(0.02, 1),
        }
        for name, change in changes.items():
            L.stout_smear(download=False)
            change()
            U = L.download_links()
            ref = oracle.stout_backward(dims, U, rho, D)
            bar = 1e-13 if precision == "f64" else 2e-5 * np.abs(ref).max()
            assert np.abs(L.stout_backward(D) - ref).max() < bar, name
        if precision == "f64":  # links that are SU(3) to float rounding only: as recompute mode does it, which keeps no Q
            L.stout_smear(download=False)
            L.round_to_float(links=True)
            din = L.stout_backward(D)
            L.stout_config(1, rho, "recompute")
            assert np.array_equal(din, L.stout_backward(D))


def test_auto_mode_leaves_room_for_back_prop(gf):
    """11.5 GB free where three levels with Q and the force's buffers take 10.1 GB, without Q 8.5 GB, and the explicit
    backward pass 1.8 GB more: auto has to choose recompute, and back_prop to work"""
    dims = (32, 32, 32, 96)
    with gf.Lattice(dims) as L:
        hip = ctypes.CDLL("libamdhip64.so.7")  # the one that the library has loaded
        free, total, filler = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_void_p()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        assert hip.hipMalloc(ctypes.byref(filler), ctypes.c_size_t(free.value - int(11.5e9))) == 0
        try:
            L.stout_config(3, 0.1, "auto")
            assert L.stout_mode() == "recompute"
            L.stout_smear(download=False)
            D = L.stout_backward(np.zeros((4, int(np.prod(dims)), 9), complex))
        finally:
            assert hip.hipFree(filler) == 0
    assert not D.any()


# Above 512 groups the pair kernel runs with four waves and the gather with whole workgroups: whole rows (640 groups) and
# rows cut by the groups with idle lanes (552).  The force, and the fused kick and link update of the force's last kernel.
# FP64: 1e-12; float forces: 2e-6 (plain) and 2e-5 (two levels) of the largest, as on the smaller lattices.  In the
# FP32-force form the links and momenta are FP64: the update agrees with the oracle's from the same momenta to 1e-13.
@pytest.mark.parametrize("precision", ["f64", "f32", "f32force"])
@pytest.mark.parametrize("dims", [(16, 16, 16, 10), (18, 14, 14, 10)])
@pytest.mark.parametrize("nlev", [0, 2])
def test_updates_of_larger_lattices(gf, oracle, dims, precision, nlev):
    print(f"[stout] updates {dims} {precision} {nlev}", flush=True)
    coeff, rho = 3.0, 0.1
    bar = 1e-12 if precision == "f64" else (2e-5 if nlev else 2e-6)
    P = gen.gaussian_momenta(dims, 72)
    with gf.Lattice(dims, precision=precision) as L:
        L.upload_links(links(oracle, dims, 71))
        L.upload_momenta(P)
        U, P = L.download_links(), L.download_momenta()
        F = oracle.stout_force(dims, U, nlev, rho, coeff) if nlev else oracle.force(dims, U, coeff)
        top = np.abs(F).max()
        for mode in ("store", "recompute") if nlev else ("store",):
            L.stout_config(nlev, rho, mode)
            L.upload_links(U)
            L.upload_momenta(P)
            L.force(coeff)
            assert np.abs(L.download_force() - F).max() < bar * top
            L.force_kick(coeff, 0.02)
            P1 = P + 0.02 * F
            assert np.abs(L.download_momenta() - P1).max() < bar * np.abs(P1).max()
            L.md_update(coeff, 0.03, 0.04)
            P1 += 0.03 * F
            got = L.download_momenta()
            assert np.abs(got - P1).max() < bar * np.abs(P1).max()
            U1 = U.copy()
            oracle.exp_update(dims, U1, got, 0.04)
            assert np.abs(L.download_links() - U1).max() < (2e-6 if precision == "f32" else 1e-13)
