"""Host arrays in and out of the device: every number back where it came from, at sizes around a wave, a slot of the
pinned ring and the whole ring, and the SU(3) check over all links.

FP64: rows 0 and 1 and the momenta bit for bit; row 2 is rebuilt from them, a few roundings of numbers up to 1
(1e-15 each).  FP32: the numbers are rounded once, row 2 is rebuilt in double from the rounded rows.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_links(rng, n):
    """n Haar-like SU(3) matrices, (n, 9) column-major"""
    z = rng.standard_normal((n, 3, 3)) + 1j * rng.standard_normal((n, 3, 3))
    r0 = z[:, 0] / np.linalg.norm(z[:, 0], axis=1)[:, None]
    r1 = z[:, 1] - np.sum(z[:, 1] * r0.conj(), axis=1)[:, None] * r0
    r1 -= np.sum(r1 * r0.conj(), axis=1)[:, None] * r0
    r1 /= np.linalg.norm(r1, axis=1)[:, None]
    m = np.stack([r0, r1, np.cross(r0, r1).conj()], axis=1)
    return m.transpose(0, 2, 1).reshape(n, 9)


def rows(U, k):
    return U.reshape(U.shape[:-1] + (3, 3))[..., k]  # [..., j, i]: column-major


@pytest.mark.parametrize("dims,precision", [
    ((1, 1, 1, 1), "f64"), ((5, 3, 2, 1), "f32"), ((9, 7, 1, 1), "f64"), ((13, 5, 1, 1), "f32force"),
    ((8, 8, 8, 7), "f64"),       # a slot less than the single copy's sizes, groups that straddle slots
    ((13, 11, 7, 10), "f64"),    # no whole groups
    ((18, 18, 10, 9), "f32"),    # links above, momenta below the size of a single copy up
    ((33, 20, 18, 10), "f64"),   # several times round the ring
    ((24, 24, 24, 10), "f32force"),
])
def test_host_arrays(gf, dims, precision):
    print(f"[transfer] {dims} {precision}", flush=True)
    rng = np.random.default_rng(17)
    V = int(np.prod(dims))
    U = random_links(rng, 4 * V).reshape(4, V, 9)
    P = rng.standard_normal((4, V, 8))
    single = precision == "f32"
    U1 = U.astype(np.complex64).astype(np.complex128) if single else U
    P1 = P.astype(np.float32).astype(np.float64) if single else P
    with gf.Lattice(dims, precision=precision) as L:
        for _ in range(2):  # the second pass finds the ring and the staging there
            L.upload_links(U)
            L.upload_momenta(P)
            W = L.download_links()
            assert np.array_equal(rows(W, 0), rows(U1, 0)) and np.array_equal(rows(W, 1), rows(U1, 1))
            r2 = np.cross(rows(U1, 0), rows(U1, 1)).conj()
            assert np.abs(rows(W, 2) - r2).max() <= 1e-15 * 4
            assert np.array_equal(L.download_momenta(), P1)
        # a refused configuration leaves the links as they were, and the worst of all links is named
        bad = U.copy()
        bad[3, V - 1, 0] += 3e-3
        bad[0, V // 2, 0] += 1e-3
        with pytest.raises(Exception, match=f"direction 4, site {V - 1} "):
            L.upload_links(bad)
        bad[2, V // 3, 4] = np.nan
        with pytest.raises(Exception, match=f"direction 3, site {V // 3} .* by nan"):
            L.upload_links(bad)
        assert np.array_equal(L.download_links(), W)


def test_densities_come_down_whole(gf):
    """the plain arrays: below and above the size of a single copy, against sums that stay on the device"""
    for dims in ((12, 12, 12, 12), (30, 26, 25, 11)):
        with gf.Lattice(dims) as L:
            L.hot_start(3)
            q = L.topological_charge_density("plaquette")
            assert q.sum() == pytest.approx(L.topological_charge("plaquette"), rel=1e-9, abs=1e-9)
            S = L.action_untraced(1.0)
            assert np.trace(S, axis1=1, axis2=2).real.sum() == pytest.approx(2 * L.plaquette_sum(), rel=1e-12)
