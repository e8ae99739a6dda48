"""Measurements on a device whose memory other programs hold: the context's own fields have to do."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fill(hip, piece):
    """device memory in pieces down to `piece` bytes, until there is no such piece any more"""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    held, size = [], free.value - 64 * piece
    while size >= piece:
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
            held.append(p)
        else:
            hip.hipGetLastError()
            size = max(size // 2, piece) if size > piece else 0
    return held


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_field_strengths_without_free_memory(gf, precision):
    """24^3x20 links: their ping-pong partner (106 MB in FP64, 53 MB in FP32) holds at least a t-slice of the improved
    charge's fields (27 MB), the free memory none; the numbers are those of a context that had its usual buffer, added up
    over other blocks (1e-12)"""
    print(f"[full device] {precision}", flush=True)
    dims = (24, 24, 24, 20)

    def measure(L):
        return (L.topological_charge_density("improved"), L.topological_charge("improved"), L.energy_density_clover(),
                L.topological_charge("clover"))

    hip = ctypes.CDLL("libamdhip64.so.7")  # the one that the library has loaded
    with gf.Lattice(dims, precision=precision) as L:
        L.hot_start(5)
        want = measure(L)
    with gf.Lattice(dims, precision=precision) as L:
        L.hot_start(5)
        L.topological_charge_density("plaquette")
        held = L.device_bytes()
        filler = fill(hip, 16 << 20)
        try:
            got = measure(L)
            assert L.device_bytes() == held  # no buffer was to be had
        finally:
            for p in filler:
                assert hip.hipFree(p) == 0
    for a, b in zip(got, want):
        assert np.abs(np.asarray(a) - b).max() <= 1e-12 * max(1.0, np.abs(b).max())
