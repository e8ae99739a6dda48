"""No kernel of the built library has a private segment (registers spilled to memory): the first launch of one that has
on a stream makes the runtime allocate it, 130 us that a context's first call would pay."""
import os
import re

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gaugefields.jl_amd", "libgfhip.so")


def msgpack_uint(b, at):
    if b[at] < 0x80:
        return b[at]
    width = {0xCC: 1, 0xCD: 2, 0xCE: 4}[b[at]]
    return int.from_bytes(b[at + 1:at + 1 + width], "big")


def test_no_private_segments():
    b = open(LIB, "rb").read()
    key = b".private_segment_fixed_size"
    sizes = [msgpack_uint(b, m.end()) for m in re.finditer(re.escape(key), b)]
    assert len(sizes) > 100  # the kernels' metadata is there and readable
    assert not any(sizes), sorted(s for s in sizes if s)
