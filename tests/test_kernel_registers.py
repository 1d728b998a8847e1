"""Scratch memory of the built FP64 kernels: register spills in the passes whose
registers are tuned against their occupancy show up as a private segment in the
code objects' metadata (read from the library this repository builds)."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(__file__), "..", "kfft_amd", "lib", "libkfft_amd.so")


def kernels():
    """{mangled name: metadata} of every gfx950 code object in the library."""
    data = open(LIB, "rb").read()
    out = {}
    for m in re.finditer(rb"\x7fELF\x02\x01\x01\x40", data):  # (64-bit, ABI: AMDGPU HSA)
        at = m.start()
        shoff, = struct.unpack_from("<Q", data, at + 0x28)
        shentsize, shnum = struct.unpack_from("<HH", data, at + 0x3A)
        for i in range(shnum):
            _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", data, at + shoff + i * shentsize)
            if kind != 7:  # SHT_NOTE
                continue
            pos, end = at + off, at + off + size
            while pos < end:
                namesz, descsz, note = struct.unpack_from("<III", data, pos)
                desc = pos + 12 + (namesz + 3) // 4 * 4
                if note == 32:  # NT_AMDGPU_METADATA
                    meta = msgpack.unpackb(data[desc:desc + descsz])
                    for k in meta["amdhsa.kernels"]:
                        out[k[".name"]] = k
                pos = desc + (descsz + 3) // 4 * 4
    return out


@pytest.fixture(scope="module")
def table():
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    return kernels()


# name pattern -> bytes of scratch a thread may use
@pytest.mark.parametrize("pattern,limit", [
    (r"k_fftIdLi16ELi0ELi0E", 16),        # the general pass, radices up to 16
    (r"k_mixgenIdLi\d+ELi\d+ELb[01]E", 64),  # shaped passes behind the general IO
])
def test_fp64_passes_do_not_spill(table, pattern, limit):
    found = {n: k[".private_segment_fixed_size"] for n, k in table.items() if re.search(pattern, n)}
    assert found, pattern
    over = {n: b for n, b in found.items() if b > limit}
    assert not over
