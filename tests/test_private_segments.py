"""The private segments of the built kernels.  The runtime backs a kernel's private segment on the hardware queue it
runs on, for every wave the chip could hold (bytes a lane x 64 lanes x 32 waves x 256 CUs), within 8 x 4 GB of address
space for all queues: three queues at the limit below hold 16.1 GB and leave one 18.2 GB.  Kernels beyond the limit run
on one stream of the device (wide_scratch.h), chosen by their class where they are launched; every other kernel that
the compiler gives such a segment has to be found here, before it is launched from several contexts."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG

LIMIT = 10240  # bytes a lane
LANES = 64 * 32 * 256
APERTURE = 8 * (4 << 30)
# k_gblock<3,2,2,2> (fd|dd) of the gradient, k_dfblock<3,3,4,0> (ff|g) of the density fitting
WIDE = {"k_gblockILi3ELi2ELi2ELi2EE", "k_dfblockILi3ELi3ELi4ELi0EE"}
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(path):
    """The gfx950 ELF images of the offload bundles in a shared library built here."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count):
            off, size, ids = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + ids].decode()
            pos += 24 + ids
            if "gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 1)


@pytest.fixture(scope="module")
def segments(tmp_path_factory):
    lib = os.path.join(PKG, "libhfg.so")
    if not (os.path.exists(lib) and os.path.exists(READELF)):
        pytest.skip("no built library, or no readelf")
    out = {}
    for i, image in enumerate(code_objects(lib)):
        f = str(tmp_path_factory.mktemp("co") / ("%d.elf" % i))
        open(f, "wb").write(image)
        notes = subprocess.run([READELF, "--notes", f], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"\n  - \.a", notes)[1:]:
            name, size = re.search(r"\.name:\s+(\S+)", k), re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)
            if name and size:
                out[name.group(1)] = int(size.group(1))
    return out


def test_large_private_segments_are_the_known_ones(segments):
    assert len(segments) > 200
    wide = {n: s for n, s in segments.items() if s > LIMIT}
    assert {w for w in WIDE if any(w in n for n in wide)} == WIDE, wide
    assert all(any(w in n for w in WIDE) for n in wide), wide
    # their largest beside the limit on the other three queues, with room to spare for fragments
    assert (max(wide.values()) + 3 * LIMIT) * LANES < 0.75 * APERTURE
