"""Vector registers of the drawn mask passes, from the built library's own kernel metadata.

These passes are bound by the random draw and run beside another stream's products: at 48
registers or fewer, eight of their waves leave a quarter of a SIMD's 512 to those products
(loads issued ahead of the draw cost 49 to 67 and made every pass slower)."""

import os
import re
import struct

import msgpack
import pytest

from param_decomp_amd import builder


def _kernels():
    """{mangled name: vector registers} over the gfx950 code objects inside the library."""
    with open(builder.LIB, "rb") as f:
        blob = f.read()
    out = {}
    for at in (m.start() for m in re.finditer(rb"\x7fELF\x02\x01\x01\x40", blob)):  # OS ABI 64: AMDGPU HSA
        shoff, = struct.unpack_from("<Q", blob, at + 0x28)
        shentsize, shnum = struct.unpack_from("<HH", blob, at + 0x3A)
        for i in range(shnum):
            _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", blob, at + shoff + i * shentsize)
            if kind != 7:  # SHT_NOTE
                continue
            p, end = at + off, at + off + size
            while p + 12 <= end:
                namesz, descsz, note = struct.unpack_from("<III", blob, p)
                desc = p + 12 + (namesz + 3) // 4 * 4
                if note == 32:  # NT_AMDGPU_METADATA
                    meta = msgpack.unpackb(blob[desc:desc + descsz], raw=False)
                    out.update((k[".name"], k[".vgpr_count"]) for k in meta["amdhsa.kernels"])
                p = desc + (descsz + 3) // 4 * 4
    return out


# template arguments: the draw's counter layout (0, 1; other forms do not draw) and the
# exponent mode; the backward's second one is "from a source table"
@pytest.mark.parametrize("pattern", [r"k_mask_fwd_tileILi[01]ELi\dE", r"k_lm_mask_fwdILi[01]ELi\dE",
                                     r"k_lm_mask_bwdILi\dELb0E"])
def test_drawn_mask_passes(pattern):
    if not os.path.exists(builder.LIB):
        pytest.skip("HIP library not built")
    found = {n: v for n, v in _kernels().items() if re.search(pattern, n)}
    assert len(found) in (4, 8)
    assert all(v <= 48 for v in found.values()), found
