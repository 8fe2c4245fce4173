"""What the compiler made of kernels whose speed hangs on their registers: no scratch memory.  Read from the kernels' own metadata in the built library."""
import re
import struct

import msgpack
import pytest

from pipeinfer_amd import lib as L


def scratch_of_kernels():
    """{kernel's symbol: bytes of scratch memory per lane}, from the code objects for gfx950 in the library"""
    L.load()
    with open(L.SO, "rb") as f:
        data = f.read()
    found = {}
    for at in (m.start() for m in re.finditer(b"\x7fELF\x02\x01", data)):
        if struct.unpack_from("<H", data, at + 18)[0] != 224:                 # (EM_AMDGPU)
            continue
        sections, size, count = struct.unpack_from("<Q", data, at + 40)[0], *struct.unpack_from("<HH", data, at + 58)
        for i in range(count):
            kind, = struct.unpack_from("<I", data, at + sections + i * size + 4)
            start, length = struct.unpack_from("<QQ", data, at + sections + i * size + 24)
            if kind != 7:                                                     # (SHT_NOTE)
                continue
            p, end = at + start, at + start + length
            while p < end:
                name, desc, note = struct.unpack_from("<III", data, p)
                body = p + 12 + (name + 3) // 4 * 4
                if note == 32:                                                # (NT_AMDGPU_METADATA)
                    for k in msgpack.unpackb(data[body:body + desc])["amdhsa.kernels"]:
                        found[k[".name"]] = k[".private_segment_fixed_size"]
                p = body + (desc + 3) // 4 * 4
    return found


@pytest.mark.parametrize("kernel", ["k_rms_scale_once", "k_prompt_attention", "k_split_attention", "k_latent_split", "k_linear_step", "k_channel_step", "k_rms_post4"])
def test_kernels_without_scratch_memory(kernel):
    mine = {n: s for n, s in scratch_of_kernels().items() if kernel in n}
    assert mine and not any(mine.values()), mine
