"""What the built kernels take: the code object's own metadata (the AMDGPU
note of each device image in liblgml_hip.so), no GPU needed."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def kernels():
    """Name -> metadata of every kernel of the library."""
    from lgml_amd import build, hip
    if not os.path.exists(hip.LIB_PATH):
        build.build()
    data = open(hip.LIB_PATH, "rb").read()
    out, at = {}, data.find(b"AMDGPU\0")
    while at >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", data, at - 12)
        if namesz == 7 and kind == 32:  # NT_AMDGPU_METADATA
            note = msgpack.unpackb(data[at + 8:at + 8 + descsz])
            for k in note.get("amdhsa.kernels", []):
                out[k[".name"]] = k
        at = data.find(b"AMDGPU\0", at + 1)
    return out


@pytest.mark.parametrize("name", ["get_rows_kernel", "swiglu_kernel", "swiglu_split_kernel",
                                  "splitk_reduce_kernel", "xsplit_kernel", "moe_sum_kernel",
                                  "rms_norm_kernel", "qkv_rope_store_kernel", "merge_kernel"])
def test_row_kernels_keep_their_values_in_registers(name):
    """The kernels between the products use no scratch memory (a spill there
    is one more pass over memory for each of a prompt chunk's rows)."""
    got = {n: k for n, k in kernels().items() if name in n}
    assert got
    for n, k in got.items():
        assert k[".private_segment_fixed_size"] == 0 and k.get(".vgpr_spill_count", 0) == 0, n


def test_grouped_wide_tiles_spill_next_to_nothing():
    """The 64-column grouped products run at 256 registers: Q8_0 with split X
    spills three, the others none (twelve made it a quarter slower)."""
    got = {n: k for n, k in kernels().items() if "qgemm_kernelILi" in n and "ELi4ELb1E" in n}
    assert len(got) == 6
    for n, k in got.items():
        q80_exact = "ILi8ELi4ELb1ELb0E" in n
        assert k[".private_segment_fixed_size"] <= (16 if q80_exact else 0), n
