"""What the built library says about its own kernels: the metadata that the
compiler writes for each one into the gfx950 code objects."""
import os
import struct

import pytest

import dage_amd._lib as lib

msgpack = pytest.importorskip("msgpack")

SO = os.path.join(os.path.dirname(lib.__file__), "libdage_ops.so")
NT_AMDGPU_METADATA = 32


def device_kernels():
    """The metadata entry of every kernel, from the note of each code object."""
    with open(SO, "rb") as f:
        data = f.read()
    out, at = [], data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            phoff, = struct.unpack_from("<Q", data, at + 32)
            phsize, phnum = struct.unpack_from("<HH", data, at + 54)
            for i in range(phnum):
                kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + i * phsize)
                p, end = at + off, at + off + size
                while kind == 4 and p + 12 <= end:  # PT_NOTE
                    nname, ndesc, ntype = struct.unpack_from("<III", data, p)
                    desc = p + 12 + (nname + 3) // 4 * 4
                    if ntype == NT_AMDGPU_METADATA:
                        out += msgpack.unpackb(data[desc:desc + ndesc])["amdhsa.kernels"]
                    p = desc + (ndesc + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)
    return out


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(SO):
        pytest.skip("the library is not built")
    return device_kernels()


@pytest.mark.parametrize("part", ["stream_xy_kernel", "stream_z_kernel", "conv_filter_mfma_kernel",
                                  "conv_filter_few_kernel"])
def test_no_register_spills(kernels, part):
    mine = [k for k in kernels if part in k[".name"]]
    assert mine
    for k in mine:
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, k[".name"]
