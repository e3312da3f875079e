"""Register spills of the kernels that sit at the register limit, from the metadata
of the code objects in the built library (no GPU)."""
import struct

import pytest


def _kernels(path):
    """The kernel entries (dicts) of every gfx950 code object in the file: the
    AMDGPU metadata notes, msgpack maps."""
    msgpack = pytest.importorskip("msgpack")
    data = open(path, "rb").read()
    out, at = [], data.find(b"AMDGPU\0\0")
    while at >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", data, at - 12)
        if (namesz, kind) == (7, 32):
            out += msgpack.unpackb(data[at + 8:at + 8 + descsz], strict_map_key=False)["amdhsa.kernels"]
        at = data.find(b"AMDGPU\0\0", at + 8)
    return out


# One-wave-per-SIMD prefill: all 512 registers.  The item's code inlined once per
# source of items spilled 28 of them (3 with one copy) and took up to 15 % longer on
# steps with more items than workgroups.
@pytest.mark.parametrize("kernel,most", [("prefill_w64_kernel", 8), ("prefill_wide8_kernel", 24)])
def test_vgpr_spills(vkv, kernel, most):
    found = [k for k in _kernels(vkv.LIB_PATH) if kernel in k[".name"]]
    assert found
    assert max(k[".vgpr_spill_count"] for k in found) <= most, found
