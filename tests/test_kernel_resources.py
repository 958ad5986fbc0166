"""What the built library's kernels take of the GPU, from the metadata the compiler writes into it."""
import struct

import msgpack
import pytest

from fluxo_amd import native

EM_AMDGPU, SHT_NOTE, NT_AMDGPU_METADATA = 224, 7, 32


def code_objects(data):
    at = data.find(b"\x7fELF\x02\x01")
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            yield at
        at = data.find(b"\x7fELF\x02\x01", at + 4)


def notes(data, at):
    shoff, = struct.unpack_from("<Q", data, at + 40)
    size, count = struct.unpack_from("<HH", data, at + 58)
    for i in range(count):
        section = struct.unpack_from("<IIQQQQ", data, at + shoff + i * size)
        if section[1] != SHT_NOTE:
            continue
        p, end = at + section[4], at + section[4] + section[5]
        while p < end:
            nname, ndesc, kind = struct.unpack_from("<III", data, p)
            desc = p + 12 + (nname + 3) // 4 * 4
            yield kind, data[desc:desc + ndesc]
            p = desc + (ndesc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    with open(native.LIB_PATH, "rb") as f:
        data = f.read()
    out = {}
    for at in code_objects(data):
        for kind, desc in notes(data, at):
            if kind == NT_AMDGPU_METADATA:
                for k in msgpack.unpackb(desc, raw=False, strict_map_key=False)["amdhsa.kernels"]:
                    out[k[".name"]] = k
    assert len(out) > 100
    return out


def instances(kernels, name):
    return {k: v for k, v in kernels.items() if k.startswith(f"_ZN2fx{len(name)}{name}I")}


def test_node_form_at_n3_keeps_its_values_in_registers(kernels):
    """4 waves per SIMD leave 128 registers; a variant that spills loses more than the form gains."""
    spilled = {k: v[".private_segment_fixed_size"] for k, v in instances(kernels, "k_volume_node").items()
               if "ILi3E" in k and v[".private_segment_fixed_size"]}
    assert not spilled
