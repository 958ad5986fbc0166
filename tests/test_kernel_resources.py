"""What the built library's kernels take of the GPU, from the metadata the compiler writes into it."""
import re
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


def test_node_form_keeps_its_values_in_registers(kernels):
    """4 waves per SIMD leave 128 registers; a variant that spills loses more than the form gains."""
    spilled = {k: v[".private_segment_fixed_size"] for k, v in instances(kernels, "k_volume_node").items()
               if v[".private_segment_fixed_size"]}
    assert not spilled


DEFAULT = {False: {2: 7, 3: 1, 4: 2, 5: 1}, True: {2: 7, 3: 4, 4: 5, 5: 3}}  # by FP32-split
TILES = {2: (7, 14, 3), 3: (4, 2, 8), 4: (5, 2, 3), 5: (3, 1, 2)}  # elements per block, those that the tuner may set


def test_volume_kernels_are_those_a_launch_can_take(kernels):
    """One tile per degree and precision, the default; the LSERK form with flux 32 all of the degree's
    (a further one, 1, in FP64 at N = 3).  FP64 runs the node form from N = 3 on, FP32-split the line form."""
    RK, seen = 1, set()
    for name in list(instances(kernels, "k_volume")) + list(instances(kernels, "k_volume_node")):
        m = re.match(r"_ZN2fx\d+k_volume(_node)?ILi(\d)ELi(\d+)ELb([01])ELi(\d)E([fd])?Li(\d+)EE", name)
        node, (N, flux, para, mode), vr, epb = m[1], map(int, m.group(2, 3, 4, 5)), m[6], int(m[7])
        fp32 = vr == "f"
        assert bool(node) == (N >= 3 and not fp32), name
        if fp32:
            assert flux in (0, 5, 10, 32), name
        if mode == RK and flux == 32:
            assert epb in TILES[N] or (N == 3 and not fp32 and epb == 1), name
        else:
            assert epb == DEFAULT[fp32][N], name
        seen.add((N, flux, para, mode, fp32))
    forms = [(0, 0), (1, 0), (0, 1), (1, 1), (0, 2)]  # (parabolic, mode)
    assert seen == {(N, f, p, m, prec) for N in TILES for f in (*range(11), 32) for p, m in forms
                    for prec in ((False, True) if f in (0, 5, 10, 32) else (False,))}
