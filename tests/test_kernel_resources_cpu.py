"""What the compiler gave the built kernels, from the code objects inside the library: registers, scratch memory and static LDS that the launch rules count on."""
import os
import re
import struct

import msgpack
import pytest

from msnhnet_amd import build

EM_AMDGPU, SHT_NOTE = 224, 7


def _kernels():
    """name -> metadata of every kernel of libmsnh_hip.so (the msgpack note of each embedded code object)"""
    path = os.path.join(build.LIB, "libmsnh_hip.so")
    if not os.path.exists(path):
        build.build_all(verbose=False)
    data = open(path, "rb").read()
    out = {}
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            table, = struct.unpack_from("<Q", data, at + 40)
            entry, count = struct.unpack_from("<HH", data, at + 58)
            for i in range(count):
                head = at + table + i * entry
                if struct.unpack_from("<I", data, head + 4)[0] == SHT_NOTE:
                    note = at + struct.unpack_from("<Q", data, head + 24)[0]
                    name, desc = struct.unpack_from("<II", data, note)
                    note += 12 + (name + 3) // 4 * 4
                    for k in msgpack.unpackb(data[note:note + desc])["amdhsa.kernels"]:
                        out[k[".name"]] = k
        at = data.find(b"\x7fELF", at + 1)
    return out


@pytest.fixture(scope="module")
def kernels():
    return _kernels()


@pytest.fixture(scope="module")
def igemm(kernels):
    """(types, BM, BN, KV, WM, WN, NS, KG, tail) -> metadata of the implicit-GEMM kernels"""
    out = {}
    for n, k in kernels.items():
        m = re.match(r"_ZN4msnh15convIgemmKernelI(\w+?)((?:Li\d+E)+)E", n)
        if m:
            out[(m.group(1),) + tuple(int(v) for v in re.findall(r"Li(\d+)E", m.group(2)))] = k
    assert len(out) == 3 * 52 + 2           # 52 tiles in three pairs of types, and two with a tail
    return out


def test_igemm_kernels_have_no_static_lds_and_one_register_file(igemm):
    """The LDS of a workgroup is what the launch asks for -- tiles are sized so that a second one fits to the byte -- and no accumulators in the second half of a
    512-register file, which admits one wavefront per SIMD."""
    for key, k in igemm.items():
        assert k[".group_segment_fixed_size"] == 0 and k[".agpr_count"] == 0, key


def test_split_product_tiles_reach_their_occupancy(igemm):
    """float32 tiles of split products: two wavefronts per SIMD with 64 x 64 wave tiles, three with smaller ones of two blocks"""
    seen = 0
    for (types, bm, bn, kv, wm, wn, ns, kg, tail), k in igemm.items():
        blocks = (bm // wm // 32) * (bn // wn // 32)
        waves = wm * wn * kg
        if types != "ff" or blocks not in (2, 4) or bm // wm > 64 or bn // wn > 64 or (blocks == 4 and waves == 12):
            continue
        seen += 1
        assert k[".vgpr_count"] <= (256 if blocks == 4 else 168) and k[".vgpr_spill_count"] == 0, (bm, bn, kv, wm, wn, ns, kg)
    assert seen == 29


def test_scratch_memory_stays_where_it_is_known(kernels, igemm):
    """Values that kernels keep in scratch memory: a few of the 64 x 128 and 128 x 64 wave tiles, the tile with a tail, one LDS-patch tile and the widest pointwise
    kernel; no other"""
    for (types, bm, bn, kv, wm, wn, ns, kg, tail), k in igemm.items():
        most = 28 if tail and bm == 256 else 4 if (bm // wm) * (bn // wn) == 64 * 128 else 0
        assert k[".vgpr_spill_count"] <= most, (types, bm, bn, kv, wm, wn, ns, kg, tail)
    for n, k in kernels.items():
        if "convIgemmKernel" not in n:
            most = 1 if "convPatch8KernelI" in n and "Li256ELi192E" in n else 14 if "convPointwiseKernelILi4ELi4EE" in n else 0
            assert k[".vgpr_spill_count"] <= most, n
