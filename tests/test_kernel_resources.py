"""Registers and LDS of the built prefill GEMM kernels, from the metadata notes
of the code objects in libchimere_hip.so: how many work-groups fit a CU is what
their tile sizes and LDS stages were chosen by, and a register spilled in the
K loop is paid on every block."""
import os
import re
import struct

import msgpack
import pytest

from chimere_amd import _lib

LDS, VGPRS, WAVES = 160 * 1024, 512, 4     # of a CU; of a SIMD's lane; per work-group (one per SIMD)
Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, IQ3_S = 2, 8, 12, 13, 14, 21


def code_objects(data):
    """Offsets of the AMDGPU ELF images (OS ABI 64) embedded in a library."""
    at = data.find(b"\x7fELF\x02\x01\x01\x40")
    while at >= 0:
        yield at
        at = data.find(b"\x7fELF\x02\x01\x01\x40", at + 4)


def kernels():
    data = open(_lib.LIB_PATH, "rb").read()
    out = {}
    for o in code_objects(data):
        phoff, = struct.unpack_from("<Q", data, o + 32)
        size, count = struct.unpack_from("<HH", data, o + 54)
        for k in range(count):
            kind, _, off = struct.unpack_from("<IIQ", data, o + phoff + k * size)
            if kind == 4:                                       # PT_NOTE
                name, desc, note = struct.unpack_from("<III", data, o + off)
                if note == 32:                                  # NT_AMDGPU_METADATA
                    at = o + off + 12 + (name + 3) // 4 * 4
                    for m in msgpack.unpackb(data[at:at + desc])["amdhsa.kernels"]:
                        out[m[".name"]] = m
    return out


@pytest.fixture(scope="module")
def gemms():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    out = {}
    for name, m in kernels().items():
        k = re.match(r"_ZN7chimere\d+k_pf_(gate_up|down)ILi(\d+)ELi(\d+)ELi(\d)EE", name)
        if k:
            out[k[1], int(k[2]), int(k[3]), int(k[4])] = m
    assert len(out) == 2 * 3 * 6 * 3
    return out


def groups_per_cu(m):
    return min(LDS // m[".group_segment_fixed_size"], VGPRS // ((m[".vgpr_count"] + 7) // 8 * 8))


def test_prefill_gemm_spills(gemms):
    """No register of a prefill GEMM is spilled, but a few at 32 pairs where three
    work-groups per CU are worth them (at most 7 of 168)."""
    for (launch, te, ts, mt), m in gemms.items():
        few = mt == 2 and (launch == "gate_up") == (ts in (Q4_K, Q5_K, Q6_K))
        assert m[".vgpr_spill_count"] <= (7 if few else 0), (launch, te, ts, mt, m[".vgpr_spill_count"])


def test_prefill_gemm_work_groups_per_cu(gemms):
    """16 pairs: three work-groups per CU, two where the expert and shared types
    are IQ3_S and Q4_0 / Q8_0 (the wider stage of the one and the codebook of
    the other: 54,816 bytes of LDS); 32 pairs: three, two in the down launch of a
    K-quant shared expert; 64 pairs: two."""
    for (launch, te, ts, mt), m in gemms.items():
        mixed = te != ts and IQ3_S in (te, ts) and {te, ts} & {Q4_0, Q8_0}
        if mt == 1:
            want = 2 if mixed else 3
        elif mt == 2:
            want = 2 if launch == "down" and ts in (Q4_K, Q5_K, Q6_K) else 3
        else:
            want = 2
        assert groups_per_cu(m) == want, (launch, te, ts, mt)
