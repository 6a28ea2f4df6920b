"""Bounds of the weight loads of the streaming kernels (CPU): the 16 bytes that
a lane quarter loads lie in its own row for every K of whole 64-value groups, a
row of one group (32 bytes at 4 bits) included, and within K they are its codes."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stark_amd", "csrc")


@pytest.fixture(scope="module")
def layout(tmp_path_factory):
    d = tmp_path_factory.mktemp("code_layout")
    src, lib = d / "wrap.cpp", d / "wrap.so"
    src.write_text('#include "code_layout.h"\n'
                   'extern "C" uint32_t offset(int bits, uint32_t k, uint32_t h, uint32_t kq, uint32_t K) {\n'
                   '    return bits == 4 ? qmm::code_offset<4>(k, h, kq, K) : qmm::code_offset<8>(k, h, kq, K);\n}\n'
                   'extern "C" uint32_t split(uint32_t k, uint32_t kq, uint32_t K) {\n'
                   '    return qmm::code_lane_offset(kq, K) + qmm::code_chunk_offset(k, kq, K);\n}\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(lib)], check=True)
    so = C.CDLL(str(lib))
    so.offset.restype = so.split.restype = C.c_uint32
    so.offset.argtypes, so.split.argtypes = [C.c_int] + [C.c_uint32] * 4, [C.c_uint32] * 3
    return so


@pytest.mark.parametrize("bits", [4, 8])
def test_loads_stay_in_the_row(layout, bits):
    for K in range(64, 1601, 64):
        row = K * bits // 8
        for k in range(0, K, 128):
            for h in range(bits // 4):
                for kq in range(4):
                    first = k + 32 * kq if bits == 4 else k + 64 * h + 16 * kq
                    offsets = [layout.offset(bits, k, h, kq, K)]
                    if bits == 4:
                        offsets.append(layout.split(k, kq, K))
                    for at in offsets:
                        assert at % 16 == 0 and at + 16 <= row, (K, k, h, kq, at)
                        assert first >= K or at == first * bits // 8


def test_kernels_use_the_checked_offsets():
    """The kernels that stream codes to registers in this form take their offsets from the checked functions."""
    for name, call, count in (("moe_group.hip", "code_lane_offset(", 2), ("moe_group.hip", "code_chunk_offset(", 1),
                              ("qmv_dense.hip", "code_offset<BITS>(", 1), ("qmv_a8_dense.hip", "code_offset<BITS>(", 1)):
        with open(os.path.join(CSRC, name)) as f:
            text = f.read()
        assert text.count(call) == count and "row_bytes + 16 * kq" not in text, name
