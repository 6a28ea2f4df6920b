"""The dispatch rules of stark_amd/csrc/dispatch_rules.h, compiled for the CPU,
so that a test can say which kernel or shape its sizes get."""
import ctypes as C
import functools
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stark_amd", "csrc")
CUS = 256  # of an MI355X

_WRAP = """
#include "dispatch_rules.h"
struct Op { uint32_t m, n, k; };
extern "C" {
int a8_wave_per_row(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t cus) {
    return qmm::a8_wave_per_row(m, n, k, bits, cus);
}
int a8_shape(const Op* ops, uint32_t count, int few, uint32_t cus, int* mt, int* kw) {
    const qmm::A8Shape& s = qmm::kA8Shapes[qmm::a8_shape(ops, count, few != 0, cus)];
    *mt = s.mt;
    *kw = s.kw;
    return 0;
}
int few_rows(const Op* ops, const int* readable, uint32_t count, int bits, uint32_t cus) {
    const auto read = [&](const Op& o) { return readable[&o - ops] != 0; };
    const qmm::FewRowsRule r = qmm::few_rows_rule(ops, count, bits, cus, read);
    return (r.idle ? 1 : 0) | (r.drag ? 2 : 0);
}
int stream_wide(const Op* ops, uint32_t count, uint32_t cus) { return qmm::stream_wide(ops, count, cus); }
int stream_takes(const Op* ops, uint32_t count, int bits, uint32_t cus) { return qmm::stream_takes(ops, count, bits, cus); }
int stream_blocks(const Op* ops, uint32_t count) { return (int)qmm::stream_blocks(ops, count); }
int sample_split(uint32_t v, uint32_t rows, int sampled, int filters) { return qmm::sample_split(v, rows, sampled != 0, filters != 0); }
int moe_grouped(uint32_t t, uint32_t e, uint32_t model, uint32_t hidden) { return qmm::moe_grouped(t, e, model, hidden); }
int small_m_long(const Op* ops, uint32_t count, uint32_t cus) { return qmm::small_m_long(ops, count, cus); }
int w8_rows5_mfma(const Op* ops, uint32_t count, uint32_t cus) { return qmm::w8_rows5_mfma(ops, count, cus); }
}
"""


class Op(C.Structure):
    _fields_ = [("m", C.c_uint32), ("n", C.c_uint32), ("k", C.c_uint32)]


@functools.lru_cache(None)
def rules():
    with tempfile.TemporaryDirectory() as d:
        src, lib = os.path.join(d, "rules.cpp"), os.path.join(d, "rules.so")
        with open(src, "w") as f:
            f.write(_WRAP)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, src, "-o", lib], check=True)
        return C.CDLL(lib)


def ops(*sizes):
    return (Op * len(sizes))(*[Op(*s) for s in sizes])


def a8_wave_per_row(m, n, k, bits, cus=CUS):
    return bool(rules().a8_wave_per_row(m, n, k, bits, cus))


def a8_shape(sizes, few, cus=CUS):
    """(16-row blocks, waves along K) of a launch of products (m, n, k)."""
    mt, kw = C.c_int(), C.c_int()
    rules().a8_shape(ops(*sizes), len(sizes), int(few), cus, C.byref(mt), C.byref(kw))
    return mt.value, kw.value


def few_rows(sizes, bits, readable=None, cus=CUS):
    """(idle, drag) of a launch's products of one or two rows; readable: those whose planes qmv_mfma can read."""
    flags = (C.c_int * len(sizes))(*([1] * len(sizes) if readable is None else [int(r) for r in readable]))
    r = rules().few_rows(ops(*sizes), flags, len(sizes), bits, cus)
    return bool(r & 1), bool(r & 2)


def w8_rows5_mfma(sizes, cus=CUS):
    return bool(rules().w8_rows5_mfma(ops(*sizes), len(sizes), cus))


def small_m_long(sizes, cus=CUS):
    return bool(rules().small_m_long(ops(*sizes), len(sizes), cus))


def moe_grouped(tokens, experts, model, hidden):
    return bool(rules().moe_grouped(tokens, experts, model, hidden))


def sample_split(vocab, rows, sampled, filters):
    return bool(rules().sample_split(vocab, rows, int(sampled), int(filters)))


def stream_wide(sizes, cus=CUS):
    return bool(rules().stream_wide(ops(*sizes), len(sizes), cus))


def stream_takes(sizes, bits, cus=CUS):
    return bool(rules().stream_takes(ops(*sizes), len(sizes), bits, cus))


def stream_blocks(sizes):
    return rules().stream_blocks(ops(*sizes), len(sizes))
