"""Which kernel or shape a size gets (CPU; the rules of csrc/dispatch_rules.h at
the 256 CUs of an MI355X): the sizes of the GPU tests reach what they are there
for, and at the measured sizes the rule takes the faster side."""
import pytest

from tests import dispatch as D
from tests import helpers as H
from tests import test_gpu_a8_dense as A8
from tests import test_gpu_affine_dense as AD
from tests import test_gpu_exact_dequant as ED
from tests import test_gpu_gemm_stream as GS
from tests import test_gpu_moe_group as MG
from tests import test_gpu_small_m as SM


def test_a8_shape_cases_reach_every_shape():
    for m, n, k, _, shape in A8.SHAPES:
        assert D.a8_shape([(m, n, k)], few=m <= 16) == shape, (m, n, k)
        passes = -(-k // (128 * shape[1]))
        assert passes >= 4 and k // 64 % 2 == 1
    assert len({c[-1] for c in A8.SHAPES}) == 6


def test_a8_few_rows_take_the_exact_shape():
    for m in (1, 5, 16):
        for n in (40, 16500, 200000):
            assert D.a8_shape([(m, n, 4096)], few=True) == (1, 8)


def test_a8_row_cases_are_on_both_sides():
    for m, n, k, wave4, wave8 in A8.ROWS:
        assert D.a8_wave_per_row(m, n, k, 4) == wave4 and D.a8_wave_per_row(m, n, k, 8) == wave8, (m, n, k)
    for m in (1, 2):
        for side in (3, 4):
            assert {c[side] for c in A8.ROWS if c[0] == m} == {True, False}
    assert not D.a8_wave_per_row(3, 64, 64, 4) and not D.a8_wave_per_row(3, 64, 64, 8)


# bits, rows, n, k, us with a wave a row, us streaming (one MI355X, graph replays over weight copies)
MEASURED = [(4, 1, 256, 8192, 7.24, 10.07), (4, 1, 512, 2048, 3.27, 4.27), (4, 1, 1024, 1024, 3.24, 3.59),
            (4, 1, 2048, 8192, 9.11, 10.23), (4, 1, 2304, 4096, 6.40, 6.75), (4, 1, 2560, 2048, 4.83, 5.07),
            (4, 1, 2560, 1024, 4.49, 4.33), (4, 1, 3584, 4096, 7.24, 6.85), (4, 1, 4608, 1024, 5.14, 4.47),
            (4, 2, 1024, 4096, 6.29, 6.75), (4, 2, 1024, 8192, 8.98, 10.23), (8, 1, 1024, 1024, 3.48, 4.59),
            (8, 1, 2560, 512, 3.71, 4.60), (8, 1, 3072, 1024, 4.62, 4.78), (8, 1, 1024, 2048, 4.59, 5.48),
            (8, 1, 512, 4096, 6.53, 7.28), (8, 1, 4608, 1024, 5.18, 4.93), (8, 1, 1536, 2048, 5.80, 5.46),
            (8, 1, 1024, 8192, 12.36, 11.53), (8, 2, 2048, 1024, 4.21, 4.80), (8, 2, 3072, 512, 4.28, 4.71)]


@pytest.mark.parametrize("bits,m,n,k,wave,stream", MEASURED)
def test_a8_row_rule_takes_the_faster_side(bits, m, n, k, wave, stream):
    assert D.a8_wave_per_row(m, n, k, bits) == (wave < stream)


def _layer(m, hidden, inter):
    kv = hidden // 4 // 64 * 64
    return [(m, hidden, hidden), (m, kv, hidden), (m, kv, hidden), (m, hidden, hidden), (m, inter, hidden),
            (m, inter, hidden), (m, hidden, inter)]


def _pair(m, hidden, inter):
    return [(m, inter, hidden)] * 2


# 4-bit, one row: products of a call, us on qmv_mfma, us dense (differences of 2% and more)
MEASURED_IDLE = [(_layer(1, 3072, 8192), 16.4, 15.4), (_layer(1, 2560, 6912), 14.6, 14.0), (_layer(1, 1536, 4096), 7.65, 7.08),
                 (_layer(1, 1280, 3584), 7.47, 6.81), (_layer(1, 2816, 8448), 16.5, 15.7), (_layer(1, 512, 1536), 6.69, 3.82),
                 (_layer(1, 1024, 2048), 4.69, 5.36), (_layer(1, 1024, 4096), 5.80, 6.58), (_layer(1, 1536, 6144), 8.43, 9.37),
                 (_layer(1, 3328, 9984), 17.9, 20.2), (_pair(1, 1024, 3072), 4.65, 3.38), (_pair(1, 2560, 6912), 9.06, 7.45),
                 (_pair(1, 3072, 8192), 9.82, 7.97), (_layer(1, 2048, 6144), 9.7, 11.0), ([(1, 3072, 8192)], 1.0, 1.1)]


@pytest.mark.parametrize("sizes,mfma,dense", MEASURED_IDLE)
def test_idle_rule_takes_the_faster_side(sizes, mfma, dense):
    assert D.few_rows(sizes, 4)[0] == (dense < mfma)
    assert D.few_rows(sizes, 8) == (False, False)


def test_unreadable_products_drag_what_a_second_launch_costs_more_for():
    for bits in (4, 8):
        layer = _layer(1, 2560, 6912)
        assert D.few_rows(layer, bits, readable=[True] * 6 + [False])[1]
        # a small one beside 600 MB stays alone
        big = [(1, 100, 4096), (1, 151936 * 8 // bits, 4096)]
        assert not D.few_rows(big, bits, readable=[False, True])[1]


# 8-bit, eight rows: products of a call, us on qmv_mfma, us dense
MEASURED_W8 = [([(8, 12288, 4096)], 16.2, 16.9), ([(8, 12288, 1024)], 5.83, 7.06), ([(8, 12288, 12288)], 39.8, 45.1),
               ([(8, 24576, 1024)], 9.61, 10.93), ([(8, 4096, 1024)], 4.22, 4.70), ([(8, 4096, 4096)], 10.9, 9.2),
               ([(8, 6912, 4096)], 21.1, 10.1), ([(8, 6912, 1024)], 7.1, 4.95), ([(8, 14336, 1024)], 7.95, 7.29),
               ([(8, 24576, 2048)], 16.7, 13.4), ([(8, 27648, 5120)], 39.1, 43.0), ([(8, 27648, 4096)], 32.6, 30.3),
               ([(8, 11008, 4096)], 1.0, 0.76), (_pair(8, 1024, 4096), 5.05, 5.45), (_pair(8, 1024, 2816), 4.84, 5.23),
               (_layer(8, 2304, 6912), 22.9, 24.6), (_layer(8, 2560, 6912), 25.1, 26.1), (_layer(8, 5120, 13824), 72.2, 75.2),
               (_layer(8, 4096, 11008), 47.0, 44.5)]


@pytest.mark.parametrize("sizes,mfma,dense", MEASURED_W8)
def test_w8_rule_takes_the_faster_side(sizes, mfma, dense):
    assert D.w8_rows5_mfma(sizes) == (mfma < dense)


def test_w8_cases_reach_both_kernels():
    for m, n, k, mfma in AD.W8_ROWS:
        assert 5 <= m <= 8 and D.w8_rows5_mfma([(m, n, k)]) == mfma, (m, n, k)
    assert {c[-1] for c in AD.W8_ROWS} == {True, False}


def test_small_m_cases_run_in_long_launches():
    """And only there: the same sizes alone are the dense kernel's."""
    for m in SM.ROWS:
        for n, k in SM.SHAPES:
            assert 9 <= m <= 16 and n >= 16 and k % 1024 == 0
            assert D.small_m_long([(m, n, k), (m,) + H.LONG_LAUNCH]) and not D.small_m_long([(m, n, k)])
    layer = _layer(16, 4096, 12288)
    assert D.small_m_long(layer) and not D.small_m_long(_layer(16, 3072, 8192)) and not D.small_m_long(_layer(16, 2048, 6144))


def test_moe_rule():
    for rows, model, hidden, experts, *_ in MG.SLOTS + MG.EXACT + [(60, 256, 192, 3)]:
        assert D.moe_grouped(rows, experts, model, hidden)
    assert not D.moe_grouped(33, 1, 1024, 512) and not D.moe_grouped(64, 1, 1024, 512)
    assert not D.moe_grouped(16, 128, 2048, 768) and D.moe_grouped(17, 2, 2048, 768) and D.moe_grouped(65, 1, 2048, 1024)


# logits, rows, sampled, filters, time in the split form over that in the row form
MEASURED_SAMPLE = [(16385, 32, False, False, 0.82), (20000, 48, False, False, 0.79), (151936, 1, False, False, 0.11),
                   (16385, 128, False, False, 1.38), (24000, 256, False, False, 1.55), (32000, 192, False, False, 0.80),
                   (32000, 512, False, False, 1.54), (65536, 512, False, False, 1.12), (2, 1, True, False, 0.60),
                   (64, 512, True, True, 1.43), (4096, 512, True, True, 1.05), (256, 128, True, True, 0.62),
                   (16384, 512, True, False, 0.60), (4096, 32, True, True, 0.61)]


@pytest.mark.parametrize("vocab,rows,sampled,filters,ratio", MEASURED_SAMPLE)
def test_sampling_rule_takes_the_faster_side(vocab, rows, sampled, filters, ratio):
    assert D.sample_split(vocab, rows, sampled, filters) == (ratio < 1)


def test_sampling_cases_reach_the_split_form():
    for vocab, batch in [(16385, 3), (20480, 2), (32769, 2), (17000, 4), (81000, 300)]:
        assert D.sample_split(vocab, batch, False, False) and D.sample_split(vocab, batch, True, True)
    assert D.sample_split(16400, 300, True, True) and not D.sample_split(600, 300, True, True)


# products of a launch, bits, us on the GEMM and streaming
MEASURED_STREAM = [([(97, 8192, 4096)], 4, 32.4, 22.5), ([(97, 10240, 4096)], 4, 32.6, 30.5), ([(97, 12288, 4096)], 4, 32.7, 34.3),
                   ([(97, 28672, 4096)], 4, 50.9, 64.1), ([(96, 12288, 8192)], 4, 59.2, 58.1), ([(96, 20480, 4096)], 4, 48.6, 46.4),
                   ([(96, 28672, 2048)], 8, 32.0, 36.1), ([(128, 8192, 4096)], 4, 30.9, 22.9), ([(128, 10240, 2048)], 4, 16.1, 19.0),
                   ([(128, 12288, 8192)], 4, 58.0, 65.6), ([(128, 10240, 8192)], 8, 66.0, 58.3), ([(128, 12288, 4096)], 8, 35.5, 38.0),
                   (_pair(100, 2048, 6144), 4, 18.6, 19.1), (_pair(128, 2048, 6144), 8, 17.4, 19.2), (_pair(100, 2560, 6912), 4, 21.8, 23.7),
                   (_layer(100, 4096, 12288), 4, 104.0, 100.0), (_layer(97, 2560, 6912), 4, 53.0, 44.0),
                   (_layer(97, 4096, 8192), 4, 73.6, 81.5), (_layer(128, 2048, 2048), 4, 19.3, 21.2)]


@pytest.mark.parametrize("sizes,bits,gemm,stream", MEASURED_STREAM)
def test_stream_rule_takes_the_faster_side(sizes, bits, gemm, stream):
    assert D.stream_takes(sizes, bits) == (stream < gemm)


# products of a launch, us with 32 and with 64 columns a workgroup
MEASURED_WIDE = [([(64, 8192, 4096)], 16.3, 22.8), ([(64, 10240, 4096)], 26.6, 22.9), ([(64, 16384, 4096)], 27.3, 23.5),
                 ([(64, 28672, 4096)], 49.9, 38.9), ([(96, 10240, 2048)], 16.1, 17.5), ([(96, 10240, 4096)], 30.4, 28.9),
                 ([(48, 12288, 8192)], 43.6, 37.0), ([(17, 10240, 8192)], 28.8, 33.4), ([(32, 28672, 4096)], 35.6, 29.9),
                 ([(128, 4096, 4096)], 13.9, 20.3), ([(128, 8192, 4096)], 25.4, 22.9), (_layer(64, 2560, 6912), 32.2, 37.7),
                 (_layer(64, 4096, 12288), 77.9, 71.9)]


@pytest.mark.parametrize("sizes,narrow,wide", MEASURED_WIDE)
def test_stream_width_takes_the_faster_side(sizes, narrow, wide):
    assert D.stream_wide(sizes) == (wide < narrow)


def test_stream_cases_reach_both_widths_and_the_kernel():
    for m, n, k, f16, wide in GS.SUMS:
        assert D.stream_wide([(m, n, k)]) == wide, (m, n, k)
        assert m <= 64 or D.stream_takes([(m, n, k)], 4)
    for m, n, k in GS.EXACT:
        assert m <= 64 or (D.stream_takes([(m, n, k)], 4) and D.stream_takes([(m, n, k)], 8)), (m, n, k)
    assert {D.stream_blocks([(m, n, k)]) for m, n, k in GS.EXACT} == {2, 3, 4}
    for bits in (4, 8):
        assert not D.stream_takes([ED.GEMM64 + (64,)], bits) and not D.stream_takes([ED.GEMM64 + (704,)], bits)
