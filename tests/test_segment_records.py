"""UnsortedSegmentSum of very many short rows: chunks whose runs are records (segments, then rows), cut at the end of a round."""
import pytest

from akg_amd import driver, op_desc
from test_segment_chunked import BY_CHUNK, _check_bits

RECORDS = BY_CHUNK + ", in records"


def _source(positions, width, segments, dtype="float32"):
    return driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, dtype, "int32", "records_%s_%d_%d_%d" % (
        dtype, positions, width, segments)), out_dir=None).source


def test_sizes_that_are_taken_in_records():
    assert RECORDS in _source(1 << 21, 3, 4954) and RECORDS in _source(24537162, 3, 4954) and RECORDS in _source(3000000, 2, 300)
    assert BY_CHUNK in _source((1 << 21) - 1, 3, 4954) and RECORDS not in _source((1 << 21) - 1, 3, 4954)


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype,ids,pattern", [
    (1, 1, 1, "float32", "int32", "uniform"), (513, 3, 700, "float32", "int32", "uniform"),
    (4097, 3, 1025, "float32", "int64", "uniform"),          # one position in the second chunk
    (300000, 1, 300, "float32", "int32", "uniform"),         # one segment a bucket: no sort
    (600000, 3, 513, "float32", "int32", "one_segment"),     # runs of whole chunks, every round cut inside one
    (70001, 4, 16384, "float32", "int32", "uniform"),        # 32 segments a bucket, rows of 16 bytes
    (100000, 3, 4954, "float32", "int32", "one_bucket"), (40000, 2, 3000, "float32", "int32", "sorted"),
    (40000, 2, 3000, "float32", "int32", "outside"), (20000, 1, 77, "float32", "int32", "nobody"),
    (70001, 2, 5000, "float16", "int32", "uniform"), (33333, 4, 999, "int8", "int32", "uniform"), (66000, 4, 1300, "bfloat16", "int64", "uniform"),
])
def test_bit_for_bit_the_serial_loop(positions, width, segments, dtype, ids, pattern, monkeypatch, tmp_path):
    monkeypatch.setenv("AKG_HIP_VARIANT", "6")
    assert RECORDS in _source(positions, width, segments, dtype)
    _check_bits(positions, width, segments, dtype, ids, pattern, tmp_path)


@pytest.mark.gpu
def test_the_default_choice(monkeypatch, tmp_path):
    monkeypatch.delenv("AKG_HIP_VARIANT", raising=False)
    _check_bits((1 << 21) + 4095, 3, 2000, "float32", "int32", "uniform", tmp_path)


def test_middling_sizes_that_are_taken_by_chunk():
    """Between 2^16 and 2^19 positions, where five launches grouped by segment or by fewer than 512 buckets."""
    for positions, width, segments in ((174184, 1, 361), (3 << 15, 3, 512), (149736, 3, 2040), (97239, 2, 3395), (70000, 3, 4088)):
        assert BY_CHUNK in _source(positions, width, segments)
    assert BY_CHUNK not in _source(70000, 3, 4096) and BY_CHUNK not in _source(70000, 4, 512)


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype,pattern", [(98304, 3, 512, "float32", "uniform"), (174184, 1, 361, "float32", "one_segment"),
                                                                     (97239, 2, 3395, "int32", "uniform"), (70000, 3, 4088, "float32", "outside")])
def test_middling_sizes_bit_for_bit(positions, width, segments, dtype, pattern, monkeypatch, tmp_path):
    monkeypatch.delenv("AKG_HIP_VARIANT", raising=False)
    _check_bits(positions, width, segments, dtype, "int32", pattern, tmp_path)
