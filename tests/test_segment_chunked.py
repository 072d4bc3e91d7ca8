"""UnsortedSegmentSum of short rows, chunks of positions grouped by bucket of segments where they lie: which sizes take it, and
its results bit for bit the serial loop's."""
import os
import re

import numpy as np
import pytest

from akg_amd import driver, harness, op_desc

BY_CHUNK = "grouped by bucket of segments, chunk by chunk"


def test_sizes_that_are_taken_by_chunk():
    def by_chunk(positions, width, segments, dtype="float32"):
        kernel = driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, dtype, "int32", "s_%s_%d_%d_%d" % (
            dtype, positions, width, segments)), out_dir=None)
        return BY_CHUNK in kernel.source
    assert by_chunk(1 << 19, 3, 4954) and by_chunk(1 << 19, 1, 300) and by_chunk(1 << 15, 4, 300) and by_chunk(65535, 2, 5)
    assert by_chunk(70000, 1, 13950) and by_chunk(70000, 4, 513) and not by_chunk(70000, 4, 512) and not by_chunk(70000, 3, 5000)
    assert not by_chunk(32767, 3, 4954)
    assert not by_chunk(1 << 19, 5, 300) and not by_chunk(1 << 19, 3, 300, "float16") and not by_chunk(1 << 15, 3, 40000)
    # 17 bytes a position are beyond the 16 MiB of a launch without allocations where 16 were within
    assert not by_chunk(1020000, 4, 100) and by_chunk(980000, 4, 100) and by_chunk(1100000, 4, 100)


@pytest.mark.parametrize("positions,width,segments", [(2000000, 3, 20000), (4000000, 4, 30000), (1200000, 3, 16385), (1 << 20, 4, 32768), (3000000, 1, 20000),
                                                      (600000, 3, 20000), (540000, 1, 32768)])
def test_more_segments_than_are_grouped_need_no_scratch_beyond_the_static_one(positions, width, segments):
    """More than 16384 segments were scanned, without a workspace: a launch that allocates nothing serves these still."""
    kernel = driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, "float32", "int32", "ws_%d_%d_%d" % (
        positions, width, segments)), out_dir=None)
    assert kernel.workspace_bytes <= 16 << 20
    assert (BY_CHUNK in kernel.source) == (kernel.workspace_bytes > 0)


def _check_bits(positions, width, segments, dtype, ids, pattern, tmp_path):
    import torch
    from oracle import cpu_ref
    name = "by_chunk_%s_%d_%d_%d_%s" % (dtype, positions, width, segments, pattern)
    text = op_desc.unsorted_segment_sum([positions], [width], segments, dtype, ids, name)
    path = os.path.join(str(tmp_path), name + ".info")
    open(path, "w").write(text)
    print("case %s" % name, flush=True)
    kernel = driver.HipKernel(text, out_dir=None)
    assert BY_CHUNK in kernel.source
    inputs = harness.make_inputs(harness.load_desc(path), seed=harness.BASE_SEED + 812)
    rng = np.random.default_rng(positions)
    at = {"uniform": rng.integers(0, segments, positions), "one_segment": np.full(positions, segments // 2),
          "one_bucket": rng.integers(10, 20, positions), "sorted": np.sort(rng.integers(0, segments, positions)),
          "outside": rng.integers(-4 * segments, 5 * segments, positions), "nobody": np.full(positions, segments)}[pattern]
    inputs[1] = at.astype(inputs[1].dtype).reshape(inputs[1].shape)
    want = cpu_ref.CpuKernel(path)(inputs)[0]
    on_device = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).cuda() for a in inputs]
    for _ in range(3):
        out = torch.full((kernel.outputs[0].nbytes,), 0x7b, dtype=torch.uint8, device="cuda")
        kernel.launch(on_device + [out])
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), np.ascontiguousarray(want).reshape(-1).view(np.uint8)), name


@pytest.mark.parametrize("positions,width,segments,dtype,split", [
    (33000, 1, 32768, "float32", 0), (33000, 3, 32768, "float32", 0), (65535, 4, 32768, "float32", 0), (40000, 4, 20000, "float32", 0),
    (40000, 3, 25000, "float32", 0), (33000, 4, 30000, "bfloat16", 0), (65535, 3, 32204, "int32", 0), (70000, 4, 16384, "float32", 0),
    (540000, 4, 16384, "float32", 0), (40000, 4, 300, "float32", 0), (33000, 3, 6400, "float32", 100), (140000, 4, 6400, "float32", 100), (100000, 4, 5000, "float32", 0),
])
def test_every_output_element_has_a_lane(positions, width, segments, dtype, split, monkeypatch):
    """One lane adds one output element: the wavefronts of the last launch have a lane for each element of a bucket."""
    monkeypatch.setenv("AKG_HIP_VARIANT", "4" if split else "0")
    monkeypatch.setenv("AKG_HIP_SPLIT", str(split))
    source = driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, dtype, "int32", "lanes_%s_%d_%d_%d" % (
        dtype, positions, width, segments)), out_dir=None).source
    assert BY_CHUNK in source
    waves, rounds, chains, per_wave = map(int, re.search(r"W = (\d+), T = (\d+), CAP = .*CHAINS = (\d+), PER_WAVE = (\d+);", source).groups())
    chunk = 512 * int(re.search(r"NW = 8, TILES = (\d+)", source).group(1))
    assert chains >= width and per_wave <= 64 and waves * per_wave >= chains and waves * rounds * 64 >= chunk
    assert waves * rounds * 64 >= (2048 if chunk > 512 else 512)   # a frequent segment takes as many rounds as its positions


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype", [(40000, 4, 20000, "float32"), (40000, 4, 32768, "float32"), (65535, 3, 32204, "float32"),
                                                            (33000, 4, 30000, "bfloat16"), (70000, 4, 16384, "int32")])
def test_buckets_of_many_output_elements(positions, width, segments, dtype, monkeypatch, tmp_path):
    """More than 128 output elements a bucket, through the default choice of the schedule."""
    monkeypatch.delenv("AKG_HIP_VARIANT", raising=False)
    _check_bits(positions, width, segments, dtype, "int32", "uniform", tmp_path)


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype,ids,pattern,chunks", [
    (1, 1, 1, "float32", "int32", "uniform", 0),
    (511, 3, 700, "float32", "int32", "uniform", 1), (513, 4, 513, "float32", "int64", "uniform", 1),   # edges of a chunk
    (4097, 2, 1025, "float32", "int32", "uniform", 8), (33000, 3, 4954, "float32", "int32", "uniform", 0),
    (300000, 1, 512, "float32", "int32", "uniform", 2),      # more chunks than a round looks up
    (9000, 4, 32768, "int32", "int32", "uniform", 4),        # 64 segments a bucket
    (70001, 4, 5000, "float32", "int32", "uniform", 2), (70001, 2, 700, "bfloat16", "int32", "one_bucket", 2),   # rounds of two chunks
    (150000, 3, 9000, "float32", "int32", "one_segment", 8), (70000, 4, 600, "float32", "int32", "one_segment", 1),
    (100000, 3, 4954, "float32", "int32", "one_bucket", 4), (40000, 2, 3000, "float32", "int32", "sorted", 0),
    (40000, 2, 3000, "float32", "int32", "outside", 2), (20000, 1, 77, "float32", "int32", "nobody", 0),
    (70001, 2, 5000, "float16", "int32", "uniform", 0), (66000, 4, 1300, "bfloat16", "int64", "uniform", 0),   # additions that round
    (33333, 4, 999, "int8", "int32", "uniform", 0), (540000, 3, 16384, "float32", "int32", "uniform", 0),
])
def test_bit_for_bit_the_serial_loop(positions, width, segments, dtype, ids, pattern, chunks, monkeypatch, tmp_path):
    monkeypatch.setenv("AKG_HIP_VARIANT", "4")
    if chunks:
        monkeypatch.setenv("AKG_HIP_CHUNKS", str(chunks))
    _check_bits(positions, width, segments, dtype, ids, pattern, tmp_path)


@pytest.mark.parametrize("positions,width,segments", [(956289, 1, 14006), (365857, 3, 609), (2180885, 3, 1444), (784959, 1, 590)])
def test_integer_sums_stay_in_registers(positions, width, segments, tmp_path):
    from gemm_checks import compiled_notes
    text = op_desc.unsorted_segment_sum([positions], [width], segments, "int32", "int32", "ints_%d_%d_%d" % (positions, width, segments))
    kernel, scratch, _ = compiled_notes(text, tmp_path)
    assert "grouped by bucket of segments" in kernel.source and scratch == 0


@pytest.mark.parametrize("positions,width,segments,dtype,values", [
    (65101, 4, 1536, "bfloat16", 16), (579545, 2, 16024, "float16", 16), (100000, 2, 196, "float16", 16), (100000, 2, 195, "float16", 48),   # 510 and 514 positions a segment
    (4405314, 4, 901, "bfloat16", 48), (65101, 4, 1536, "float32", 48), (365857, 3, 609, "int32", 16),
])
def test_values_of_a_list_in_flight(positions, width, segments, dtype, values):
    kernel = driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, dtype, "int32", "flight_%s_%d_%d_%d" % (dtype, positions, width, segments)), out_dir=None)
    assert "constexpr int ADD_BLOCK = %d;" % values in kernel.source


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype", [(65101, 4, 1536, "bfloat16"), (100000, 2, 196, "float16"), (100000, 2, 195, "float16"), (70001, 4, 2000, "int32")])
def test_lists_with_fewer_and_more_values_in_flight(positions, width, segments, dtype, tmp_path):
    for pattern in ("uniform", "one_segment"):
        _check_bits(positions, width, segments, dtype, "int32", pattern, tmp_path)
