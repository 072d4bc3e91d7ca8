"""UnsortedSegmentSum of wide rows, positions listed by segment in LDS: which sizes take it, and its results bit for bit the
serial loop's."""
import os

import numpy as np
import pytest

from akg_amd import driver, harness, op_desc

LISTED = "positions listed by segment"


def test_sizes_whose_positions_are_listed():
    def listed(positions, width, segments, dtype="float32"):
        kernel = driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, dtype, "int32", "s_%s_%d_%d_%d" % (
            dtype, positions, width, segments)), out_dir=None)
        assert LISTED not in kernel.source or kernel.workspace_bytes == 0
        return LISTED in kernel.source
    assert listed(512, 128, 1000) and listed(32768, 2048, 32768) and listed(65535, 65, 5, "bfloat16") and listed(100000, 128, 20000)
    assert not listed(511, 128, 1000) and not listed(32768, 64, 1000) and not listed(65536, 128, 1000) and not listed((1 << 20) + 1, 128, 20000)


def test_few_positions_load_their_ids_once_and_write_zeros_by_share():
    def source(positions, width, segments):
        return driver.HipKernel(op_desc.unsorted_segment_sum([positions], [width], segments, "float32", "int32", "f_%d" % positions), out_dir=None).source
    assert "U = 1;" in source(512, 1000, 32768) and "U = 2;" in source(2000, 128, 2000) and "U = 8;" in source(8192, 256, 8000)
    assert "BY_SHARE = true" in source(4096, 128, 2000) and "BY_SHARE = false" in source(4097, 128, 2000)


@pytest.mark.gpu
@pytest.mark.parametrize("positions,width,segments,dtype,ids,pattern", [
    (1, 65, 1, "float32", "int32", "uniform"), (3, 256, 7, "float32", "int64", "uniform"),
    (700, 257, 50, "float32", "int32", "uniform"),             # one column beyond a tile
    (4097, 128, 1000, "float32", "int32", "words"), (32768, 264, 32768, "float32", "int32", "words"),
    (8192, 200, 3000, "float32", "int32", "one_segment"),      # as many as the list holds
    (8193, 200, 3000, "float32", "int32", "one_segment"), (30001, 130, 3000, "float32", "int32", "one_group"),   # by windows
    (9000, 100, 40000, "float32", "int32", "sorted"), (5000, 96, 3000, "float32", "int32", "outside"),
    (2000, 80, 77, "float32", "int32", "nobody"),
    # zeros by share of adjacent segments: the last position count, pieces of 1 to 16 bytes, shares beyond the last segment
    (4096, 128, 1000, "float32", "int32", "words"), (512, 65, 40001, "float32", "int32", "uniform"), (600, 129, 3000, "bfloat16", "int32", "words"),
    (700, 130, 300, "int8", "int32", "uniform"), (1000, 68, 2000, "int64", "int64", "outside"), (520, 1026, 5000, "float16", "int32", "sorted"),
    (2000, 300, 1025, "float32", "int32", "one_segment"), (4000, 72, 70000, "float32", "int32", "nobody"),
    (30001, 72, 900, "float16", "int32", "words"), (9000, 520, 1300, "bfloat16", "int64", "one_segment"),   # additions that round
    (3333, 100, 999, "int8", "int32", "uniform"), (5001, 70, 333, "int64", "int32", "words"), (100000, 66, 20000, "int32", "int32", "uniform"),
])
def test_bit_for_bit_the_serial_loop(positions, width, segments, dtype, ids, pattern, monkeypatch, tmp_path):
    import torch
    from oracle import cpu_ref
    monkeypatch.setenv("AKG_HIP_VARIANT", "5")
    name = "listed_%s_%d_%d_%d_%s" % (dtype, positions, width, segments, pattern)
    text = op_desc.unsorted_segment_sum([positions], [width], segments, dtype, ids, name)
    path = os.path.join(str(tmp_path), name + ".info")
    open(path, "w").write(text)
    print("case %s" % name, flush=True)
    kernel = driver.HipKernel(text, out_dir=None)
    assert LISTED in kernel.source
    inputs = harness.make_inputs(harness.load_desc(path), seed=harness.BASE_SEED + 813)
    rng = np.random.default_rng(positions)
    at = {"uniform": rng.integers(0, segments, positions), "one_segment": np.full(positions, segments // 2),
          "words": np.exp(rng.random(positions) * np.log(segments)) - 1, "one_group": 1024 * rng.integers(0, 2, positions),
          "sorted": np.sort(rng.integers(0, segments, positions)), "outside": rng.integers(-4 * segments, 5 * segments, positions),
          "nobody": np.full(positions, segments)}[pattern]
    inputs[1] = at.astype(inputs[1].dtype).reshape(inputs[1].shape)
    want = cpu_ref.CpuKernel(path)(inputs)[0]
    on_device = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).cuda() for a in inputs]
    for _ in range(3):
        out = torch.full((kernel.outputs[0].nbytes,), 0x7b, dtype=torch.uint8, device="cuda")
        kernel.launch(on_device + [out])
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), np.ascontiguousarray(want).reshape(-1).view(np.uint8)), name
