"""The small-tile contraction kernel: which products take it, and its results at the edges of tiles, steps and splits."""
import json
import os

import pytest

from akg_amd import driver, op_desc


def _product(m, k, n, dtype, tb, name):
    """A @ B + bias [N] with the accumulator's type as the result."""
    b = op_desc.DescBuilder(name)
    x, w = b.input([m, k], dtype), b.input([n, k] if tb else [k, n], dtype)
    acc = "int32" if dtype == "int8" else "float32"
    bias = b.input([n], acc)
    attrs = [{"data_type": "bool", "name": "transpose_a", "value": False}, {"data_type": "bool", "name": "transpose_b", "value": tb}]
    return b.dumps([b.add(b.op("MatMul", [x, w], [m, n], acc, attrs=attrs), bias)])


def _schedule(text, directory):
    driver.HipKernel(text, out_dir=str(directory))
    return json.load(open(os.path.join(str(directory), json.loads(text)["op"] + ".json")))["schedule"]


def test_products_that_take_small_tiles(tmp_path, monkeypatch):
    def tile(m, k, n, dtype="bfloat16", tb=True):
        note = _schedule(_product(m, k, n, dtype, tb, "tiles_%s_%d_%d_%d_%d" % (dtype, m, k, n, tb)), tmp_path)
        splits = [w for w in note.split() if w.startswith("k_splits=")]
        return [w for w in note.split() if w.startswith("tile=") or w == "skinny:"][0].split("x64")[0], splits
    assert tile(300, 1024, 1024) == ("tile=64", [])                       # 64 x 64 x 64
    assert "tile=64x64" in _schedule(_product(128, 2048, 4096, "float16", False, "tiles_split"), tmp_path)
    assert tile(128, 2048, 4096)[1] == ["k_splits=2"]
    assert tile(300, 4096, 11000)[0] == "tile=64x128"
    assert tile(640, 4096, 11000)[0] == "tile=128x128"
    assert tile(48, 2048, 4096)[0] == "tile=64"
    # large products, small weights, at most 32 rows, and rows of B that are not whole 16-byte chunks keep their kernels
    assert tile(4096, 8192, 8192)[0] == tile(1200, 8192, 2048)[0] == tile(512, 1024, 768)[0] == "tile=256x256"
    assert tile(32, 2048, 4096)[0] == "skinny:"
    assert tile(300, 2048, 1028, tb=False)[0] == "tile=256x256" and tile(300, 2048, 1028)[0] == "tile=64"
    monkeypatch.setenv("AKG_HIP_VARIANT", "128")
    assert tile(300, 4096, 11000)[0] == "tile=256x256"


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype,tb,tile", [
    (65, 1032, 1096, "bfloat16", True, "64x64"),      # one row and eight columns beyond a tile, a K tail of eight
    (65, 1032, 1096, "bfloat16", False, "64x64"),
    (33, 4096, 1024, "float16", False, "64x64"),      # the fewest rows, eight splits
    (130, 8200, 1032, "float16", True, "64x64"),      # ragged splits with a K tail
    (300, 4096, 11000, "bfloat16", False, "64x128"),  # ragged tiles of 128 columns
    (700, 1000, 4100, "bfloat16", True, "128x128"),   # columns that are not a multiple of 8
    (645, 1024, 6008, "float16", False, "128x128"),
    (192, 4112, 4112, "int8", False, "64x64"),        # 8-bit operands: whole steps of 128, a tail of 16
    (64, 4096, 4100, "int8", True, "64x64"),
    (1200, 1040, 6016, "int8", False, "128x128"),
    (1200, 4096, 1536, "bfloat16", False, "64x128"),
])
def test_small_tiles_against_float64(m, k, n, dtype, tb, tile, tmp_path):
    """float32 sums of k products differ from the exact sum by at most k * 2^-24 of the sum of the products' magnitudes
    (whatever their order), plus the bias addition's half unit; 8-bit products are exact. Twice: the counters of a split
    must be left ready."""
    import torch
    text = _product(m, k, n, dtype, tb, "small_tile_%s_%dx%dx%d_%d" % (dtype, m, k, n, tb))
    note = _schedule(text, tmp_path)
    assert "tile=%sx" % tile in note
    kernel = driver.HipKernel(text, out_dir=str(tmp_path))
    print("case", note, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    if dtype == "int8":
        a = torch.randint(-128, 128, (m, k), generator=g, device="cuda", dtype=torch.int8)
        b = torch.randint(-128, 128, (n, k) if tb else (k, n), generator=g, device="cuda", dtype=torch.int8)
        bias = torch.randint(-1000, 1000, (n,), generator=g, device="cuda", dtype=torch.int32)
    else:
        td = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
        a = torch.randn((m, k), generator=g, device="cuda").to(td)
        b = torch.randn((n, k) if tb else (k, n), generator=g, device="cuda").to(td)
        bias = torch.randn((n,), generator=g, device="cuda")
    wide = b.double().t().contiguous() if tb else b.double()
    exact = a.double() @ wide + bias.double()
    slack = (a.double().abs() @ wide.abs()) * (k * 2.0 ** -24) + exact.abs() * 2.0 ** -23 if dtype != "int8" else torch.zeros_like(exact)
    out = torch.empty((m, n), dtype=bias.dtype, device="cuda")
    for launch in range(2):
        out.fill_(-7)
        kernel.launch([a, b, bias, out])
        torch.cuda.synchronize()
        bad = (out.double() - exact).abs() > slack
        assert not bool(bad.any()), "launch %d: %d wrong, first %s" % (launch, int(bad.sum()), bad.nonzero()[0].tolist())


@pytest.mark.parametrize("m,k,n,dtype,tb,kernel", [
    # [K,N] weights: the skinny kernel is the faster one where the tiles leave CUs with two workgroups
    (33, 8192, 6144, "bfloat16", False, "skinny"), (33, 8192, 2048, "bfloat16", False, "tile"), (64, 4096, 4096, "bfloat16", False, "tile"),
    (33, 14336, 4096, "bfloat16", False, "skinny"), (33, 8192, 8184, "bfloat16", False, "tile"),   # (rows of B inside cache lines)
    (33, 4096, 6144, "int8", False, "skinny"), (48, 6144, 9216, "int8", False, "skinny"), (64, 4096, 4096, "int8", False, "tile"),
    (33, 2048, 4096, "int8", False, "tile"),
    # [N,K] weights
    (33, 11008, 5120, "bfloat16", True, "skinny"), (64, 11008, 5120, "bfloat16", True, "skinny"), (33, 4096, 4096, "bfloat16", True, "tile"),
    (33, 8192, 4096, "bfloat16", True, "tile"), (33, 8192, 8184, "bfloat16", True, "skinny"), (33, 4096, 11008, "int8", True, "tile"), (33, 8192, 6144, "int8", True, "tile"),
])
def test_33_to_64_rows_take_the_faster_of_skinny_and_small_tiles(m, k, n, dtype, tb, kernel, tmp_path):
    note = _schedule(_product(m, k, n, dtype, tb, "rows_%s_%d_%d_%d_%d" % (dtype, m, k, n, tb)), tmp_path)
    assert (" skinny" in note) == (kernel == "skinny") and ("tile=64x64" in note) == (kernel == "tile"), note


@pytest.mark.parametrize("m,k,n,dtype,tb", [
    (800, 11008, 1536, "bfloat16", False), (1600, 11008, 768, "bfloat16", True), (1200, 11008, 1024, "float16", True),   # more than 16 MiB
    (1000, 11008, 1536, "bfloat16", True), (2048, 11008, 768, "bfloat16", False), (3000, 8192, 512, "int8", False),      # at most, for more
    (1000, 8192, 768, "bfloat16", True), (256, 8192, 4096, "bfloat16", False),
])
def test_split_small_tiles_stay_within_the_static_scratch_where_the_large_ones_do(m, k, n, dtype, tb, tmp_path, monkeypatch):
    """16 MiB is what a launch without allocations has. (The largest workspaces among 12000 products that take small tiles, M 33 ..
    8192, K 256 .. 16384, N 64 .. 32768, reach 15 MiB; the first three here had more than 16 while the 256 x 256 kernel did too.)"""
    text = _product(m, k, n, dtype, tb, "scratch_%s_%d_%d_%d_%d" % (dtype, m, k, n, tb))
    small = driver.HipKernel(text, out_dir=None)
    assert "gemm_small_tile<" in small.source
    monkeypatch.setenv("AKG_HIP_VARIANT", "128")
    large = driver.HipKernel(text, out_dir=None)
    assert "gemm_small_tile<" not in large.source
    assert small.workspace_bytes <= 16 << 20 or large.workspace_bytes > 16 << 20
