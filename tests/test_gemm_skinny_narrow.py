"""The skinny kernel on narrow strips: which products take them, and their results at the edges of strips, units of K and rows."""
import re

import pytest

from akg_amd import driver, op_desc
from gemm_checks import compiled_notes


def _columns(text):
    """Columns of a strip; none of another kernel."""
    found = re.search(r"gemm_skinny<.*akg::NarrowStrips<(\d+)>\(\)", driver.HipKernel(text, out_dir=None).source)
    return found and int(found.group(1))


def test_products_that_take_narrow_strips():
    def columns(m, k, n, dtype="bfloat16", tb=True):
        if dtype == "int8":
            return _columns(op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=tb))
        return _columns(op_desc.gemm_bias_act(m, k, n, dtype, "none", transpose_b=tb))
    assert columns(8, 640, 1336) == 16 and columns(9, 1024, 8000) == 32 and columns(25, 896, 5656, tb=False) == 32
    assert columns(1, 1920, 4808, "int8", False) == 64 and columns(9, 2688, 3760, "int8") == 16
    # few strips with a long K, rows of A that weigh more than the columns, weights from 96 MiB on (24 with more than 32 rows)
    assert columns(5, 6592, 560, tb=False) is None and columns(62, 6272, 6720) is None and columns(16, 8192, 8192) is None
    assert columns(33, 4096, 11008, "int8") is None
    assert columns(16, 1040, 2016) is None   # K is not a multiple of 64 bytes


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype,tb", [
    (1, 640, 20, "bfloat16", True), (1, 640, 1216, "bfloat16", False),      # one row; fewer columns than a strip
    (8, 672, 1336, "float16", True), (9, 672, 1300, "float16", False),      # half a unit of K behind the last one; a ninth row
    (16, 4928, 4004, "bfloat16", True), (15, 1344, 1684, "bfloat16", False),
    (17, 2560, 10756, "bfloat16", True), (25, 896, 5656, "float16", False),  # two row tiles, strips of 64 and of 32
    (32, 1312, 1096, "float16", True), (33, 320, 1032, "bfloat16", True), (59, 768, 1028, "bfloat16", False),   # three and four row tiles
    (64, 704, 1060, "float16", True), (3, 1696, 12064, "bfloat16", False),
    (1, 704, 4808, "int8", False), (17, 1984, 4164, "int8", False), (49, 1856, 11256, "int8", False),
    (5, 1344, 764, "int8", True), (32, 832, 4580, "int8", True), (60, 1216, 736, "int8", True),   # columns that begin inside a line
    (16, 1152, 11204, "bfloat16", True), (29, 1376, 11988, "float16", True), (25, 1600, 8740, "int8", True),   # eight wavefronts, strips of 64 of [N,K]
])
def test_narrow_strips_against_float64(m, k, n, dtype, tb):
    """float32 sums of k products differ from the exact sum by at most k * 2^-24 of the sum of the products' magnitudes, in
    whatever order, and a result by one half unit of its type; 8-bit sums are exact."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    dev = "cuda"
    weight = (n, k) if tb else (k, n)
    if dtype == "int8":
        text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=tb)
        a, w = (torch.randint(-127, 128, s, generator=g, device=dev).to(torch.int8) for s in ((m, k), weight))
        scale, scale_n = torch.full((m, 1), 2.0 ** -6, device=dev), torch.full((n,), 2.0 ** -10, device=dev)
        bias = torch.randn(n, generator=g, device=dev).bfloat16()
        wide = w.double().t().contiguous() if tb else w.double()
        y = a.double() @ wide * 2.0 ** -16 + bias.double()
        y = y * (torch.tanh((y + y ** 3 * 0.044715) * 0.7978845608028654) + 1) * 0.5
        # the factors are powers of two; float32 GELU: 2^-20 of the argument's magnitude, and the rounding to bfloat16
        inputs, td, bound = [a, scale, w, scale_n, bias], torch.bfloat16, y.abs() * (2.0 ** -8 + 2.0 ** -19) + 2.0 ** -16
    else:
        td = getattr(torch, dtype)
        text = op_desc.gemm_bias_act(m, k, n, dtype, "none", transpose_b=tb)
        a, w, bias = (torch.randn(s, generator=g, device=dev).to(td) for s in ((m, k), weight, (n,)))
        wide = w.double().t().contiguous() if tb else w.double()
        y = a.double() @ wide + bias.double()
        unit = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
        inputs, bound = [a, w, bias], (a.double().abs() @ wide.abs()) * (k * 2.0 ** -24) + y.abs() * (unit + 2.0 ** -23) + 2.0 ** -24
    print("case", m, k, n, dtype, tb, _columns(text), flush=True)
    assert _columns(text) is not None
    kernel = driver.HipKernel(text, out_dir=None)
    assert kernel.workspace_bytes == 0
    out = torch.full((m, n), float("nan"), device=dev, dtype=td)
    kernel.launch(inputs + [out])
    torch.cuda.synchronize()
    gap = (out.double() - y).abs()
    assert bool((gap <= bound).all()), float((gap / bound).max())


@pytest.mark.parametrize("m,k,n,dtype", [
    (4, 960, 15104, "float16"), (9, 768, 12096, "float16"), (16, 1152, 11200, "bfloat16"), (16, 3072, 10708, "int8"), (20, 1472, 9192, "bfloat16"),
    (25, 1600, 8736, "int8"), (30, 2048, 11000, "int8"), (32, 1024, 12288, "bfloat16"), (32, 2048, 12288, "bfloat16"), (29, 1344, 11984, "float16"),
])
def test_eight_wavefronts_of_64_columns_stay_in_registers(m, k, n, dtype, tmp_path):
    text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=True) if dtype == "int8" else op_desc.gemm_bias_act(m, k, n, dtype, "relu", transpose_b=True)
    kernel, scratch, _ = compiled_notes(text, tmp_path)
    assert "akg::NarrowStrips<64>()" in kernel.source and kernel.block[0] == 512 and scratch == 0


@pytest.mark.parametrize("m,k,n,dtype,tb", [
    # rows of a [K,N] weight that lie a multiple of 256 bytes apart: us on strips of 128 columns / narrow ones
    (2, 3584, 5120, "int8", False), (8, 2240, 23552, "int8", False),             # 8.3 / 13.1, 15.0 / 20.6
    (8, 4096, 8192, "float16", False), (3, 3584, 3072, "bfloat16", False),       # 14.9 / 19.5, 8.9 / 10.9
    (2, 2080, 5120, "bfloat16", False), (16, 3584, 4608, "int8", False),         # 8.3 / 9.4, 8.5 / 9.7
    (4, 2048, 5120, "int8", False), (2, 2560, 6144, "int8", False),              # 7.0 / 8.5, 7.6 / 8.4
    (29, 3616, 7424, "bfloat16", False), (16, 5824, 8960, "int8", False),        # 15.1 / 18.3, 15.3 / 19.9
    # long columns of a [N,K] weight that begin inside lines
    (4, 5216, 256, "bfloat16", True), (2, 6880, 936, "bfloat16", True), (2, 13888, 1008, "int8", True),   # 6.0 / 6.9, 7.8 / 9.1, 8.0 / 8.9
    # small tiles without a split
    (43, 1184, 4416, "bfloat16", True), (46, 1088, 4208, "float16", True), (45, 2176, 7720, "int8", True),   # 6.8 / 7.4, 6.1 / 6.6, 7.2 / 7.7
])
def test_products_that_narrow_strips_would_slow_down(m, k, n, dtype, tb):
    text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=tb) if dtype == "int8" else op_desc.gemm_bias_act(m, k, n, dtype, "none", transpose_b=tb)
    assert _columns(text) is None


@pytest.mark.parametrize("tb,way", [(True, "by whole lines, all of K"), (False, "transposed in registers, all of K")])
def test_the_schedule_note_says_how_the_weight_is_read(tb, way, tmp_path):
    kernel = driver.HipKernel(op_desc.gemm_bias_act(8, 640, 1336, "bfloat16", "none", transpose_b=tb), out_dir=str(tmp_path))
    assert "akg::NarrowStrips<" in kernel.source
    assert any("B " + way in f.read_text() for f in tmp_path.glob("*.json"))
