"""The skinny kernel on a [N,K] weight: whole lines of K through LDS, their tails, ragged columns and split ranges."""
import pytest

from akg_amd import driver, op_desc


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype", [
    (16, 240, 136, "bfloat16"),     # below one line per wavefront: the operands as they are
    (16, 256, 128, "bfloat16"),     # one line each, one strip
    (3, 272, 132, "float16"),       # a quarter of a line behind the last one, four columns beyond a strip
    (1, 1024, 1000, "bfloat16"),    # one row, ragged last strip, split ranges
    (32, 4144, 520, "bfloat16"),    # splits that end on whole lines, a tail of three quarters
    (33, 2048, 516, "float16"),     # two row tiles
    (64, 8192, 264, "bfloat16"),    # the most rows and splits
    (7, 11008, 1040, "bfloat16"),   # more strips than a range has lines: the rotation wraps
    (16, 8192, 6400, "bfloat16"),   # read past the caches
    (32, 8256, 272, "int8"), (5, 544, 140, "int8"),
    # columns that end inside a line: whole lines from 4 MiB of weight on, tails of a quarter, a half and three quarters
    (3, 272, 7720, "float16"), (5, 8256, 520, "int8"), (40, 2096, 1012, "bfloat16"),
    (39, 528, 516, "bfloat16"), (64, 1088, 904, "int8"),   # ... and below: as they are, two row tiles, ragged strips
])
def test_lines_of_a_transposed_weight_against_float64(m, k, n, dtype):
    """float32 sums of k products differ from the exact sum by at most k * 2^-24 of the sum of the products' magnitudes, in
    whatever order, and a result by one half unit of its type; 8-bit sums are exact. Twice: the counters of the split are left ready."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    dev = "cuda"
    if dtype == "int8":
        text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=True)
        a, w = (torch.randint(-127, 128, s, generator=g, device=dev).to(torch.int8) for s in ((m, k), (n, k)))
        scale, scale_n = torch.full((m, 1), 2.0 ** -6, device=dev), torch.full((n,), 2.0 ** -10, device=dev)
        bias = torch.randn(n, generator=g, device=dev).bfloat16()
        y = a.double() @ w.double().t().contiguous() * 2.0 ** -16 + bias.double()
        y = y * (torch.tanh((y + y ** 3 * 0.044715) * 0.7978845608028654) + 1) * 0.5
        # the factors are powers of two; float32 GELU: 2^-20 of the argument's magnitude, and the rounding to bfloat16
        inputs, td, bound = [a, scale, w, scale_n, bias], torch.bfloat16, y.abs() * (2.0 ** -8 + 2.0 ** -19) + 2.0 ** -16
    else:
        td = getattr(torch, dtype)
        text = op_desc.gemm_bias_act(m, k, n, dtype, "none", transpose_b=True)
        a, w, bias = (torch.randn(s, generator=g, device=dev).to(td) for s in ((m, k), (n, k), (n,)))
        y = a.double() @ w.double().t().contiguous() + bias.double()
        sums = a.double().abs() @ w.double().abs().t().contiguous()
        unit = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
        inputs, bound = [a, w, bias], sums * (k * 2.0 ** -24) + y.abs() * (unit + 2.0 ** -23) + 2.0 ** -24
    kernel = driver.HipKernel(text, out_dir=None)
    assert "gemm_skinny<" in kernel.source
    print("case", m, k, n, dtype, kernel.grid, flush=True)
    for _ in range(2):
        out = torch.full((m, n), float("nan"), device=dev, dtype=td)
        kernel.launch(inputs + [out])
        torch.cuda.synchronize()
        gap = (out.double() - y).abs()
        assert bool((gap <= bound).all()), float((gap / bound).max())


def test_every_line_of_the_weight_is_requested_once(tmp_path):
    """512 bytes of K and one strip: each of the four wavefronts has one line of 128 columns, 16 loads of 16 bytes a lane, and
    four of its row of A. A request for a line beyond the last one would be further loads in the code."""
    import glob
    import os
    import subprocess
    driver.HipKernel(op_desc.gemm_bias_act(16, 256, 128, "bfloat16", "none", transpose_b=True), out_dir=str(tmp_path))
    path = glob.glob(os.path.join(str(tmp_path), "**", "*.hsaco"), recursive=True)[0]
    objdump = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
    code = subprocess.run([objdump, "-d", path], check=True, capture_output=True, text=True).stdout
    assert code.count("global_load_dwordx4") == 16 + 4


def test_lines_are_read_past_the_caches_from_96_mib_of_all_batches_on(monkeypatch):
    def streamed(text):
        kernel = driver.HipKernel(text, out_dir=None)
        assert "gemm_skinny<" in kernel.source
        return "akg::StreamedLines()" in kernel.source
    assert streamed(op_desc.gemm_bias_act(16, 8192, 6144, "bfloat16", "none", transpose_b=True))
    assert not streamed(op_desc.gemm_bias_act(16, 8192, 6140, "bfloat16", "none", transpose_b=True))
    assert not streamed(op_desc.gemm_int8_dequant_bias_gelu(16, 8192, 8192, transpose_b=True))
    assert not streamed(op_desc.gemm_bias_act(16, 4112, 12288, "bfloat16", "none", transpose_b=True))   # columns end inside a line
    assert not streamed(op_desc.gemm_bias_act(16, 128, 524288, "bfloat16", "none", transpose_b=True))   # operands as they are
    assert not streamed(op_desc.gemm_bias_act(16, 8192, 8192, "bfloat16", "none", transpose_b=False))
    assert streamed(op_desc.batch_matmul_scale_mask(192, 16, 512, 512, "bfloat16", True, "lines_batch"))
    assert not streamed(op_desc.batch_matmul_scale_mask(191, 16, 512, 512, "bfloat16", True, "lines_batch"))
    monkeypatch.setenv("AKG_HIP_NT", "0")
    assert not streamed(op_desc.gemm_bias_act(16, 8192, 8192, "bfloat16", "none", transpose_b=True))


def test_lines_of_columns_that_end_inside_one_are_whole_from_4_mib_of_all_batches_on():
    def whole(text):
        kernel = driver.HipKernel(text, out_dir=None)
        assert "gemm_skinny<" in kernel.source
        return "akg::NoLines()" not in kernel.source
    assert whole(op_desc.gemm_bias_act(16, 1040, 2020, "bfloat16", "none", transpose_b=True))
    assert not whole(op_desc.gemm_bias_act(16, 1040, 2016, "bfloat16", "none", transpose_b=True))
    assert whole(op_desc.gemm_int8_dequant_bias_gelu(2, 1056, 3972, transpose_b=True))
    assert not whole(op_desc.gemm_int8_dequant_bias_gelu(2, 1056, 3968, transpose_b=True))
    assert whole(op_desc.gemm_bias_act(16, 256, 128, "bfloat16", "none", transpose_b=True))       # columns of whole lines
    assert not whole(op_desc.gemm_bias_act(16, 240, 16384, "bfloat16", "none", transpose_b=True))  # not a line per wavefront
    assert whole(op_desc.batch_matmul_scale_mask(8, 16, 528, 512, "bfloat16", True, "lines_seam"))
    assert not whole(op_desc.batch_matmul_scale_mask(7, 16, 528, 512, "bfloat16", True, "lines_seam"))


def _takes_wide_strips(text):
    source = driver.HipKernel(text, out_dir=None)
    assert "gemm_skinny<" in source.source and "NarrowStrips" not in source.source and source.workspace_bytes > 0
    return source


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype", [(1, 1024, 1000, "bfloat16"), (33, 2048, 516, "float16"), (32, 8256, 272, "int8"), (5, 8256, 520, "int8"), (64, 1088, 904, "int8")])
def test_lines_of_strips_of_128_columns_where_narrow_ones_are_the_default(m, k, n, dtype, monkeypatch):
    """Split ranges, tails and ragged strips of a [N,K] weight, with the bounds of the test above."""
    monkeypatch.setenv("AKG_HIP_VARIANT", "256")
    _takes_wide_strips(op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=True) if dtype == "int8" else op_desc.gemm_bias_act(m, k, n, dtype, "none", transpose_b=True))
    test_lines_of_a_transposed_weight_against_float64(m, k, n, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,k,n,tb", [
    ("bf16", 1, 1024, 520, False), ("bf16", 16, 4096, 1024, False), ("bf16", 33, 2048, 264, False), ("i8", 32, 4096, 260, False), ("i8", 64, 4096, 520, False),
    ("f16", 16, 2048, 264, True), ("f16", 48, 1024, 136, True), ("bf16", 32, 8192, 136, True), ("i8", 50, 8192, 128, True),
])
def test_strips_of_128_columns_with_a_split_against_the_oracle(kind, m, k, n, tb, monkeypatch, tmp_path):
    """One row to 64, both layouts, three element types, ranges of K that workgroups share."""
    from test_gpu_parity import test_skinny_matmul_streams_b_into_mfma_operands as against_the_oracle
    monkeypatch.setenv("AKG_HIP_VARIANT", "256")
    _takes_wide_strips(op_desc.gemm_int8_dequant_bias_gelu(m, k, n, "bfloat16", tb) if kind == "i8" else
                       op_desc.gemm_bias_act(m, k, n, "bfloat16" if kind == "bf16" else "float16", "gelu", tb))
    against_the_oracle((kind, m, k, n, tb), tmp_path)
