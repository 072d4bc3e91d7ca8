"""The 256 x 256 tile kernel on several rows of tiles whose last row, last column or last step of K is not whole."""
import pytest

from akg_amd import driver, op_desc
from gemm_checks import compiled_notes, disassembled


@pytest.mark.gpu
@pytest.mark.parametrize("tb", [True, False])
@pytest.mark.parametrize("m,k,n,dtype", [
    (257, 512, 260, "bfloat16"), (511, 40, 516, "float16"),         # one row, four columns behind a tile; less than a step of K
    (512, 608, 8200, "bfloat16"), (300, 2056, 1016, "float16"),     # whole rows of tiles only; 16 bytes of K behind the last step, split
    (770, 2104, 1276, "bfloat16"), (1500, 1088, 4092, "float16"),   # 112 bytes of K behind the last step; many tiles, none of them split
    (300, 1056, 1024, "bfloat16"), (600, 544, 4160, "float16"), (513, 1040, 1088, "int8"),   # rows of whole 64-byte pieces
    (300, 2064, 1028, "int8"), (513, 1136, 2296, "int8"), (768, 64, 4100, "int8"), (2048, 4112, 2052, "int8"),
])
def test_ragged_tiles_against_float64(m, k, n, dtype, tb, monkeypatch):
    """float32 sums of k products differ from the exact sum by at most k * 2^-24 of the sum of the products' magnitudes, in
    whatever order, and a result by one half unit of its type; 8-bit sums are exact."""
    import torch
    monkeypatch.setenv("AKG_HIP_VARIANT", "128")   # (small tiles take some of them)
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
    print("case", m, k, n, dtype, tb, flush=True)
    kernel = driver.HipKernel(text, out_dir=None)
    assert "gemm_256x256<" in kernel.source
    # (behind the result: nothing of a row or column that the product does not have)
    out = torch.full((m + 1, n), float("nan"), device=dev, dtype=td)
    kernel.launch(inputs + [out[:m]])
    torch.cuda.synchronize()
    gap = (out[:m].double() - y).abs()
    assert bool((gap <= bound).all()), float((gap / bound).max())
    assert bool(out[m].isnan().all())


@pytest.mark.gpu
def test_k_rows_behind_a_weight_of_nearly_2_gib_read_zero(monkeypatch):
    """The last step of K has 8 of its 64 k-rows; those from 4112 on would begin 2 GiB and more behind the weight's first byte. An infinity in
    one place of the weight (row 7, where an offset that has wrapped around would lie) reaches its own columns only."""
    import torch
    monkeypatch.setenv("AKG_HIP_VARIANT", "128")
    m, k, n, at = 257, 4104, 261632, 257536
    assert 2 * n * k < 1 << 31 <= 2 * n * 4112 and 2 * n * 4112 - (1 << 31) == 2 * (7 * n + at)
    kernel = driver.HipKernel(op_desc.gemm_bias_act(m, k, n, "bfloat16", "none", transpose_b=False), out_dir=None)
    assert "gemm_256x256<" in kernel.source
    print("case", m, k, n, flush=True)
    dev = "cuda"
    a, w = torch.ones((m, k), device=dev, dtype=torch.bfloat16), torch.zeros((k, n), device=dev, dtype=torch.bfloat16)
    w[7, at:at + 8] = float("inf")
    out = torch.zeros((m, n), device=dev, dtype=torch.bfloat16)
    kernel.launch([a, w, torch.ones(n, device=dev, dtype=torch.bfloat16), out])
    torch.cuda.synchronize()
    own = torch.zeros(n, device=dev, dtype=torch.bool)
    own[at:at + 8] = True
    assert bool(out[:, own].isinf().all()) and bool((out[:, ~own] == 1).all())


@pytest.mark.parametrize("m,k,n,dtype", [
    (3979, 360, 8780, "float16"), (571, 352, 9424, "bfloat16"), (2804, 304, 9272, "bfloat16"), (5850, 440, 11392, "float16"),
    (4033, 272, 2376, "bfloat16"), (512, 232, 1024, "float16"), (300, 168, 516, "bfloat16"), (6986, 384, 12096, "bfloat16"), (7857, 448, 2368, "int8"),
])
def test_few_steps_of_k_stay_in_registers(m, k, n, dtype, monkeypatch, tmp_path):
    """A [K,N] weight and three to eight steps of K, the last one ragged or not."""
    monkeypatch.setenv("AKG_HIP_VARIANT", "128")
    text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n) if dtype == "int8" else op_desc.gemm_bias_act(m, k, n, dtype, "relu")
    kernel, scratch, _ = compiled_notes(text, tmp_path)
    assert "gemm_256x256<" in kernel.source and scratch == 0


@pytest.mark.parametrize("n,swaps", [(12, False), (64, False), (80, False), (124, False), (128, False), (132, True), (192, False), (200, True)])
def test_up_to_128_columns_are_stored_by_every_lane(n, swaps, tmp_path):
    """The exchange between column groups leaves the lanes of the second one idle where that has no columns."""
    text = op_desc.batch_matmul_scale_mask(4, 158, 128, n, "bfloat16", True, "pairs_%d" % n)
    kernel, code = disassembled(text, tmp_path)
    assert "gemm_256x256<" in kernel.source and ("v_permlane16_swap" in code) == swaps
