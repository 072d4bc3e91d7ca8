"""Workgroups of several small tiles: which products take them, and their results at the edges."""
import re
import subprocess

import pytest

from akg_amd import driver, op_desc
from test_gemm_small_tiles import _product, test_small_tiles_against_float64 as _against_float64


def _tile(m, k, n, dtype, tb):
    """Rows, columns and splits of a workgroup; none of another kernel."""
    source = driver.HipKernel(_product(m, k, n, dtype, tb, "groups"), out_dir=None).source
    found = re.search(r"gemm_small_tile<[^,]+, (\d+), (\d+), [^(]*?(\d+)>\(", source)
    return found and tuple(int(x) for x in found.groups())


def test_products_that_take_several_tiles_a_workgroup():
    assert _tile(1059, 1704, 3604, "bfloat16", True) == (192, 128, 1)
    assert _tile(1589, 2968, 5200, "bfloat16", False) == (192, 192, 1)
    assert _tile(1312, 2432, 5040, "int8", False) == (128, 256, 1)
    # at most 16 steps of K take single tiles, at most 64 rows always
    assert _tile(1059, 1024, 3604, "bfloat16", True) == (64, 128, 1)
    assert _tile(48, 4096, 4096, "bfloat16", True)[:2] == (64, 64)
    # weights below 2 MiB, unless their columns are whole tiles of the 256 x 256 kernel or there are few rows
    assert _tile(365, 1408, 744, "bfloat16", False)[:2] == (64, 64)
    assert _tile(365, 1408, 512, "bfloat16", False) is None and _tile(48, 1408, 744, "bfloat16", False) is None


@pytest.mark.parametrize("m,k,n,dtype,tb", [
    (69, 11776, 4504, "bfloat16", True), (1079, 12080, 464, "float16", False), (338, 13712, 1368, "bfloat16", True),
    (4329, 11200, 120, "bfloat16", False), (4816, 2240, 840, "int8", False), (2518, 2528, 808, "int8", True), (8176, 2176, 584, "int8", True),
    (370, 4088, 3440, "bfloat16", False),
])
def test_partials_fit_a_launch_without_allocations(m, k, n, dtype, tb):
    """Such a launch has 16 MiB; the kernels that these products had before ask for less or nothing."""
    kernel = driver.HipKernel(_product(m, k, n, dtype, tb, "partials"), out_dir=None)
    assert "gemm_small_tile" in kernel.source and kernel.workspace_bytes <= 16 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype,tb,tile", [
    (1059, 1704, 3604, "bfloat16", True, (192, 128, 1)),    # ragged rows and columns, a K tail of 80 bytes
    (1102, 1592, 5120, "float16", False, (192, 128, 1)),
    (1240, 2384, 3360, "int8", False, (192, 128, 1)),
    (1460, 2080, 2984, "int8", True, (192, 128, 1)),
    (1580, 1576, 5008, "bfloat16", True, (192, 192, 1)),
    (1365, 2104, 6144, "bfloat16", False, (192, 192, 1)),
    (2371, 2368, 3440, "int8", False, (192, 192, 1)),       # 192 columns of 8 bits: two k-rows a cycle of banks
    (1383, 1520, 4808, "bfloat16", True, (128, 256, 1)),
    (1133, 2520, 5520, "float16", False, (128, 256, 1)),
    (1312, 2432, 5040, "int8", False, (128, 256, 1)),
    (370, 4088, 3440, "bfloat16", False, (128, 128, 2)),    # split 128 x 128 tiles
    (340, 9792, 2792, "int8", True, (128, 128, 2)),
    (365, 1408, 744, "bfloat16", False, (64, 64, 1)),       # small weights
    (365, 2088, 492, "bfloat16", True, (64, 64, 4)),
    (85, 4000, 248, "float16", True, (64, 64, 8)),
    (71, 14272, 4496, "bfloat16", True, (64, 64, 4)),       # eight would ask for more than the launch without allocations has
    (2518, 2528, 808, "int8", True, (128, 128, 1)),         # ... as would two
    (65, 64, 68, "bfloat16", True, (64, 64, 1)),            # one step
    (219, 3776, 5640, "int8", False, None),                 # rows of B that are not whole 16-byte chunks
    (836, 2064, 9240, "int8", False, None), (97, 1040, 1004, "int8", False, None),
])
def test_tile_groups_against_float64(m, k, n, dtype, tb, tile, tmp_path):
    """The bound of the small tiles' own test: any order of float32 sums, 8-bit products exactly."""
    got = _tile(m, k, n, dtype, tb)
    assert got == tile if tile else got
    units = "%dx%d" % tuple(128 if x % 128 == 0 else 64 for x in got[:2])
    _against_float64(m, k, n, dtype, tb, units, tmp_path)


@pytest.mark.parametrize("m,k,n", [(1576, 1728, 2640), (2282, 1792, 11456), (801, 960, 11712), (1249, 1728, 9368)])
def test_two_workgroups_of_128_x_128_fit_a_cu(m, k, n, tmp_path):
    """Their four wavefronts have 256 registers each; with more a CU takes one of them only."""
    assert _tile(m, k, n, "int8", False) == (128, 128, 1)
    kernel = driver.HipKernel(_product(m, k, n, "int8", False, "registers"), out_dir=str(tmp_path))
    code = next(str(f) for f in tmp_path.glob("*.hsaco") if kernel.kernel_name.startswith(f.stem))
    notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", code], capture_output=True, text=True, check=True).stdout
    assert int(re.search(r"\.vgpr_count:\s+(\d+)", notes).group(1)) <= 256
    assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", notes).group(1)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,dtype,tb", [
    (65, 448, 256, "bfloat16", False), (257, 64, 512, "float16", True), (512, 1008, 768, "bfloat16", True),   # K below 512 and 1024
    (513, 1024, 256, "float16", False), (300, 1024, 1024, "int8", False), (2048, 768, 768, "bfloat16", False),
    (513, 2040, 512, "bfloat16", True), (1500, 1088, 1792, "int8", True),
    (65, 8192, 8196, "bfloat16", True), (300, 8192, 8200, "float16", False), (320, 8208, 8200, "int8", True), (129, 8208, 8196, "int8", False),   # large ones
])
def test_small_weights_of_whole_wide_columns_and_large_ones_of_ragged(m, k, n, dtype, tb, tmp_path):
    """Weights below 2 MiB whose columns are whole 256-wide tiles take small tiles too, but for a few products with a long K,
    and so do those from 2^26 elements on whose columns are not."""
    got = _tile(m, k, n, dtype, tb)
    assert got is not None
    _against_float64(m, k, n, dtype, tb, "%dx%d" % tuple(128 if x % 128 == 0 else 64 for x in got[:2]), tmp_path)


@pytest.mark.parametrize("m,k,n,dtype,act,tb", [
    (4630, 14424, 432, "bfloat16", "none", False), (1106, 13632, 2992, "bfloat16", "gelu", False), (5852, 8160, 368, "bfloat16", "gelu", True),
    (8100, 8128, 384, "bfloat16", "none", False),
])
def test_products_of_small_tiles_fit_a_launch_without_allocations_still(m, k, n, dtype, act, tb):
    """The 256 x 256 kernel would ask for 40 to 67 MB of partials here."""
    kernel = driver.HipKernel(op_desc.gemm_bias_act(m, k, n, dtype, act, transpose_b=tb), out_dir=None)
    assert kernel.workspace_bytes <= 16 << 20


@pytest.mark.parametrize("m,k,n,dtype,act,tb,small", [
    # few steps of K, and GELU behind the sums: us on small tiles / 256 x 256
    (6345, 448, 5164, "bfloat16", "none", True, True), (3822, 704, 9200, "bfloat16", "relu", True, True),      # 43 / 54, 59 / 71
    (5859, 320, 11392, "float16", "none", False, True), (6660, 128, 3088, "bfloat16", "gelu", True, True),     # 63 / 76, 20 / 30
    (7633, 832, 2704, "float16", "gelu", False, True), (4524, 312, 5368, "bfloat16", "gelu", False, True),     # 54 / 62, 30 / 40
    (618, 384, 15488, "float16", "relu", False, True),                                                        # 15.3 / 17.4
    (216, 16128, 8872, "float16", "none", False, False),                                                      # 151 / 141
    (3520, 4096, 7892, "int8", "none", True, False), (5072, 1984, 5568, "float16", "relu", False, False),     # 126 / 121, 120 / 112
    (216, 12544, 9016, "int8", "gelu", True, True),
])
def test_the_faster_tiles_are_chosen(m, k, n, dtype, act, tb, small):
    text = op_desc.gemm_int8_dequant_bias_gelu(m, k, n, transpose_b=tb) if dtype == "int8" else op_desc.gemm_bias_act(m, k, n, dtype, act, transpose_b=tb)
    assert ("gemm_small_tile<" in driver.HipKernel(text, out_dir=None).source) == small
