"""Column sums over rows that are not whole cache lines: the strips of a row run on one XCD, and their loads take no hint."""
import json

import numpy as np
import pytest

from akg_amd import driver, harness, op_desc


def test_rows_of_whole_lines_keep_the_hint():
    ragged = driver.HipKernel(op_desc.bias_grad(4100, 3000, "bfloat16"), out_dir=None).source
    assert "xcd_contiguous_id" in ragged and "V, true>(b_in" not in ragged
    whole = driver.HipKernel(op_desc.bias_grad(4100, 3072, "bfloat16"), out_dir=None).source
    assert "xcd_contiguous_id" not in whole and "V, true>(b_in" in whole
    one_strip = driver.HipKernel(op_desc.bias_grad(40000, 60, "float32"), out_dir=None).source   # nothing that another strip reads
    assert "xcd_contiguous_id" not in one_strip and "V, true>(b_in" in one_strip


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,dtype", [(700, 1111, "bfloat16"), (4100, 130, "float32"), (3000, 4095, "float16"), (257, 72, "bfloat16"), (5000, 60, "float32")])
def test_column_sums_of_ragged_rows(rows, cols, dtype):
    """Against float64, with the bound of a reassociated float32 sum of `rows` terms; an elementwise result stored beside it
    bit for bit."""
    import torch
    from oracle import np_ref
    b = op_desc.DescBuilder("ragged_%s_%dx%d" % (dtype, rows, cols))
    x = b.input([rows, cols], dtype)
    y = b.mul(b.cast(x, "float32") if dtype != "float32" else x, b.const(3.0, "float32"))
    text = b.dumps([y, b.reduce("ReduceSum", y, [0], False)])
    kernel = driver.HipKernel(text, out_dir=None)
    print("case %s: grid %d" % (kernel.kernel_name, kernel.grid[0]), flush=True)
    assert kernel.family == "stream_reduce"
    desc = json.loads(text)
    inputs = harness.make_inputs(desc, seed=harness.BASE_SEED + 813)
    exact = np_ref.evaluate(harness.widen_to_float64(desc), [a.astype(np.float64) if a.dtype == np.float32 else a for a in inputs])
    plain = np_ref.evaluate(desc, inputs)
    for _ in range(2):
        outs = [torch.full(d.shape, float("nan"), device="cuda") for d in kernel.outputs]
        kernel.launch([torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda() for a in inputs] + outs)
        torch.cuda.synchronize()
        assert np.array_equal(outs[0].cpu().numpy(), plain[0])
        ok, msg = harness.compare_reassociated(outs[1].cpu().numpy(), exact[1], "float32", 9 * rows)
        assert ok, msg
