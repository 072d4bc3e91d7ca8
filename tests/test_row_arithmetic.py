"""Float32 arithmetic of the row kernels: the exponential over its whole range, division by a per-row value bit for bit the
IEEE quotient, and rows of any length in a bucket, among them those whose wavefronts leave out chunks."""
import json

import numpy as np
import pytest

from akg_amd import driver, op_desc


def _run(kernel, arrays):
    import torch
    outs = [torch.full(d.shape, float("nan"), device="cuda") for d in kernel.outputs]
    kernel.launch([torch.from_numpy(a).cuda() for a in arrays] + outs)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in outs]


@pytest.mark.gpu
def test_the_exponential_over_its_whole_range():
    """One unit in the last place at most where the result is normal, one step of 2^-149 where it is subnormal (the hardware's
    2^f is good to one unit, f to 2^-26); 0, infinity and NaN where they belong."""
    b = op_desc.DescBuilder("exp_range")
    n = 1 << 21
    kernel = driver.HipKernel(b.dumps([b.unary("Exp", b.input([n], "float32"))]), out_dir=None)
    rng = np.random.default_rng(11)
    for low, high in ((-104.0, 88.722), (-1.0, 1.0), (-1e-5, 1e-5)):
        x = rng.uniform(low, high, n).astype(np.float32)
        special = np.float32([np.inf, -np.inf, np.nan, 88.72283, 88.72284, 100.5, 3e38, -104.0, -120.5, -3e38, 0.0, -0.0, 1e-45, -87.33655, -103.2])
        x[:special.size] = special
        got = _run(kernel, [x])[0]
        with np.errstate(over="ignore", under="ignore"):
            want = np.exp(x.astype(np.float64))
            rounded = want.astype(np.float32)
        finite = np.isfinite(rounded)
        assert np.array_equal(got[~finite], rounded[~finite], equal_nan=True)
        unit = np.maximum(np.spacing(np.abs(rounded[finite])).astype(np.float64), 2.0 ** -149)
        assert (np.abs(got[finite].astype(np.float64) - want[finite]) / unit).max() <= 1.0


@pytest.mark.gpu
def test_division_by_a_row_value_is_the_ieee_quotient():
    """Zeros of both signs, subnormal and tiny dividends, infinities and NaN over positive, negative, tiny and huge divisors."""
    rng = np.random.default_rng(12)
    special = np.float32([0.0, -0.0, 1e-45, -1e-40, 1e-30, 2.0 ** -60, 2.0 ** -61, 2.0 ** 60, 2.0 ** 61, np.inf, -np.inf, np.nan, 3e38])
    for divisors in (np.float32([3.0, -7.0, 1.0, 1e-3, 2.0 ** -60, 2.0 ** 60]), np.float32([1e-25, 1e30, np.inf, 0.0, -0.0, np.nan])):
        x = (rng.standard_normal((6, 1030)) * 10.0 ** rng.uniform(-5, 5, (6, 1030))).astype(np.float32)
        x[:, 5:5 + special.size] = special
        x[:, 600:900] = 0.0
        b = op_desc.DescBuilder("row_division")
        t, d = b.input(list(x.shape), "float32"), b.input([6, 1], "float32")
        kernel = driver.HipKernel(b.dumps([b.div(t, d)]), out_dir=None)
        got = _run(kernel, [x, divisors.reshape(6, 1)])[0]
        with np.errstate(all="ignore"):
            want = x / divisors.reshape(6, 1)
        same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
        assert same.all(), np.argwhere(~same)[:5]


@pytest.mark.gpu
def test_division_by_a_row_maximum_is_the_ieee_quotient():
    """The row kernel's form: the divisor is a reduction, the dividends come in chunks."""
    rng = np.random.default_rng(13)
    x = np.abs(rng.standard_normal((33, 1030))).astype(np.float32)
    x[:, ::3] = 0.0
    x[7, 5:9] = np.float32([1e-40, -0.0, 1e-25, -3.0])
    x[8] = 0.0
    x[9, 4] = np.inf
    b = op_desc.DescBuilder("row_by_maximum")
    t = b.input(list(x.shape), "float32")
    kernel = driver.HipKernel(b.dumps([b.div(t, b.reduce("ReduceMax", t, [1], True))]), out_dir=None)
    assert kernel.family == "row_reduce"
    got = _run(kernel, [x])[0]
    with np.errstate(all="ignore"):
        want = x / x.max(1, keepdims=True)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), np.argwhere(~same)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [257, 300, 383, 385, 509, 511, 1025, 1535, 2047])
def test_rows_that_leave_out_chunks(cols):
    """One code object for every length of the bucket; softmax with a shared mask against float64: relative error of the
    exponential's argument (2^-24 * 130), of the exponential (2^-23) and of a sum of `cols` terms in trees of four."""
    b = op_desc.DescBuilder("chunks_left_out")
    mask, x = b.input([7777, 1, 7778], "float32"), b.input([7777, 5, 7778], "float32")
    s = b.add(x, mask)
    e = b.unary("Exp", b.sub(s, b.reduce("ReduceMax", s, [2], True)))
    doc = json.loads(b.dumps([b.div(e, b.reduce("ReduceSum", e, [2], True))]))
    text = json.dumps(doc).replace("7777", "-1").replace("7778", "-1")
    kernel = driver.HipDynamicKernel(text, None).specialize([[3, 1, cols], [3, 5, cols]])
    rng = np.random.default_rng(cols)
    m = np.where(rng.random((3, 1, cols)) < 0.3, -10000.0, 0.0).astype(np.float32)
    a = (rng.standard_normal((3, 5, cols)) * 4).astype(np.float32)
    got = _run(kernel, [m, a])[0]
    t = a.astype(np.float64) + m
    want = np.exp(t - t.max(2, keepdims=True))
    want /= want.sum(2, keepdims=True)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max() and (np.abs(got - want) <= 2e-5 * want + 1e-30).all()


def _scaled_masked_softmax():
    """softmax(0.125 x + (1 - mask) * -10000) with every extent open."""
    b = op_desc.DescBuilder("scaled_masked_softmax")
    mask, x = b.input([7777, 1, 7778, 7779], "float32"), b.input([7777, 12, 7778, 7779], "float32")
    s = b.add(b.mul(b.sub(b.const(1.0, "float32"), mask), b.const(-10000.0, "float32")), b.mul(b.const(0.125, "float32"), x))
    e = b.unary("Exp", b.sub(s, b.reduce("ReduceMax", s, [3], True)))
    text = b.dumps([b.div(e, b.reduce("ReduceSum", e, [3], True))])
    return text.replace("7777", "-1").replace("7778", "-1").replace("7779", "-1")


def test_rows_that_leave_out_chunks_are_many_and_full_of_arithmetic():
    kernel = driver.HipDynamicKernel(_scaled_masked_softmax(), None)

    def leaves_out(batch, rows, cols):
        return "akg_some" in kernel.specialize([[batch, 1, rows, cols], [batch, 12, rows, cols]]).source
    assert leaves_out(32, 333, 333) and leaves_out(16, 342, 509)
    assert leaves_out(32, 333, 400) and leaves_out(32, 333, 700) and not leaves_out(16, 341, 333) and not leaves_out(3, 2, 471)
    b = op_desc.DescBuilder("plain_softmax")
    x = b.input([7777, 7778], "float32")
    e = b.unary("Exp", b.sub(x, b.reduce("ReduceMax", x, [1], True)))
    text = b.dumps([b.div(e, b.reduce("ReduceSum", e, [1], True))]).replace("7777", "-1").replace("7778", "-1")
    assert "akg_some" not in driver.HipDynamicKernel(text, None).specialize([[100000, 333]]).source


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [130, 257, 258, 383, 385, 400, 509, 511, 700])
def test_many_rows_that_leave_out_chunks(cols):
    """As above, 65664 rows; the argument of the exponential is at most 10000 + 2 wide where it is masked (then the exponential is
    zero on both sides) and 4 elsewhere."""
    import torch
    shapes = [[16, 1, 342, cols], [16, 12, 342, cols]]
    kernel = driver.HipDynamicKernel(_scaled_masked_softmax(), None).specialize(shapes)
    assert "akg_some" in kernel.source
    g = torch.Generator(device="cuda").manual_seed(cols)
    mask = (torch.rand(shapes[0], generator=g, device="cuda") > 0.3).float()
    x = torch.randn(shapes[1], generator=g, device="cuda") * 4
    out = torch.full(shapes[1], float("nan"), device="cuda")
    kernel.launch([mask, x, out])
    want = torch.softmax((1.0 - mask.double()) * -10000.0 + 0.125 * x.double(), -1)
    wrong = (out.double() - want).abs()
    assert bool((wrong <= 2e-5 * want + 1e-30).all())


def _row_kernel(kind, rows, cols, dtype):
    name = "threads_%s_%s_%d_%d" % (kind, dtype, rows, cols)
    text = {"softmax": lambda: op_desc.softmax_last_axis(rows, cols, dtype, name), "rmsnorm": lambda: op_desc.rmsnorm(rows, cols, dtype, name=name),
            "rmsnorm_add": lambda: op_desc.rmsnorm(rows, cols, dtype, residual=True, name=name), "layernorm": lambda: op_desc.layernorm_residual(rows, cols, dtype, name=name),
            "quant": lambda: op_desc.quant_int8_residual(rows, cols, dtype, name=name), "argmax": lambda: op_desc.argmax_last_axis([rows, cols], dtype, name=name)}[kind]()
    return text, driver.HipKernel(text, out_dir=None)


@pytest.mark.parametrize("kind,rows,cols,dtype,grid,block", [
    # us on the threads of the rules for many rows / until each has one chunk
    ("argmax", 1908, 1104, "float16", 239, 256), ("argmax", 243, 656, "float32", 61, 256), ("argmax", 96, 8600, "bfloat16", 96, 256),   # 2.0 / 2.8, 1.8 / 2.0, 2.3 / 2.4
    ("rmsnorm", 11, 3024, "float32", 11, 256), ("rmsnorm_add", 30, 2584, "float32", 30, 256), ("layernorm", 16, 5888, "float16", 16, 256),   # 1.8 / 1.9, 2.1 / 2.3, 2.4 / 2.6
    ("softmax", 83, 8350, "bfloat16", 83, 256), ("rmsnorm", 68, 14108, "bfloat16", 68, 256),                       # 2.9 / 3.1, 3.0 / 3.2
    ("layernorm", 29, 512, "float32", 8, 256), ("softmax", 39, 512, "float32", 10, 256),                           # 1.75 / 1.87, 1.88 / 1.94
    ("rmsnorm_add", 3345, 560, "float32", 419, 256), ("layernorm", 1997, 1496, "bfloat16", 500, 256),              # 4.0 / 4.6, 3.7 / 4.2
    ("layernorm", 3302, 304, "float32", 413, 256),                                                                # 2.6 / 2.9 on 64 threads
    ("layernorm", 705, 528, "float32", 177, 256), ("layernorm", 1439, 684, "bfloat16", 180, 256),                  # 2.0 / 2.3, 2.4 / 2.6
    # ... and where they pay
    ("quant", 152, 7120, "bfloat16", 152, 512), ("layernorm", 25, 13480, "bfloat16", 25, 512), ("quant", 744, 810, "bfloat16", 372, 256),   # 6.6 / 3.8, 4.9 / 3.9, 6.2 / 3.3
])
def test_threads_of_few_rows(kind, rows, cols, dtype, grid, block):
    _, kernel = _row_kernel(kind, rows, cols, dtype)
    assert kernel.grid[0] == grid and kernel.block[0] == block


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,dtype,block", [
    ("softmax", 33, 3376, "float16", 512), ("softmax", 67, 3401, "bfloat16", 512),      # one ragged chunk a thread; the last one overlaps
    ("softmax", 129, 1536, "float32", 512), ("rmsnorm", 78, 1584, "float32", 512),      # four float32 a thread
    ("rmsnorm", 127, 2535, "bfloat16", 512), ("rmsnorm_add", 77, 4800, "bfloat16", 512),   # two chunks of 512 threads, the second one ragged
    ("rmsnorm", 10, 1023, "float32", 256), ("softmax", 10, 24, "float16", 256),         # the fewest rows; of three chunks
    ("rmsnorm_add", 1023, 1000, "float32", 256), ("layernorm", 21, 2296, "bfloat16", 512), ("layernorm", 1253, 712, "bfloat16", 256),
    ("argmax", 39, 1111, "float32", 256),
])
def test_rows_on_more_threads_against_the_oracle(kind, rows, cols, dtype, block):
    """float32 results of sums of `cols` terms: 1e-5 relative to the float64 evaluation, with 1e-6 of the root of the terms for sums that cancel;
    16-bit ones and integers with the bars of their type against the oracle."""
    import torch
    from akg_amd import harness
    from oracle import np_ref
    text, kernel = _row_kernel(kind, rows, cols, dtype)
    assert kernel.block[0] == block
    print("case", kind, rows, cols, dtype, kernel.grid, kernel.block, flush=True)
    desc = json.loads(text)
    inputs = harness.make_inputs(desc, seed=harness.BASE_SEED + 850)
    expect = np_ref.evaluate(desc, inputs)
    exact = np_ref.evaluate(harness.widen_to_float64(desc), [a.astype(np.float64) if a.dtype == np.float32 else a for a in inputs])
    on_device = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).cuda() for a in inputs]
    for _ in range(2):
        outs = [torch.full((d.nbytes,), 0x7f, dtype=torch.uint8, device="cuda") for d in kernel.outputs]
        kernel.launch(on_device + outs)
        torch.cuda.synchronize()
        for d, o, e, x in zip(kernel.outputs, outs, expect, exact):
            got = o.cpu().numpy().view(driver.NP_HOST_DTYPE[d.dtype]).reshape(d.shape)
            ok, msg = harness.compare_reassociated(got, x, d.dtype, cols) if d.dtype == "float32" else harness.compare(got, e, d.dtype)
            assert ok, "%s %s: %s" % (kind, d.name, msg)
