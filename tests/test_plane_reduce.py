"""Reductions on both sides of the kept axes whose results meet the tensor again (family plane_reduce): which descriptions
take it, and its results against the oracle's evaluation in float64."""
import json

import numpy as np
import pytest

from akg_amd import driver, harness, op_desc


def _bn(n, c, h, w, dtype):
    return op_desc.batchnorm_train_forward(n, c, h, w, dtype)


def _backward(n, c, h, w):
    """Batch-norm backward: two full-sized inputs, statistics per channel, two sums, three outputs (one without the reduced axes)."""
    b = op_desc.DescBuilder("bn_backward_%dx%dx%dx%d" % (n, c, h, w))
    x, dy = b.input([n, c, h, w], "bfloat16"), b.input([n, c, h, w], "float32")
    gamma, mean = b.input([1, c, 1, 1], "float32"), b.input([1, c, 1, 1], "float32")
    xc = b.sub(b.cast(x, "float32"), mean)
    dgamma = b.reduce("ReduceSum", b.mul(dy, xc), [0, 2, 3], True)
    dbeta = b.reduce("ReduceSum", dy, [0, 2, 3], False)
    inv = b.const(1.0 / (n * h * w), "float32")
    part = b.mul(b.add(b.reshape(dbeta, [1, c, 1, 1]), b.mul(xc, dgamma)), inv)
    return b.dumps([b.mul(b.sub(dy, part), gamma), dgamma, dbeta])


def _range(shape, axes, dtype):
    """(x - min) beside max - min: extrema, two reductions of one level, no rounding at all."""
    b = op_desc.DescBuilder("range_%s_%s" % (dtype, "x".join(map(str, shape))))
    x = b.input(shape, dtype)
    low, high = b.reduce("ReduceMin", x, axes, True), b.reduce("ReduceMax", x, axes, True)
    return b.dumps([b.sub(x, low), b.sub(high, low)])


def _statistics(n, c, h, w):
    """Mean and variance alone: the last launch of the form with several workgroups per channel has values per channel only."""
    b = op_desc.DescBuilder("bn_mean_var_%dx%dx%dx%d" % (n, c, h, w))
    x = b.input([n, c, h, w], "float32")
    inv = b.const(1.0 / (n * h * w), "float32")
    mean = b.mul(b.reduce("ReduceSum", x, [0, 2, 3], True), inv)
    xc = b.sub(x, mean)
    return b.dumps([mean, b.mul(b.reduce("ReduceSum", b.mul(xc, xc), [0, 2, 3], True), inv)])


def test_descriptions_that_take_the_plane_kernel_and_those_that_do_not():
    def family(text):
        return driver.HipKernel(text, out_dir=None).family
    assert family(_bn(4, 16, 8, 8, "bfloat16")) == family(_range([8, 40, 5, 7], [0, 2, 3], "int32")) == "plane_reduce"
    assert family(_bn(4, 15, 8, 8, "bfloat16")) == "staged"       # few channels
    assert family(_bn(2, 16, 8, 8, "bfloat16")) == "staged"       # channels of less than half a wavefront
    b = op_desc.DescBuilder("kept_on_both_sides")
    x = b.input([8, 32, 40, 24], "float32")
    assert family(b.dumps([b.sub(x, b.reduce("ReduceMax", x, [0, 2], True))])) == "staged"
    b = op_desc.DescBuilder("sums_that_round")
    x = b.input([8, 32, 40, 24], "float16")
    assert family(b.dumps([b.sub(x, b.reduce("ReduceSum", x, [0, 2, 3], True))])) == "staged"
    b = op_desc.DescBuilder("dropped_axes_meet_the_last_one")
    x = b.input([8, 32, 40, 32], "float32")
    assert family(b.dumps([b.sub(x, b.reduce("ReduceMax", x, [0, 2, 3], False))])) == "staged"
    b = op_desc.DescBuilder("weight_per_column")
    x, w = b.input([8, 32, 40, 24], "float32"), b.input([24], "float32")
    y = b.mul(x, w)
    assert family(b.dumps([b.sub(y, b.reduce("ReduceMax", y, [0, 2, 3], True))])) == "staged"


def _mixed(shape, dtype):
    """float32 results of a narrow input: chunks of four elements, less than 16 bytes each."""
    b = op_desc.DescBuilder("mixed_%s_%s" % (dtype, "x".join(map(str, shape))))
    x = b.cast(b.input(shape, dtype), "float32")
    return b.dumps([b.sub(x, b.reduce("ReduceMax", x, [0, 2, 3], True))])


def _peak_and_sum(n, c, h, w):
    """A maximum and a sum of one walk."""
    b = op_desc.DescBuilder("peak_and_sum_%dx%dx%dx%d" % (n, c, h, w))
    x = b.input([n, c, h, w], "float16")
    f = b.cast(x, "float32")
    s = b.reduce("ReduceSum", b.mul(f, f), [0, 2, 3], True)
    return b.dumps([b.sub(x, b.reduce("ReduceMax", x, [0, 2, 3], True)), s])


def test_few_channels_of_many_chunks_take_a_launch_per_level():
    def by_level(text):
        kernel = driver.HipKernel(text, out_dir=None)
        assert kernel.family == "plane_reduce"
        return "_level0" in kernel.source
    assert by_level(_range([30000, 32, 2, 3], [0, 2, 3], "int8")) and by_level(_range([64, 32, 64, 64], [0, 2, 3], "int8"))
    assert by_level(_range([8000, 128, 2, 3], [0, 2, 3], "float16")) and by_level(_mixed([64, 16, 63, 63], "int8"))
    assert not by_level(_bn(64, 128, 28, 28, "bfloat16")) and not by_level(_range([64, 128, 64, 64], [0, 2, 3], "int8"))
    assert not by_level(_bn(80, 16, 28, 28, "bfloat16"))    # eight chunks a thread


CASES = [
    (_bn(64, 16, 7, 7, "bfloat16"), "1"),            # a chunk shared by two slots of a run of 49
    (_bn(33, 17, 28, 28, "bfloat16"), "1"),          # whole chunks, the last ones of a thread beyond the channel
    (_bn(40, 16, 3, 1, "float32"), "1"),             # runs of three elements: narrow chunks
    (_bn(127, 16, 31, 33, "float16"), "1"),          # nearly the registers of a workgroup
    (_bn(6, 300, 9, 9, "float16"), "1"),             # many channels of one short workgroup
    (_bn(64, 16, 7, 7, "bfloat16"), "3"),            # several workgroups per channel
    (_bn(9, 19, 33, 35, "float32"), "11"),
    (_bn(5, 16, 200, 210, "float32"), "0"),          # beyond a workgroup's registers
    (_bn(3, 16, 100, 100, "bfloat16"), "60/64"),     # sixty short workgroups per channel
    (_bn(2, 16, 120, 150, "float32"), "150/64"),     # more workgroups per channel than threads in one
    (_backward(12, 20, 14, 14), "1"), (_backward(12, 20, 14, 14), "4"),
    (_range([8, 40, 5, 7], [0, 2, 3], "int32"), "1"), (_range([3, 4, 2, 9, 1, 70], [0, 1, 4, 5], "float16"), "2"),
    (_statistics(8, 24, 30, 30), "1"), (_statistics(8, 24, 30, 30), "5"),
    # extrema: a chunk beyond the channel by a branch, whole and shared ones
    (_range([41, 20, 7, 7], [0, 2, 3], "float16"), "1"), (_range([33, 17, 8, 8], [0, 2, 3], "int8"), "1"), (_range([130, 18, 5, 5], [0, 2, 3], "int8"), "1"),
    (_peak_and_sum(40, 16, 7, 9), "1"), (_peak_and_sum(40, 16, 7, 9), "3"), (_mixed([600, 16, 9, 9], "int8"), "0"), (_range([5000, 16, 2, 3], [0, 2, 3], "int8"), "0"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("index", range(len(CASES)))
def test_results_against_the_oracle(index, monkeypatch):
    """Sums against float64 with the bound of a reassociated float32 sum of their terms; extrema and their differences bit
    for bit. Three launches of one handle give the same bits."""
    import torch
    from oracle import np_ref
    text, schedule = CASES[index]
    split, _, block = schedule.partition("/")
    if split != "0":
        monkeypatch.setenv("AKG_HIP_SPLIT", split)
    if block:
        monkeypatch.setenv("AKG_HIP_BLOCK", block)
    desc = json.loads(text)
    kernel = driver.HipKernel(text, out_dir=None)
    print("case %s split %s: grid %d block %d" % (desc["op"], schedule, kernel.grid[0], kernel.block[0]), flush=True)
    assert kernel.family == "plane_reduce" and (kernel.workspace_bytes > 0) == (split != "1")
    inputs = harness.make_inputs(desc, seed=harness.BASE_SEED + 811 + index)
    wide = [a.astype(np.float64) if a.dtype == np.float32 else a for a in inputs]
    exact = np_ref.evaluate(harness.widen_to_float64(desc), wide)
    sums = any(o["name"] == "ReduceSum" for o in desc["op_desc"])
    terms = int(np.prod(desc["input_desc"][0][0]["shape"]))
    on_device = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).cuda() for a in inputs]
    first = None
    for _ in range(3):
        outs = [torch.full(d.shape, 77, dtype={"bfloat16": torch.int16, "float16": torch.float16, "float32": torch.float32, "int32": torch.int32, "int8": torch.int8}[d.dtype],
                           device="cuda") for d in kernel.outputs]
        kernel.launch(on_device + outs)
        torch.cuda.synchronize()
        got = [o.cpu().numpy() for o in outs]
        first = first or got
        for d, g, f, x in zip(kernel.outputs, got, first, exact):
            assert np.array_equal(g.view(np.uint8), f.view(np.uint8)), d.name
            g = g.view(np.uint16) if d.dtype == "bfloat16" else g
            if d.dtype == "float32" and sums:
                ok, msg = harness.compare_reassociated(g, x, d.dtype, terms)
            else:
                ok, msg = harness.compare(g, x, d.dtype)
            assert ok, "%s output %s: %s" % (desc["op"], d.name, msg)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [((64, 128, 28, 28), "float32"), ((128, 64, 14, 14), "float32"), ((16, 16, 64, 64), "bfloat16")])
def test_mean_and_variance_are_as_exact_as_by_one_kernel_per_level(shape, dtype, monkeypatch):
    """Error of the statistics against float64, 2-norm over channels and draws: at most a tenth above that of the schedule of several
    kernels, whose partial sums meet in trees (the draws scatter by a few hundredths)."""
    import torch

    def errors(kernel):
        wrong = [0.0, 0.0]
        for seed in range(6):
            g = torch.Generator().manual_seed(seed)
            x = (torch.randn(shape, generator=g) + 0.3).to(torch.float32 if dtype == "float32" else torch.bfloat16).cuda()
            ones, zeros = (torch.full((1, shape[1], 1, 1), v, device="cuda") for v in (1.0, 0.0))
            outs = [torch.empty_like(x), torch.empty_like(ones), torch.empty_like(ones)]
            kernel.launch([x, ones, zeros] + outs)
            wide = x.cpu().double()
            mean = wide.mean((0, 2, 3), keepdim=True)
            for i, want in enumerate((mean, ((wide - mean) ** 2).mean((0, 2, 3), keepdim=True))):
                wrong[i] += float(((outs[i + 1].cpu().double() - want).norm() / want.norm()) ** 2)
        return np.sqrt(wrong)
    text = _bn(*shape, dtype)
    one = driver.HipKernel(text, out_dir=None)
    monkeypatch.setenv("AKG_HIP_VARIANT", "7")
    several = driver.HipKernel(text, out_dir=None)
    assert one.family == "plane_reduce" and several.family == "staged"
    assert (errors(one) <= 1.1 * errors(several)).all()


def test_elements_that_stay_unpacked_from_walk_to_walk():
    """Where they fit half of the registers, and where there is something to unpack or to compute: of a single float32 input there is not."""
    def kept(text):
        kernel = driver.HipKernel(text, out_dir=None)
        assert kernel.family == "plane_reduce" and "_level0" not in kernel.source
        return "akg::forget_unpacked" not in kernel.source
    assert kept(_bn(64, 128, 28, 28, "bfloat16")) and kept(_backward(12, 20, 14, 14)) and kept(_range([41, 20, 7, 7], [0, 2, 3], "float16"))
    assert not kept(_range([79, 803, 8, 8], [0, 2, 3], "float32")) and not kept(_bn(64, 128, 28, 28, "float32"))
    assert not kept(_bn(19, 766, 51, 51, "bfloat16")) and kept(_bn(19, 236, 51, 51, "bfloat16"))    # 1024 threads: two workgroups a CU with half of the registers
    assert kept(_bn(127, 49, 21, 24, "float16")) and not kept(_bn(128, 49, 24, 24, "float16"))     # 64 elements a thread of 1024, 72


def test_channels_on_either_side_of_a_launch_per_level():
    def by_level(text):
        return "_level0" in driver.HipKernel(text, out_dir=None).source
    assert not by_level(_bn(73, 16, 28, 32, "bfloat16")) and by_level(_bn(74, 16, 28, 32, "bfloat16"))      # eight and nine chunks a thread
    # us, resident / by level: 13.1 / 7.4, 14.3 / 7.9, 11.9 / 7.8, 9.0 / 7.2
    assert by_level(_bn(201, 16, 21, 21, "float16")) and by_level(_bn(931, 24, 9, 9, "bfloat16")) and by_level(_bn(38, 28, 19, 105, "bfloat16"))
    assert by_level(_bn(73, 21, 32, 36, "float16"))
    assert not by_level(_bn(61, 31, 33, 17, "float32")) and not by_level(_bn(57, 29, 23, 47, "float32"))    # 5.1 / 7.3, 7.4 / 8.2
    assert not by_level(_bn(112, 48, 28, 36, "bfloat16")) and by_level(_bn(116, 48, 28, 36, "bfloat16"))    # 112 and 120
    assert not by_level(_bn(116, 56, 28, 36, "bfloat16"))
