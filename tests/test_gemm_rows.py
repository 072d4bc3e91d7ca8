"""A contraction and the reductions over its rows in one kernel (family gemm_rows): which descriptions take it, and its
results against float64."""
import numpy as np
import pytest

from akg_amd import driver, op_desc


def _scores(batch, m, k, n, dtype, mask, outputs, transpose_b=True):
    """exp(s - max s) and friends of s = Q K^T * scale + mask; mask: shape of a float32 input or None."""
    b = op_desc.DescBuilder("scores_%s_%dx%dx%dx%d_%s" % (dtype, batch, m, k, n, "_".join(outputs)))
    lead = [batch] if batch else []
    q, kk = b.input(lead + [m, k], dtype), b.input(lead + ([n, k] if transpose_b else [k, n]), dtype)
    x = b.input(mask, "float32") if mask else None
    attrs = [{"data_type": "bool", "name": "transpose_a", "value": False},
             {"data_type": "bool", "name": "transpose_b", "value": transpose_b}]
    s = b.op("BatchMatMul" if batch else "MatMul", [q, kk], lead + [m, n], "float32", attrs=attrs)
    s = b.mul(s, b.const(k ** -0.5, "float32"))
    if mask:
        s = b.add(s, x)
    axis = [len(lead) + 1]
    top = b.reduce("ReduceMax", s, axis, True)
    e = b.unary("Exp", b.sub(s, top))
    total = b.reduce("ReduceSum", e, axis, True)
    made = {"p": lambda: b.cast(b.div(e, total), dtype), "p32": lambda: b.div(e, total), "max": lambda: top, "sum": lambda: total,
            "sum_flat": lambda: b.reduce("ReduceSum", e, axis, False)}
    return b.dumps([made[o]() for o in outputs])


def test_descriptions_that_take_the_row_kernel_and_those_that_do_not():
    def family(text):
        return driver.HipKernel(text, out_dir=None).family
    assert family(op_desc.attention_probabilities(64, 333, 64, 328, "float16")) == "gemm_rows"
    assert family(_scores(0, 2048, 64, 512, "bfloat16", [1, 512], ["p32", "max"])) == "gemm_rows"
    for text in (op_desc.attention_probabilities(2, 512, 64, 64, "bfloat16"),           # scores that stay in the caches
                 op_desc.attention_probabilities(384, 3, 64, 2048, "bfloat16"),         # too few rows
                 op_desc.attention_probabilities(16, 256, 128, 2048, "bfloat16"),       # a large B
                 op_desc.attention_probabilities(64, 256, 64, 324, "bfloat16"),         # N is not a multiple of 8
                 op_desc.attention_probabilities(64, 256, 72, 328, "bfloat16"),         # K is not whole MFMA slabs
                 _scores(64, 256, 64, 256, "bfloat16", [64, 256, 256], ["p"], transpose_b=False)):
        assert family(text) == "staged"


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,k,n,dtype,mask,outputs", [
    (64, 333, 64, 328, "bfloat16", [64, 333, 328], ["p"]),          # ragged rows and columns, two row tiles
    (70, 17, 32, 1160, "float16", [70, 1, 1160], ["p"]),            # a mask per batch; units beyond N in the last wavefront
    (300, 4, 128, 512, "bfloat16", None, ["p", "sum_flat"]),        # the fewest rows
    (9, 150, 64, 2048, "float16", [1, 150, 2048], ["p"]),          # a mask shared by the batches; sixteen wavefronts a row
    (380, 77, 64, 16, "bfloat16", [380, 77, 16], ["p"]),            # half a unit of columns, four row groups
    (0, 2048, 64, 256, "float16", [1, 256], ["p32", "max", "sum"]),  # no batch; float32 results and values per row
    (33, 200, 96, 72, "bfloat16", [33, 200, 1], ["p", "max"]),      # a value per row; three slabs of K
])
def test_scores_and_their_row_reductions(batch, m, k, n, dtype, mask, outputs):
    """Against float64. Relative error of a probability: the scores' absolute error (float32 sum of k products of 16-bit
    N(0,1) values: k * 2^-24 * |q||k| <= 2e-5 here) twice, the exponential's (2^-22), the row sum's (n / 32 + 32 additions
    of positive terms: 2^-17): below 1e-4 together, and half a unit of the result's type."""
    import torch
    text = _scores(batch, m, k, n, dtype, mask, outputs)
    kernel = driver.HipKernel(text, out_dir=None)
    assert kernel.family == "gemm_rows"
    print("case", batch, m, k, n, dtype, kernel.grid, kernel.block, flush=True)
    g = torch.Generator(device="cuda").manual_seed(k + n)
    td = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    q = torch.randn([max(batch, 1), m, k], generator=g, device="cuda").to(td)
    kk = torch.randn([max(batch, 1), n, k], generator=g, device="cuda").to(td)
    x = torch.randn(mask, generator=g, device="cuda") * 2 if mask else torch.zeros(1, device="cuda")
    if mask and n in mask:
        x = torch.where(torch.rand(mask, generator=g, device="cuda") < 0.3, torch.full_like(x, -10000.0), x)
    outs = [torch.full([d.nbytes], 255, dtype=torch.uint8, device="cuda") for d in kernel.outputs]
    s = torch.matmul(q.double(), kk.double().transpose(1, 2).contiguous()) * float(np.float32(k ** -0.5)) + x.double()
    top = s.amax(2, keepdim=True)
    e = torch.exp(s - top)
    exact = {"p": torch.softmax(s, 2), "p32": torch.softmax(s, 2), "max": top, "sum": e.sum(2, keepdim=True), "sum_flat": e.sum(2, keepdim=True)}
    unit = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11}[dtype]   # half of the last of 8 (11) significant bits
    for launch in range(2):
        kernel.launch([q, kk] + ([x] if mask else []) + outs)
        torch.cuda.synchronize()
        for name, d, o in zip(outputs, kernel.outputs, outs):
            got = o.view({"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}[d.dtype]).double()
            want = exact[name].reshape(-1)
            rel = 1e-4 + (unit if name == "p" else 0.0)
            floor = 2.0 ** -25 if d.dtype == "float16" else 2.0 ** -126   # half a subnormal unit; results that underflow
            bad = (got - want).abs() > rel * want.abs() + (1e-4 if name == "max" else floor)
            assert not bool(bad.any()), "%s: %d of %d, first %d" % (name, int(bad.sum()), bad.numel(), int(bad.nonzero()[0]))


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,k,n,dtype,mask,outputs", [
    (1, 1, 64, 16, "bfloat16", None, ["p"]), (6, 3, 128, 88, "float16", [6, 3, 88], ["p"]),      # one row, three
    (3, 127, 256, 64, "bfloat16", [1, 127, 64], ["p", "max"]), (0, 17, 32, 1024, "float16", [1, 1024], ["p32", "sum"]),   # the most of B
    (3, 320, 64, 320, "float16", [3, 320, 320], ["p"]), (5, 161, 96, 168, "bfloat16", None, ["p"]),   # from 128 rows on: more than 512 KiB of scores
    (33, 56, 64, 56, "bfloat16", [33, 1, 56], ["p", "sum_flat"]),
])
def test_one_launch_for_few_rows_and_scores(batch, m, k, n, dtype, mask, outputs):
    """Up to 64 KiB of B a batch; bounds as above."""
    test_scores_and_their_row_reductions(batch, m, k, n, dtype, mask, outputs)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,k,n,dtype,mask,outputs", [
    (40, 401, 64, 520, "bfloat16", [40, 401, 520], ["p"]),                  # eight wavefronts, two row tiles: a row and eight columns over
    (64, 249, 96, 1000, "float16", [1, 249, 1000], ["p"]),                  # a slab of K without a second one
    (40, 25, 128, 544, "bfloat16", [40, 25, 544], ["p", "max"]),              # one row tile
    (3, 1985, 64, 1032, "float16", [3, 1985, 1032], ["p"]), (5, 1601, 64, 1960, "bfloat16", [1, 1, 1960], ["p"]),   # sixteen wavefronts
])
def test_whole_lines_and_two_row_tiles(batch, m, k, n, dtype, mask, outputs):
    """32-bit tensors and B by whole lines of eight rows, rows and columns beyond the last; bounds as above."""
    test_scores_and_their_row_reductions(batch, m, k, n, dtype, mask, outputs)


def _scratch_bytes(directory):
    """Private bytes per lane of the code objects under `directory` (the kernel descriptor's note, a MessagePack map)."""
    import glob
    import os
    sizes = []
    for path in glob.glob(os.path.join(str(directory), "**", "*.hsaco"), recursive=True):
        data = open(path, "rb").read()
        key = b".private_segment_fixed_size"
        at = data.index(key) + len(key)
        width = {0xcc: 1, 0xcd: 2, 0xce: 4}.get(data[at], 0)
        sizes.append(int.from_bytes(data[at + 1:at + 1 + width], "big") if width else data[at])
    return sizes


@pytest.mark.parametrize("batch,m,k,n,family", [
    (0, 16384, 224, 320, "gemm_rows"), (0, 16384, 256, 320, "staged"),      # one batch of many rows
    (0, 8192, 384, 320, "gemm_rows"), (0, 8192, 416, 312, "staged"),        # ... of fewer
    (0, 32768, 512, 64, "gemm_rows"), (0, 32768, 544, 64, "staged"), (0, 33024, 256, 64, "staged"),   # few columns
    (0, 65536, 4096, 24, "gemm_rows"), (0, 65536, 4128, 24, "staged"), (0, 65536, 7168, 16, "staged"),
    (0, 16384, 2048, 64, "staged"), (0, 16384, 1024, 128, "staged"),        # routers whose rows the registers did not hold
    (64, 512, 512, 256, "gemm_rows"), (64, 512, 1024, 128, "staged"), (64, 46, 512, 224, "staged"), (64, 46, 384, 224, "gemm_rows"),
    (20, 1378, 256, 176, "staged"), (107, 2032, 384, 56, "gemm_rows"),
])
def test_a_long_k_takes_the_row_kernel_where_it_is_the_faster_one_and_needs_no_scratch(batch, m, k, n, family, tmp_path):
    kernel = driver.HipKernel(_scores(batch, m, k, n, "bfloat16", None, ["p"]), out_dir=str(tmp_path))
    assert kernel.family == family
    if family == "gemm_rows":
        sizes = _scratch_bytes(tmp_path)
        assert sizes and not any(sizes), sizes


def test_wide_descriptions_run_as_two_kernels():
    def family(n, masks, outputs, batch=64):
        b = op_desc.DescBuilder("wide_%d_%d_%s" % (n, masks, outputs.replace("+", "_")))
        q, kk = b.input([batch, 512, 64], "bfloat16"), b.input([batch, n, 64], "bfloat16")
        attrs = [{"data_type": "bool", "name": "transpose_a", "value": False}, {"data_type": "bool", "name": "transpose_b", "value": True}]
        raw = b.op("BatchMatMul", [q, kk], [batch, 512, n], "float32", attrs=attrs)
        s = raw
        for _ in range(masks):
            s = b.add(s, b.input([batch, 512, n], "float32"))
        e = b.unary("Exp", b.sub(s, b.reduce("ReduceMax", s, [2], True)))
        p = b.div(e, b.reduce("ReduceSum", e, [2], True))
        made = {"raw": lambda: raw, "masked": lambda: s, "p": lambda: p, "half": lambda: b.cast(p, "bfloat16")}
        return driver.HipKernel(b.dumps([made[o]() for o in outputs.split("+")]), out_dir=None).family
    assert family(2048, 3, "half", 32) == "gemm_rows" and family(2048, 4, "half", 32) == "staged"     # two row tiles: 4 and 5 beside the scores
    assert family(2048, 4, "half", 16) == "gemm_rows" and family(2048, 5, "half", 16) == "staged"     # one: 5 and 6
    assert family(2048, 2, "p", 32) == "gemm_rows" and family(2048, 1, "masked+p", 32) == "staged"
    assert family(1024, 5, "half", 32) == "gemm_rows" and family(1024, 6, "half", 32) == "staged"
    assert family(512, 8, "half") == "gemm_rows"
    # scores that are written anyway
    assert family(264, 1, "raw+half") == "staged" and family(256, 1, "raw+half") == "gemm_rows"


def test_what_two_kernels_refuse_is_refused(monkeypatch):
    """An output that is listed twice, more batches than the contraction kernel takes: refused whichever kernel is asked first."""
    text = _scores(64, 256, 64, 256, "bfloat16", None, ["p32", "p32"])
    b = op_desc.DescBuilder("scores_twice")
    q, kk = b.input([64, 256, 64], "bfloat16"), b.input([64, 256, 64], "bfloat16")
    attrs = [{"data_type": "bool", "name": "transpose_a", "value": False}, {"data_type": "bool", "name": "transpose_b", "value": True}]
    s = b.op("BatchMatMul", [q, kk], [64, 256, 256], "float32", attrs=attrs)
    p = b.sub(s, b.reduce("ReduceMax", s, [2], True))
    assert driver.HipKernel(text, out_dir=None).family == "gemm_rows"    # (two results that happen to be equal)
    for variant in ("0", "16"):
        monkeypatch.setenv("AKG_HIP_VARIANT", variant)
        with pytest.raises(driver.AkgHipError):
            driver.HipKernel(b.dumps([p, p]), out_dir=None)
        assert driver.HipKernel(_scores(65535, 8, 32, 8, "bfloat16", None, ["p"]), out_dir=None).family == ("gemm_rows" if variant == "0" else "staged")
        with pytest.raises(driver.AkgHipError):
            driver.HipKernel(_scores(65536, 8, 32, 8, "bfloat16", None, ["p"]), out_dir=None)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,k,n,dtype", [
    (64, 70, 160, 72, "bfloat16"),      # five slabs of K held whole
    (40, 130, 224, 104, "float16"),     # seven
    (40, 130, 256, 200, "bfloat16"),    # two blocks
    (33, 65, 288, 136, "bfloat16"),     # a block of one slab behind two
    (0, 6100, 352, 264, "float16"),     # ... of three; three units of columns, one beyond N in part
    (64, 70, 512, 248, "bfloat16"),
    (0, 20000, 1056, 24, "bfloat16"),   # 33 slabs; fewer columns than a unit
    (0, 33000, 4096, 8, "float16"),
])
def test_blocks_of_a_long_k(batch, m, k, n, dtype):
    """Against float64. A score's float32 sum of k products is off by at most k * 2^-24 of the sum of the products'
    magnitudes, a probability by twice the largest such error of its row (relative), beside 2^-14 for the exponential and
    the row sum and half a unit of the result's type."""
    import torch
    kernel = driver.HipKernel(_scores(batch, m, k, n, dtype, None, ["p", "max"]), out_dir=None)
    assert kernel.family == "gemm_rows"
    print("case", batch, m, k, n, dtype, kernel.grid, kernel.block, flush=True)
    g = torch.Generator(device="cuda").manual_seed(k + n)
    td = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    q = torch.randn([max(batch, 1), m, k], generator=g, device="cuda").to(td)
    kk = torch.randn([max(batch, 1), n, k], generator=g, device="cuda").to(td)
    outs = [torch.full([d.nbytes], 255, dtype=torch.uint8, device="cuda") for d in kernel.outputs]
    scale = float(np.float32(k ** -0.5))
    s = torch.matmul(q.double(), kk.double().transpose(1, 2).contiguous()) * scale
    off = torch.matmul(q.double().abs(), kk.double().abs().transpose(1, 2).contiguous()).amax(2, keepdim=True) * (scale * k * 2.0 ** -24)
    for launch in range(2):
        kernel.launch([q, kk] + outs)
        torch.cuda.synchronize()
        p, top = outs[0].view(td).double().reshape(s.shape), outs[1].view(torch.float32).double().reshape(off.shape)
        want = torch.softmax(s, 2)
        unit = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
        bad = (p - want).abs() > (2 * off + 2.0 ** -14 + unit) * want + 2.0 ** -25
        assert not bool(bad.any()), "%d of %d, first %s" % (int(bad.sum()), bad.numel(), bad.nonzero()[0].tolist())
        assert bool(((top - s.amax(2, keepdim=True)).abs() <= off + top.abs() * 2.0 ** -23).all())


def _typed(mask_type, n, batch=48, m=250):
    """Scores with a mask of `mask_type` and results of several types, among them whole numbers and truth values."""
    b = op_desc.DescBuilder("typed_%s_%d" % (mask_type, n))
    q, kk = b.input([batch, m, 64], "bfloat16"), b.input([batch, n, 64], "bfloat16")
    x = b.input([batch, m, n], mask_type)
    attrs = [{"data_type": "bool", "name": "transpose_a", "value": False}, {"data_type": "bool", "name": "transpose_b", "value": True}]
    s = b.mul(b.op("BatchMatMul", [q, kk], [batch, m, n], "float32", attrs=attrs), b.const(0.125, "float32"))
    if mask_type == "bool":
        s = b.op("Select", [x, s, b.const(-10000.0, "float32")], [batch, m, n], "float32")
    else:
        s = b.add(s, x if mask_type == "float32" else b.cast(x, "float32"))
    top = b.reduce("ReduceMax", s, [2], True)
    e = b.unary("Exp", b.sub(s, top))
    p = b.div(e, b.reduce("ReduceSum", e, [2], True))
    if mask_type == "float32":
        return b.dumps([b.cast(p, "float16"), top])
    if mask_type == "bool":
        return b.dumps([b.op("Greater", [p, b.const(0.01, "float32")], [batch, m, n], "bool")])
    if mask_type == "int8":
        return b.dumps([b.cast(b.mul(p, b.const(127.0, "float32")), "int8"), b.reduce("ReduceMax", b.cast(s, "int32"), [2], True)])
    if mask_type == "int64":
        return b.dumps([b.cast(p, "bfloat16"), b.reduce("ReduceMin", s, [2], False)])
    return b.dumps([b.cast(p, "float64")])


@pytest.mark.parametrize("mask_type", ["float32", "bool", "int8", "int64", "float64"])
def test_types_that_take_the_row_kernel(mask_type):
    assert driver.HipKernel(_typed(mask_type, 200), out_dir=None).family == "gemm_rows"


@pytest.mark.gpu
@pytest.mark.parametrize("n", [200, 1032])
@pytest.mark.parametrize("mask_type", ["float32", "bool", "int8", "int64", "float64"])
def test_types_masks_and_values_at_the_ends_against_two_kernels(mask_type, n, monkeypatch):
    """The one-kernel form against a contraction and a row kernel, which work on the same float32 scores. Scores that are
    masked throughout, by a large number, the lowest one or -inf, and NaN and infinity in an operand: where the two forms
    have NaN or infinity has to be the same. Finite results: a score differs by the order of 64 products of bfloat16 (2 * 64 * 2^-24
    of the sum of their magnitudes, below 2^-10 here: |q k| < 300), a probability by twice that, 2^-13 for the exponential
    and the row sums, and a unit of its type; a whole number by one and a truth value only next to the line."""
    import torch
    text = _typed(mask_type, n)
    one = driver.HipKernel(text, out_dir=None)
    monkeypatch.setenv("AKG_HIP_VARIANT", "16")
    two = driver.HipKernel(text, out_dir=None)
    assert one.family == "gemm_rows" and two.family == "staged"
    print("case", mask_type, n, one.grid, one.block, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn([48, 250, 64], generator=g, device="cuda").bfloat16()
    kk = torch.randn([48, n, 64], generator=g, device="cuda").bfloat16()
    x = torch.randn([48, 250, n], generator=g, device="cuda")
    if mask_type == "bool":
        x = x > -0.5
        x[0, 0] = False
        x[5, 249, n - 1] = False
    elif mask_type in ("int8", "int64"):
        x = (x * 3).to(getattr(torch, mask_type))
        x[0, 0] = -128
    else:
        low = float(np.finfo(np.float32).min)
        x = torch.where(torch.rand(x.shape, generator=g, device="cuda") < 0.3, torch.full_like(x, -10000.0), x).to(getattr(torch, mask_type))
        x[0, 0], x[0, 1], x[0, 2, : n // 2], x[47, 249, 1:] = float("-inf"), low, float("-inf"), low
        x[1, 7, n - 1] = float("nan")
    q[2, 3, 5] = float("nan")
    kk[3, n - 1, 0] = float("nan")
    q[4, 249, 63] = float("inf")
    results = []
    for kernel in (one, two):
        outs = [torch.full([d.nbytes], 255, dtype=torch.uint8, device="cuda") for d in kernel.outputs]
        kernel.launch([q, kk, x] + outs)
        torch.cuda.synchronize()
        results.append([o.view(getattr(torch, d.dtype)).double() for o, d in zip(outs, kernel.outputs)])
    unit = {"bfloat16": 2.0 ** -7, "float16": 2.0 ** -10, "float32": 2.0 ** -22, "float64": 2.0 ** -22}
    for d, a, b in zip(one.outputs, *results):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), d.dtype
        finite = a.isfinite()
        a, b = a[finite], b[finite]
        if d.dtype == "bool":
            assert int((a != b).sum()) <= a.numel() // 1000       # (|p - 0.01| < 0.01 * 2^-8 for fewer than one in a thousand)
        elif d.dtype in ("int8", "int32"):
            assert bool(((a - b).abs() <= 1).all()) and int((a != b).sum()) <= a.numel() // 100
        else:
            bound = b.abs() * (2.0 ** -9 + 2.0 ** -13 + unit[d.dtype]) + (2.0 ** -9 if a.numel() <= 48 * 250 else 2.0 ** -24)
            assert bool(((a - b).abs() <= bound).all()), (d.dtype, float(((a - b).abs() / bound).max()))


@pytest.mark.parametrize("batch,m,k,n,lines", [
    (60, 640, 64, 640, True), (108, 568, 32, 568, True), (115, 864, 128, 864, True),             # us by half lines / by whole ones: 48.5 / 44.9, 39.5 / 38.4, 223 / 218
    (63, 712, 128, 712, False), (78, 648, 192, 648, False), (109, 142, 96, 712, False),          # 59.1 / 61.3, 103 / 107, 21.1 / 21.8
    (192, 512, 64, 512, False),
])
def test_masks_by_whole_lines_with_a_short_k(batch, m, k, n, lines):
    kernel = driver.HipKernel(op_desc.attention_probabilities(batch, m, k, n, "bfloat16", "lines_%d_%d_%d_%d" % (batch, m, k, n)), out_dir=None)
    assert kernel.family == "gemm_rows" and ("akg::load_own_row_if<" in kernel.source) == lines
