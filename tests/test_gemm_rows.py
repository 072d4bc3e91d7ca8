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
