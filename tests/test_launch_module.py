"""The native launch path: what it serves, and that everything else ends in the errors of the Python path."""
import pytest
import torch

from akg_amd import driver, op_desc


def _dynamic():
    b = op_desc.DescBuilder("launch_module_dynamic")
    x = b.input([-1, 64], "float32")
    return b.dumps([b.op("Tanh", [x], [-1, 64], "float32")])


def test_arguments_that_the_native_path_leaves_to_python():
    k = driver.HipKernel(op_desc.elementwise_tanh_add_mul(7, 33), out_dir=None)
    host = [torch.zeros(7, 33) for _ in range(4)]
    with pytest.raises(ValueError, match="contiguous device tensor"):
        k.launch(host)
    with pytest.raises(AttributeError):
        k.launch([None] * 4)
    n = driver._launch.launch
    assert n(k._handle.value, k._nbytes, host, None, int, int) is None            # not on a device
    assert n(k._handle.value, k._nbytes, host[:3], None, int, int) is None        # too few
    assert n(k._handle.value, list(k._nbytes), host, None, int, int) is None      # not a tuple
    assert n("x", k._nbytes, host, None, int, int) is None
    d = driver.HipDynamicKernel(_dynamic(), out_dir=None)
    p = driver._launch.launch_packed
    assert p(d._handle.value, [1, 2], [[5, 64]], 0) is None                       # a shape is missing
    assert p(d._handle.value, [1, "x"], [[5, 64], [5, 64]], 0) is None
    assert p(d._handle.value, [1, 2], [[5, 64.0], [5, 64]], 0) is None
    assert p(d._handle.value, [1, 2], [[5] * 9, [5, 64]], 0) is None
    with pytest.raises(driver.AkgHipError, match="does not follow from the input shapes"):
        d.launch_packed([1, 2], [[5, 64], [6, 64]])
    with pytest.raises(driver.AkgHipError, match="2 |outputs"):
        d.launch_packed([1], [[5, 64]])


@pytest.mark.gpu
def test_launches_on_the_current_and_on_a_given_stream():
    k = driver.HipKernel(op_desc.elementwise_tanh_add_mul(37, 130), out_dir=None)
    a, b, c = (torch.randn(37, 130, device="cuda") for _ in range(3))
    want = torch.tanh((a + b) * c)
    side = torch.cuda.Stream()
    for stream in (None, side):
        out = torch.zeros(37, 130, device="cuda")
        torch.cuda.synchronize()
        k.launch((a, b, c, out), stream)
        torch.cuda.synchronize()
        assert torch.allclose(out, want, rtol=1e-5, atol=1e-6)
    with torch.cuda.stream(side):
        out.zero_()
        k.launch([a, b, c, out])
    side.synchronize()
    assert torch.allclose(out, want, rtol=1e-5, atol=1e-6)
    with pytest.raises(ValueError, match="contiguous"):
        k.launch([a.t().contiguous().t(), b, c, out])
    with pytest.raises(ValueError, match="bytes"):
        k.launch([a[:36], b, c, out])
    with pytest.raises(ValueError, match="takes 4 tensors"):
        k.launch([a, b, c])
    d = driver.HipDynamicKernel(_dynamic())
    for rows in (3, 200):
        x, y = torch.randn(rows, 64, device="cuda"), torch.zeros(rows, 64, device="cuda")
        used = d.launch_packed([x.data_ptr(), y.data_ptr()], [x.shape, list(y.shape)], torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.allclose(y, torch.tanh(x), rtol=1e-5, atol=1e-6) and used is d.launch_packed([x.data_ptr(), y.data_ptr()], [x.shape, y.shape])
