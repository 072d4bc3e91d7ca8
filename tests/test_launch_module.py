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


def test_without_the_module_launches_go_through_ctypes():
    """An interpreter that no module was built for imports the driver all the same, and what is refused is refused alike."""
    import os
    import subprocess
    import sys
    import sysconfig
    assert os.path.basename(driver._launch.__file__) == "_launch" + sysconfig.get_config_var("EXT_SUFFIX")   # (no other one loads it)
    code = """
import sys
class Absent:
    def find_spec(self, name, path=None, target=None):
        if name == "akg_amd._launch":
            raise ImportError("built for another interpreter")
sys.meta_path.insert(0, Absent())
import torch
from akg_amd import driver, op_desc
k = driver.HipKernel(op_desc.elementwise_tanh_add_mul(7, 33), out_dir=None)
assert driver._launch is None
try:
    k.launch([torch.zeros(7, 33) for _ in range(4)])
except ValueError as e:
    assert "contiguous device tensor" in str(e)
else:
    raise AssertionError("a host tensor was launched on")
b = op_desc.DescBuilder("launch_module_absent")
x = b.input([-1, 64], "float32")
d = driver.HipDynamicKernel(b.dumps([b.op("Tanh", [x], [-1, 64], "float32")]), out_dir=None)
try:
    d.launch_packed([1, 2], [[5, 64], [6, 64]])
except driver.AkgHipError as e:
    assert "does not follow from the input shapes" in str(e)
else:
    raise AssertionError("inconsistent shapes were launched")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    subprocess.run([sys.executable, "-c", code], check=True, cwd=root, env=dict(os.environ, PYTHONPATH=root))


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


@pytest.mark.gpu
def test_without_the_module_the_results_are_the_same(monkeypatch):
    k = driver.HipKernel(op_desc.elementwise_tanh_add_mul(37, 130), out_dir=None)
    d = driver.HipDynamicKernel(_dynamic())
    a, b, c = (torch.randn(37, 130, device="cuda") for _ in range(3))
    x = torch.randn(5, 64, device="cuda")
    results = []
    for module in (driver._launch, None):
        monkeypatch.setattr(driver, "_launch", module)
        out, y = torch.zeros(37, 130, device="cuda"), torch.zeros(5, 64, device="cuda")
        k.launch([a, b, c, out])
        d.launch_packed([x.data_ptr(), y.data_ptr()], [x.shape, y.shape], torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        results.append((out, y))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.gpu
def test_two_threads_launch_through_the_module():
    """One static and one dynamic handle, launched by two threads on streams of their own: each gets its own results and its
    own errors (a refused launch in one thread says nothing in the other)."""
    import threading
    k = driver.HipKernel(op_desc.elementwise_tanh_add_mul(37, 130), out_dir=None)
    k.prepare()
    d = driver.HipDynamicKernel(_dynamic())
    failures = []

    def work(seed):
        try:
            g = torch.Generator(device="cuda").manual_seed(seed)
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                a, b, c = (torch.randn(37, 130, generator=g, device="cuda") for _ in range(3))
                x = torch.randn(5 + seed, 64, generator=g, device="cuda")
                for step in range(50):
                    out, y = torch.zeros(37, 130, device="cuda"), torch.zeros(5 + seed, 64, device="cuda")
                    k.launch([a, b, c, out])
                    d.launch_packed([x.data_ptr(), y.data_ptr()], [x.shape, y.shape], stream.cuda_stream)
                    with pytest.raises(driver.AkgHipError, match="does not follow"):
                        d.launch_packed([x.data_ptr(), y.data_ptr()], [x.shape, (4 + seed, 64)], stream.cuda_stream)
                    stream.synchronize()
                    assert torch.allclose(out, torch.tanh((a + b) * c), rtol=1e-5, atol=1e-6), step
                    assert torch.allclose(y, torch.tanh(x), rtol=1e-5, atol=1e-6), step
        except BaseException as e:   # pylint: disable=broad-except
            failures.append((seed, e))

    threads = [threading.Thread(target=work, args=(seed,)) for seed in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
