"""Stream-ordered tensor memory (tt_malloc_ordered / tt_free_ordered) and the
small downloads: the allocator's lists on the CPU under sanitizers, and on
the GPU the hand-over of a freed tensor's storage to a caller stream and
downloads around the small path's limits, byte for byte."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_ordered_blocks_under_asan(tmp_path):
    exe = str(tmp_path / "ordered")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "pku-aiprogramming_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "ordered_checks.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "ordered checks passed" in r.stdout, r.stdout + r.stderr


@pytest.mark.gpu
def test_freed_tensor_storage_on_a_caller_stream():
    """A layer's result is dropped while its kernels run; a buffer of the same
    size filled on a caller stream right after keeps its values."""
    import myLayer as ml
    import myTensor as mt
    import tt_capi as T

    n = 2048
    rng = np.random.default_rng(0)
    a, b = (mt.Tensor_float(rng.standard_normal((n, n)).astype(np.float32), "gpu") for _ in range(2))
    bias = mt.Tensor_float([n], "gpu").zeros()
    stream = T.Stream()
    T.lib().sync()
    for _ in range(5):
        out = mt.Tensor_float([1], "gpu")
        for _ in range(8):
            ml.FcForward(a, out, b, bias)
        del out
        buf = T.DeviceBuffer((n, n), "f32")
        T.lib().call("tt_elementwise", 2, T.TT_F32, buf.ptr, None, None, n * n, 3.0, 0.0, 0, stream.handle)
        stream.sync()
        T.lib().sync()
        assert np.all(buf.download() == 3.0)
        buf.free()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 131071, 131072, 131073, 300000])
def test_small_downloads(n):
    import myTensor as mt
    import tt_capi as T

    rng = np.random.default_rng(n)
    for name, host in (("float", rng.standard_normal(n).astype(np.float32)), ("double", rng.standard_normal(n)),
                       ("int", rng.integers(-2**31, 2**31 - 1, n).astype(np.int32))):
        np.testing.assert_array_equal(getattr(mt, "Tensor_" + name)(host[None], "gpu").numpy(), host[None])
    bits = rng.integers(0, 1 << 16, n).astype(np.uint16)  # every kind of bf16, NaN among them
    buf = T.DeviceBuffer.from_numpy(bits, "bf16")
    np.testing.assert_array_equal(buf.download().view(np.uint32), bits.astype(np.uint32) << 16)
    np.testing.assert_array_equal(buf.download_bytes(), bits)
    if n > 2:  # a source that is not 16-byte aligned
        part = np.empty(n - 1, np.uint16)
        T.lib().call("tt_memcpy_d2h", part.ctypes.data, buf.ptr + 2, 2 * (n - 1))
        np.testing.assert_array_equal(part, bits[1:])
