"""GPU tests of the gathered convolution products (tt_conv_forward /
tt_conv_backward, csrc/conv.hip) where they can go wrong: channel counts
around the 32- and 64-row tiles, chunks that cross image rows and images,
strides with uneven phases, phases without taps, windows that do not overlap
or leave pixels uncovered, sums split over workgroups.  Reference: numpy
float64 on the same (for bf16: bf16-rounded) values.  Bars (normwise
max|x - ref| / max|ref|): fp32 1e-5 (fp32 products and sums), bf16 8e-3 (one
rounding of the result)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import attn_oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.gpu

TOL = {"float": 1e-5, "bf16": 8e-3}

# (N, Cin, H, W, Cout, kh, kw, pad_h, pad_w, stride_h, stride_w)
CASES = [
    (3, 1, 5, 5, 1, 1, 1, 0, 0, 1, 1),       # 1 x 1: windows do not overlap
    (2, 33, 6, 7, 31, 3, 3, 1, 1, 1, 1),     # rows past the 32-row tile, rows of 7 pixels
    (2, 65, 5, 3, 64, 3, 1, 1, 0, 1, 1),     # past the 64-row tile
    (5, 3, 11, 13, 6, 5, 5, 2, 2, 2, 2),     # uneven phases
    (2, 4, 10, 9, 5, 3, 2, 0, 1, 2, 1),      # stride in one axis
    (2, 3, 13, 13, 4, 3, 3, 1, 1, 4, 3),     # gaps between windows in one axis
    (2, 3, 16, 12, 5, 4, 3, 0, 0, 4, 3),     # windows tile the image
    (2, 3, 17, 14, 5, 4, 3, 1, 0, 4, 3),     # windows tile it with a pad and a remainder
    (1, 2, 4, 4, 3, 2, 2, 0, 0, 9, 9),       # stride past the image: one output pixel
    (1, 2, 6, 5, 3, 6, 5, 0, 0, 2, 2),       # kernel as large as the image
    (4, 2, 40, 40, 3, 3, 3, 1, 1, 1, 1),     # dW sums 6400 pixels over many splits
    (1, 200, 7, 7, 40, 3, 3, 1, 1, 1, 1),    # dX splits its contraction
    (1, 40, 14, 14, 200, 3, 3, 1, 1, 2, 2),  # and by phases
    # dX of few channels at stride 1: its channel counts, output channels around
    # its four groups, a ragged last workgroup, pads beyond the kernel, the
    # longest chains of a small and a large grid and one output channel more
    (3, 1, 9, 7, 8, 5, 5, 2, 2, 1, 1),
    (2, 2, 8, 8, 3, 3, 4, 1, 0, 1, 1),
    (1, 3, 5, 17, 5, 2, 7, 3, 8, 1, 1),
    (2, 4, 12, 11, 9, 3, 3, 0, 0, 1, 1),
    (1, 4, 6, 9, 24, 4, 4, 1, 2, 1, 1),
    (1, 4, 6, 9, 25, 4, 4, 1, 2, 1, 1),
    (12, 4, 64, 64, 40, 4, 4, 1, 2, 1, 1),
    (12, 4, 64, 64, 41, 4, 4, 1, 2, 1, 1),
    (12, 1, 64, 64, 128, 4, 4, 1, 2, 1, 1),
    (12, 1, 64, 64, 129, 4, 4, 1, 2, 1, 1),
    (2, 5, 6, 9, 6, 3, 3, 1, 1, 1, 1),
]


def _ref(x, w, go, ph, pw, sh, sw, blas=False):
    N, C, H, W = x.shape
    Co, _, kh, kw = w.shape
    oh, ow = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    xp = np.zeros((N, C, H + 2 * ph, W + 2 * pw))
    xp[:, :, ph:ph + H, pw:pw + W] = x
    out, gw, gxp = np.zeros((N, Co, oh, ow)), np.zeros(w.shape), np.zeros(xp.shape)
    for ky in range(kh):
        for kx in range(kw):
            at = (slice(None), slice(None), slice(ky, ky + sh * (oh - 1) + 1, sh), slice(kx, kx + sw * (ow - 1) + 1, sw))
            out += np.einsum("oc,ncyx->noyx", w[:, :, ky, kx], xp[at], optimize=blas)
            gw[:, :, ky, kx] = np.einsum("noyx,ncyx->oc", go, xp[at], optimize=blas)
            gxp[at] += np.einsum("oc,noyx->ncyx", w[:, :, ky, kx], go, optimize=blas)
    return out, gw, gxp[:, :, ph:ph + H, pw:pw + W]


@pytest.mark.parametrize("dt", ["float", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_conv_products(dt, case):
    import myLayer as ml
    import myTensor as mt

    T = getattr(mt, "Tensor_" + dt)
    N, C, H, W, Co, kh, kw, ph, pw, sh, sw = case
    rng = np.random.default_rng(sum(case))
    oh, ow = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    x, w, go = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (Co, C, kh, kw), (N, Co, oh, ow)))
    if dt == "bf16":
        x, w, go = orc.bf16_round(x), orc.bf16_round(w), orc.bf16_round(go)
    X, Wt, GO = (T(a, "gpu") for a in (x, w, go))
    out, gx, gw = (T([1], "gpu") for _ in range(3))
    ml.ConvForward(X, out, Wt, ph, pw, sh, sw)
    ml.ConvBackward(X, out, Wt, gx, GO, gw, ph, pw, sh, sw)
    ref = _ref(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), ph, pw, sh, sw)
    for name, got, r in zip(("out", "grad_weight", "grad_input"), (out, gw, gx), ref):
        a = np.asarray(got.numpy()).reshape(r.shape)
        if r.size == 0 or not np.any(r):
            assert not np.any(a)
            continue
        e = orc.max_rel_err(a, r)
        print(f"  {name} {e:.2e}", flush=True)
        assert e <= TOL[dt], (name, e)


@pytest.mark.parametrize("dt", ["float", "bf16"])
@pytest.mark.parametrize("case", [(2, 1, 9, 7, 8, 5, 5, 2, 2, 1, 1), (1, 4, 6, 9, 24, 4, 4, 1, 2, 1, 1),  # a lane per pixel
                                  (2, 6, 9, 7, 8, 5, 5, 2, 2, 1, 1), (2, 3, 11, 13, 6, 5, 5, 2, 2, 2, 2),  # products: one split,
                                  (1, 200, 7, 7, 40, 3, 3, 1, 1, 1, 1), (1, 40, 14, 14, 200, 3, 3, 1, 1, 2, 2),  # several
                                  (2, 3, 16, 12, 5, 4, 3, 1, 0, 4, 3)], ids=str)  # windows that do not overlap
def test_image_gradient_of_non_finite_weights(dt, case):
    """An infinite or NaN weight reaches the pixels its tap has an output pixel for, and no other."""
    import myLayer as ml
    import myTensor as mt

    T = getattr(mt, "Tensor_" + dt)
    N, C, H, W, Co, kh, kw, ph, pw, sh, sw = case
    rng = np.random.default_rng(sum(case))
    oh, ow = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    x, w, go = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (Co, C, kh, kw), (N, Co, oh, ow)))
    w[0, 0, 0, 0], w[1, C - 1, kh - 1, kw - 1], w[2, C - 1, 0, kw - 1] = np.inf, np.nan, -np.inf
    if dt == "bf16":
        x, w, go = orc.bf16_round(x), orc.bf16_round(w), orc.bf16_round(go)
    X, Wt, GO = (T(a, "gpu") for a in (x, w, go))
    out, gx, gw = (T([1], "gpu") for _ in range(3))
    ml.ConvBackward(X, out, Wt, gx, GO, gw, ph, pw, sh, sw)
    with np.errstate(invalid="ignore"):
        ref = _ref(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), ph, pw, sh, sw)[2]
    got = np.asarray(gx.numpy()).reshape(ref.shape)
    fin = np.isfinite(ref)
    assert fin.any() and not fin.all()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    np.testing.assert_array_equal(got[inf], ref[inf])
    assert np.abs(got[fin] - ref[fin]).max() <= TOL[dt] * np.abs(ref[fin]).max()


@pytest.mark.parametrize("case", [(1, 3, 1200, 1200, 1, 1200, 1200, 0, 0, 1200, 1200),  # C kh kw rows, windows apart
                                  (1, 1, 1, 1, 4194304, 1, 1, 0, 0, 1, 1),  # output channels
                                  (1, 4194304, 1, 1, 1, 2, 1, 1, 0, 1, 1)],  # input channels
                         ids=["kernel", "out_channels", "in_channels"])
def test_rows_beyond_the_grid(case):
    """More rows than 65535 tiles of 64: the layer takes the column matrix."""
    import myLayer as ml
    import myTensor as mt

    N, C, H, W, Co, kh, kw, ph, pw, sh, sw = case
    rng = np.random.default_rng(Co + kh)
    oh, ow = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    x, w, go = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (Co, C, kh, kw), (N, Co, oh, ow)))
    X, Wt, GO = (mt.Tensor_float(a, "gpu") for a in (x, w, go))
    out, gx, gw = (mt.Tensor_float([1], "gpu") for _ in range(3))
    ml.ConvForward(X, out, Wt, ph, pw, sh, sw)
    ml.ConvBackward(X, out, Wt, gx, GO, gw, ph, pw, sh, sw)
    if oh * ow == 1 and Co == 1:  # one window: the kernel's sums are single products
        refs = ((x * w).sum(dtype=np.float64), go.item() * x, go.item() * w)
    else:
        refs = _ref(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), ph, pw, sh, sw)
    for name, got, r in zip(("out", "grad_weight", "grad_input"), (out, gw, gx), refs):
        r = np.asarray(r, np.float64)
        e = orc.max_rel_err(np.asarray(got.numpy()).reshape(r.size), r.ravel())
        print(f"  {name} {e:.2e}", flush=True)
        assert e <= TOL["float"], (name, e)


# Channels wide enough for the column matrix: one image both ways, a batch in
# two parts backward, a stride, windows apart (bf16)
@pytest.mark.parametrize("dt", ["float", "bf16"])
@pytest.mark.parametrize("case", [(1, 320, 28, 28, 512, 3, 3, 1, 1, 1, 1), (4, 320, 40, 40, 512, 3, 3, 1, 1, 1, 1),
                                  (1, 257, 63, 64, 257, 3, 3, 1, 1, 2, 2), (1, 3, 1024, 1024, 768, 16, 16, 0, 0, 16, 16)],
                         ids=str)
def test_wide_products(dt, case):
    import myLayer as ml
    import myTensor as mt

    T = getattr(mt, "Tensor_" + dt)
    N, C, H, W, Co, kh, kw, ph, pw, sh, sw = case
    rng = np.random.default_rng(sum(case))
    oh, ow = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    x, w, go = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (Co, C, kh, kw), (N, Co, oh, ow)))
    if dt == "bf16":
        x, w, go = orc.bf16_round(x), orc.bf16_round(w), orc.bf16_round(go)
    X, Wt, GO = (T(a, "gpu") for a in (x, w, go))
    out, gx, gw = (T([1], "gpu") for _ in range(3))
    ml.ConvForward(X, out, Wt, ph, pw, sh, sw)
    ml.ConvBackward(X, out, Wt, gx, GO, gw, ph, pw, sh, sw)
    ref = _ref(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), ph, pw, sh, sw, blas=True)
    for name, got, r in zip(("out", "grad_weight", "grad_input"), (out, gw, gx), ref):
        a = np.asarray(got.numpy()).reshape(r.shape)
        e, two = orc.max_rel_err(a, r), np.linalg.norm(a - r) / np.linalg.norm(r)
        print(f"  {name} {e:.2e} 2-norm {two:.2e}", flush=True)
        assert e <= TOL[dt], (name, e)
        # bf16: one rounding of each result and none before it: 2^-8 / sqrt(3) x 0.74 = 1.66e-3 over significands
        # spread evenly in the logarithm (a rounding of the columns' gradients too would give 2.3e-3)
        assert two <= (1e-6 if dt == "float" else 2e-3), (name, two)


def test_wide_products_under_capture():
    """Captured on the library stream they are gathered: no memory that other tensors get before a replay."""
    import ctypes as C

    import myLayer as ml
    import myTensor as mt
    import tt_capi as T
    from test_capture_gpu import Capture

    rng = np.random.default_rng(3)
    shapes = ((1, 320, 28, 28), (512, 320, 3, 3), (1, 512, 28, 28))
    x, w, go = (rng.standard_normal(s).astype(np.float32) for s in shapes)
    X, Wt, GO = (mt.Tensor_float(a, "gpu") for a in (x, w, go))
    out, gx, gw = (mt.Tensor_float(list(s), "gpu") for s in (shapes[2], shapes[0], shapes[1]))

    def run():
        ml.ConvForward(X, out, Wt, 1, 1, 1, 1)
        ml.ConvBackward(X, out, Wt, gx, GO, gw, 1, 1, 1, 1)

    run()  # leaves the columns' block with the allocator
    stream = T.lib().lib.tt_stream()
    yes = C.c_int()
    with Capture(T, stream) as c:
        T.lib().call("tt_stream_capturing", None, C.byref(yes))
        run()
    assert yes.value == 1
    ref = _ref(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), 1, 1, 1, 1, blas=True)
    others = [mt.Tensor_float([n], "gpu").zeros() for n in (1 << 20, 2 << 20, 4 << 20, 8 << 20)]
    for _ in range(2):
        for t in (out, gx, gw):
            t.zeros()
        T.lib().sync()
        c.launch()
        for got, r in zip((out, gw, gx), ref):
            assert orc.max_rel_err(np.asarray(got.numpy()).reshape(r.shape), r) <= TOL["float"]
        assert not any(np.asarray(t.numpy()).any() for t in others)
    c.destroy()


def test_wide_products_without_scratch():
    """The gathered products take over where the columns' memory is refused."""
    code = (
        "import ctypes as C, numpy as np, myLayer as ml, myTensor as mt, tt_capi as T\n"
        "from test_conv_products_gpu import _ref\n"
        "from oracle import attn_oracle as orc\n"
        "r = np.random.default_rng(1)\n"
        "x, w, go = (r.standard_normal(s).astype(np.float32) for s in ((1, 320, 28, 28), (512, 320, 3, 3), (1, 512, 28, 28)))\n"
        "t = [mt.Tensor_float(a, 'gpu') for a in (x, w, go)]\n"
        "out, gx, gw = (mt.Tensor_float(list(s), 'gpu') for s in ((1, 512, 28, 28), x.shape, w.shape))\n"
        "def in_use():\n"
        "    a = C.c_size_t(); T.lib().call('tt_mem_stats', C.byref(a), None); return a.value\n"
        "before = in_use()\n"
        "ml.ConvForward(t[0], out, t[1], 1, 1, 1, 1)\n"
        "ml.ConvBackward(t[0], out, t[1], gx, t[2], gw, 1, 1, 1, 1)\n"
        "assert in_use() == before, 'scratch was not refused'\n"
        "ref = _ref(*(a.astype(np.float64) for a in (x, w, go)), 1, 1, 1, 1, blas=True)\n"
        "for a, b in zip((out, gw, gx), ref):\n"
        "    assert orc.max_rel_err(np.asarray(a.numpy()).reshape(b.shape), b) <= 1e-5\n"
        "try:\n"
        "    T.DeviceBuffer((1 << 20,))\n"
        "except T.TTError as e:\n"
        "    print('REFUSED', e.code == T.TT_ERR_NOMEM)\n")
    env = dict(os.environ, TT_FAIL_ALLOC_AFTER="6", PYTHONPATH=os.pathsep.join(
        [ROOT, os.path.join(ROOT, "tests"), os.path.join(ROOT, "pku-aiprogramming_amd"), os.environ.get("PYTHONPATH", "")]))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "REFUSED True" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("k,stride,cout", [(2, 1000, 3), (3, 2, 1)], ids=["windows_apart", "phases"])
def test_batches_beyond_one_launch(k, stride, cout):
    """Two images of more than 2^29 elements are taken one by one: the outputs and image gradients of each alone,
    bit for bit; the weight gradient their sum (bf16, three roundings of 2^-8)."""
    import tt_capi as T

    L, H = T.lib(), 23200
    oh = (H - k) // stride + 1
    x, go, w = (T.DeviceBuffer(s, "bf16") for s in ((2, 1, H, H), (2, cout, oh, oh), (cout, 1, k, k)))
    for i, b in enumerate((x, go, w)):
        b.fill_normal(i + 1)

    def run(n, first):
        out, gx, gw = (T.DeviceBuffer(s, "bf16") for s in ((n, cout, oh, oh), (n, 1, H, H), (cout, 1, k, k)))
        geo = (n, 1, H, H, cout, k, k, 0, 0, stride, stride, None)
        xp, gp = x.ptr + 2 * first * H * H, go.ptr + 2 * first * cout * oh * oh
        L.call("tt_conv_forward", T.TT_BF16, xp, w.ptr, out.ptr, *geo)
        L.call("tt_conv_backward", T.TT_BF16, xp, w.ptr, gp, gx.ptr, gw.ptr, *geo)
        return out.download_bytes(), gx.download_bytes(), gw.download()

    both, first, second = run(2, 0), run(1, 0), run(1, 1)
    for i, name in ((0, "out"), (1, "grad_input")):
        print(f"  {name}", flush=True)
        assert both[i].any()
        np.testing.assert_array_equal(both[i][0], first[i][0])
        np.testing.assert_array_equal(both[i][1], second[i][0])
    bound = 2.0 ** -8 * (np.abs(both[2]) + np.abs(first[2]) + np.abs(second[2]))
    # the sums themselves: fp32 over up to 1.3e8 products of either sign
    assert np.all(np.abs(both[2] - first[2] - second[2]) <= bound + 1e-4 * oh)
