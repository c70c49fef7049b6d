"""GPU tests of the split-contraction GEMM (csrc/gemm_split.h), the fully
connected layer's fused bias and the column sums, at the sizes where their
tiles, k-steps, splits and row blocks begin and end, against float64.

Bars (normwise max|x - ref| / max|ref|): fp32 1e-5 as for the GEMM (fp32
products and sums); bf16 results 8e-3 (one rounding to bf16, 2^-9 of a value
that may be the largest, plus fp32 sums)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-5, "bf16": 8e-3}
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


def _vals(rng, shape, dt):
    x = rng.standard_normal(shape).astype(np.float32)
    return orc.bf16_round(x) if dt == "bf16" else x


# tile edges (32 x 128 up to 32 rows, 64 x 64 above), k-step edges (32 fp32, 64 bf16), one, few and many splits
SHAPES = [(32, 128, 64), (33, 129, 65), (31, 127, 31), (64, 64, 129), (65, 63, 127), (1, 200, 513), (200, 1, 4097),
          (63, 65, 16391), (320, 192, 191), (1000, 700, 300)]


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=[str(s) for s in SHAPES])
def test_split_gemm(capi, dt, ta, tb, off, shape):
    """off: every matrix starts one element into its buffer (no 16-byte alignment)."""
    m, n, k = shape
    rng = np.random.default_rng(m + 3 * n + 5 * k + 7 * ta + 11 * tb)
    A, B, C = _vals(rng, (k, m) if ta else (m, k), dt), _vals(rng, (n, k) if tb else (k, n), dt), _vals(rng, (m, n), dt)
    bufs = [capi.DeviceBuffer.from_numpy(np.concatenate([np.zeros(off, np.float32), x.ravel()]), dt)
            for x in (A, B, C)]
    at = off * (2 if dt == "bf16" else 4)
    capi.lib().call("tt_gemm_" + dt, ta, tb, m, n, k, 0.5, bufs[0].ptr + at, bufs[1].ptr + at, 1.5, bufs[2].ptr + at,
                    None)
    out = bufs[2].download()
    assert not np.any(out[:off])
    ref = orc.gemm_f64(bool(ta), bool(tb), 0.5, A, B, 1.5, C)
    assert orc.max_rel_err(out[off:].reshape(m, n), ref) <= TOL[dt]


# bf16 operands with C in fp32: the split, the direct-to-LDS and the other 128-row kernel
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("shape", [(33, 129, 65), (64, 200, 4097), (2048, 4096, 64), (2100, 4100, 50)], ids=str)
def test_gemm_fp32_result(capi, ta, tb, shape):
    """No rounding of C: the products of bf16 values are exact in fp32, the sums fp32."""
    m, n, k = shape
    rng = np.random.default_rng(m + n + k + ta + 2 * tb)
    A, B = _vals(rng, (k, m) if ta else (m, k), "bf16"), _vals(rng, (n, k) if tb else (k, n), "bf16")
    C = _vals(rng, (m, n), "f32")
    a, b, c = (capi.DeviceBuffer.from_numpy(x, dt) for x, dt in ((A, "bf16"), (B, "bf16"), (C, "f32")))
    capi.lib().call("tt_gemm_bf16_f32", ta, tb, m, n, k, 0.5, a.ptr, b.ptr, 1.5, c.ptr, None)
    assert orc.max_rel_err(c.download(), orc.gemm_f64(bool(ta), bool(tb), 0.5, A, B, 1.5, C)) <= TOL["f32"]


@pytest.mark.parametrize("n", [1, 255, 70000])
def test_round_bf16(capi, n):
    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    x[:4] = np.array([np.nan, np.inf, -np.inf, 3.3895e38], np.float32)[:n]  # the last one rounds to infinity
    src, dst = capi.DeviceBuffer.from_numpy(x), capi.DeviceBuffer((n,), "bf16")
    capi.lib().call("tt_round_bf16", src.ptr, dst.ptr, n, None)
    bits = dst.download_bytes()
    assert np.isnan(orc.bf16_to_f32(bits[:1]))[0]
    np.testing.assert_array_equal(bits[1:], capi.bf16_bits(x)[1:])


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("scalar", [0, 1])
@pytest.mark.parametrize("shape", [(5, 9, 3), (64, 200, 100), (2048, 512, 4096)], ids=str)
def test_fc_forward_bias(capi, dt, scalar, shape):
    """Split, unsplit and (the last shape, bf16) direct-to-LDS kernels."""
    b, fin, fout = shape
    rng = np.random.default_rng(b + fin + fout + scalar)
    x, w, bias = _vals(rng, (b, fin), dt), _vals(rng, (fin, fout), dt), _vals(rng, (1 if scalar else fout,), dt)
    dx, dw, db = (capi.DeviceBuffer.from_numpy(a, dt) for a in (x, w, bias))
    out = capi.DeviceBuffer((b, fout), dt)
    code = capi.TT_BF16 if dt == "bf16" else capi.TT_F32
    capi.lib().call("tt_fc_forward", code, b, fin, fout, dx.ptr, dw.ptr, db.ptr, scalar, out.ptr, None)
    ref = x.astype(np.float64) @ w.astype(np.float64) + bias.astype(np.float64)
    assert orc.max_rel_err(out.download(), ref) <= TOL[dt]


# rows around the 16 waves, the 8-load step (128) and the row block (2048); columns around the 64 lanes
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("rows", [0, 1, 15, 17, 127, 129, 2048, 2049, 9000])
@pytest.mark.parametrize("cols", [1, 63, 65])
def test_col_sum(capi, dt, rows, cols):
    x = _vals(np.random.default_rng(rows + cols), (rows, cols), dt)
    dx = capi.DeviceBuffer.from_numpy(x, dt) if rows else capi.DeviceBuffer((1,), dt)
    y = capi.DeviceBuffer((cols,), dt)
    capi.lib().call("tt_col_sum", capi.TT_BF16 if dt == "bf16" else capi.TT_F32, dx.ptr, y.ptr, rows, cols, None)
    ref = x.astype(np.float64).sum(0)
    got = y.download()
    # |error| <= 2^-24 per addition over sums of absolute values, one bf16 rounding of the result
    bound = np.abs(x).astype(np.float64).sum(0) * 2.0 ** -20 + (np.abs(ref) * 2.0 ** -8 if dt == "bf16" else 0)
    assert np.all(np.abs(got - ref) <= bound)


def test_refused_scratch_runs_unsplit(capi):
    """With the scratch allocation (the one after the three matrices) refused the product still comes out."""
    code = (
        "import ctypes as C, numpy as np, tt_capi as T\n"
        "def in_use():\n"
        "    n = C.c_size_t(); T.lib().call('tt_mem_stats', C.byref(n), None); return n.value\n"
        "r = np.random.default_rng(1)\n"
        "A, B = (r.standard_normal(s).astype(np.float32) for s in ((48, 4096), (4096, 40)))\n"
        "a, b, c = T.DeviceBuffer.from_numpy(A), T.DeviceBuffer.from_numpy(B), T.DeviceBuffer((48, 40))\n"
        "before = in_use()\n"
        "T.gemm(False, False, 48, 40, 4096, 1.0, a, b, 0.0, c)\n"
        "assert in_use() == before, 'the scratch was not refused'\n"
        "ref = A.astype(np.float64) @ B.astype(np.float64)\n"
        "e = np.abs(c.download() - ref).max() / np.abs(ref).max()\n"
        "assert e <= 1e-5, e\n"
        "try:\n"
        "    T.DeviceBuffer((1 << 20,))\n"
        "except T.TTError as x:\n"
        "    print('REFUSED', x.code == T.TT_ERR_NOMEM)\n")
    env = dict(os.environ, TT_FAIL_ALLOC_AFTER="3",
               PYTHONPATH=os.path.join(ROOT, "pku-aiprogramming_amd") + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "REFUSED True" in r.stdout, r.stdout + r.stderr
