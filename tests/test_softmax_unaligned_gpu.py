"""GPU tests of the row softmax on rows that are not 16-byte aligned
(csrc/softmax.hip): the split kernel beyond 12288 columns (lengths around its
chunks, partial last vectors, buffers that begin at any float, in place, chunks
without a finite value) and the rows of up to 16384 columns that are too few
to split, the one-workgroup kernel from 3329 to 12288 columns.  Against float64
at the softmax tests' bar (1e-5 normwise)."""
import numpy as np
import pytest

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


def _run(capi, x, xo, yo, in_place=False):
    rows, cols = x.shape
    bx = capi.DeviceBuffer.from_numpy(np.concatenate([np.zeros(xo, np.float32), x.ravel(), np.full(5, 7, np.float32)]))
    by = bx if in_place else capi.DeviceBuffer.from_numpy(np.full(yo + x.size + 5, 7, np.float32))
    yo = xo if in_place else yo
    capi.lib().call("tt_softmax_rows_f32", bx.ptr + 4 * xo, by.ptr + 4 * yo, rows, cols, None)
    out = by.download()
    assert np.all(out[yo + x.size:] == 7)  # nothing past the last row
    return out[yo:yo + x.size].reshape(x.shape)


@pytest.mark.parametrize("rows,cols", [(17, 8193), (16, 12287), (16, 12289), (20, 16383), (5, 16385), (3, 65535),
                                       (3, 65537), (2, 262143), (2, 262145), (1, 2097151), (16, 12288),
                                       # on both sides of the fewest unaligned rows that are split, and aligned ones
                                       (15, 12289), (15, 16383), (16, 12290), (3, 12292), (1, 16384)])
@pytest.mark.parametrize("xo,yo", [(0, 0), (1, 2), (3, 0)])
def test_unaligned_rows(capi, rows, cols, xo, yo):
    x = (3 * np.random.default_rng(cols).standard_normal((rows, cols))).astype(np.float32)
    ref = orc.softmax_rows_f64(x)
    assert orc.max_rel_err(_run(capi, x, xo, yo), ref) <= 1e-5
    assert orc.max_rel_err(_run(capi, x, xo, 0, in_place=True), ref) <= 1e-5


def test_chunks_without_finite_values(capi):
    x = np.random.default_rng(1).standard_normal((18, 12291)).astype(np.float32)
    x[2, :4096] = -np.inf       # the first chunk
    x[3, 12288:] = -np.inf      # the partial last chunk
    x[4, :] = -np.inf           # a whole row: NaN
    x[5, 9000] = np.nan
    y = _run(capi, x, 1, 1)
    bad = [4, 5]
    assert np.isnan(y[bad]).all()
    keep = np.delete(np.arange(18), bad)
    assert orc.max_rel_err(y[keep], orc.softmax_rows_f64(x[keep])) <= 1e-5
    assert np.all(y[2, :4096] == 0) and np.all(y[3, 12288:] == 0)


@pytest.mark.parametrize("cols", [65537, 100003, 262145])
def test_long_rows_round_each_element_alike(capi, cols):
    """Unaligned rows beyond 65536 columns: exp(x - M) / S from the row's maximum, so that equal elements
    give equal bits whatever the maximum of their chunk; rows and chunks without a finite value."""
    x = (3 * np.random.default_rng(cols).standard_normal((12, cols))).astype(np.float32)
    last = cols - 700
    x[:, last:last + 500] = x[:, 100:600]
    x[1, last + 600] = 25.0  # a chunk far above the others
    x[2, 20000:60000] = -np.inf
    x[3, :] = -np.inf
    x[4, 17] = np.nan
    x[5, -1] = np.inf
    y = _run(capi, x, 1, 2)
    assert np.isnan(y[[3, 4, 5]]).all()
    keep = np.delete(np.arange(12), [3, 4, 5])
    assert orc.max_rel_err(y[keep], orc.softmax_rows_f64(x[keep])) <= 1e-5
    np.testing.assert_array_equal(y[keep, last:last + 500], y[keep, 100:600])
    assert np.all(y[2, 20000:60000] == 0)


# one workgroup per row, vectors from 128-byte lines: around its range and the
# counts of vectors per lane (1024 k and 2048 k floats less the shift of up to 31)
@pytest.mark.parametrize("cols", [3328, 3329, 4064, 4065, 4096, 4097, 8160, 8161, 8162, 8192, 8193, 10209, 10240, 12257,
                                  12288])
@pytest.mark.parametrize("xo,yo", [(0, 0), (1, 2), (3, 31)])
def test_vector_rows(capi, cols, xo, yo):
    x = (3 * np.random.default_rng(cols).standard_normal((37, cols))).astype(np.float32)
    x[3, :] = -np.inf
    x[4, -1] = np.nan
    x[5, 0] = np.inf
    x[6, 1:] = -np.inf
    keep = np.delete(np.arange(37), [3, 4, 5])
    ref = orc.softmax_rows_f64(x[keep])
    for in_place in (False, True):
        y = _run(capi, x, xo, yo, in_place)
        assert np.isnan(y[[3, 4]]).all() and np.isnan(y[5, 0])
        assert orc.max_rel_err(y[keep], ref) <= 1e-5
