"""GPU tests of the decode's short splits and its merge (csrc/attn_decode.hip):
key counts around one split (8 rows per thread: 64 to 512 keys by head size
and type), many splits (more than one pass of the merge), partial last
splits, a split whose scores are all -inf, against the float64 oracle at the
usual bars."""
import numpy as np
import pytest

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


def _run(capi, dt, q, k, v):
    bufs = [capi.DeviceBuffer.from_numpy(a, dt) for a in (q, k, v)]
    o, lse = capi.DeviceBuffer(q.shape, dt), capi.DeviceBuffer(q.shape[:2], "f32")
    capi.attn_decode(*bufs, o, lse, 0.125)
    return o.download(), lse.download()


def _inputs(dt, B, H, L, d, seed):
    rng = np.random.default_rng(seed)
    x = [rng.standard_normal(s).astype(np.float32) for s in ((B, H, 1, d), (B, H, L, d), (B, H, L, d))]
    return [orc.bf16_round(a) for a in x] if dt == "bf16" else x


@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("chunks", [(0, 1), (0, 3), (1, -1), (1, 0), (1, 1), (2, 1), (70, 5)])
def test_short_splits(capi, dt, d, chunks):
    one = 8 * 256 // (d // (8 if dt == "bf16" else 4))  # keys of one split
    L = chunks[0] * one + chunks[1]
    q, k, v = _inputs(dt, 1, 3, L, d, L + d)
    o, lse = _run(capi, dt, q, k, v)
    ro, rl = orc.attn_decode_f64(q, k, v, 0.125)
    assert orc.max_rel_err(o, ro) <= orc.TOL[dt]
    assert orc.max_rel_err(lse.reshape(np.shape(rl)), rl) <= 1e-5  # fp32 weights and sums


def test_split_without_finite_scores(capi):
    q, k, v = _inputs("f32", 1, 2, 1000, 64, 1)
    q[..., 0] = 1.0
    k[:, :, 128:400, 0] = -np.inf  # whole splits of 128 keys among them
    o, lse = _run(capi, "f32", q, k, v)
    keep = np.r_[0:128, 400:1000]
    ro, rl = orc.attn_decode_f64(q, k[:, :, keep], v[:, :, keep], 0.125)
    assert orc.max_rel_err(o, ro) <= orc.TOL["f32"]
    assert orc.max_rel_err(lse.reshape(np.shape(rl)), rl) <= 1e-5
