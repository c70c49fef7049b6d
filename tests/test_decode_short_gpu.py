"""GPU tests of the decode's short splits and its merge (csrc/attn_decode.hip):
key counts around one split (8 rows per thread: 64 to 512 keys by head size
and type), many splits (more than one pass of the merge), partial last
splits, a split whose scores are all -inf, their scratch (refused, and under
capture), against the float64 oracle at the usual bars."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import attn_oracle as orc
from test_capture_gpu import Capture

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


def _run(capi, dt, q, k, v, scale=0.125):
    bufs = [capi.DeviceBuffer.from_numpy(a, dt) for a in (q, k, v)]
    o, lse = capi.DeviceBuffer(q.shape, dt), capi.DeviceBuffer(q.shape[:2], "f32")
    capi.attn_decode(*bufs, o, lse, scale)
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


@pytest.mark.parametrize("d,L", [(64, 128), (64, 200), (64, 256), (128, 64), (128, 128), (128, 200), (128, 256)])
def test_merged_splits_are_as_precise_as_one(capi, d, L):
    """fp32, one and several splits.  The 2-norm error of one split is that of its weights: 2^(s - m) to a few
    2^-24 each, 1.35e-7 to 1.6e-7 here.  Weights of the splits taken from an LSE each (a number of about 8,
    rounded to 2^-21) would add to it: 1.7e-7 to 1.95e-7 beyond one split."""
    q, k, v = _inputs("f32", 1, 240, L, d, L + d)
    scale = float(np.float32(d ** -0.5))
    o, _ = _run(capi, "f32", q, k, v, scale)
    s = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)) * scale
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)
    e = np.linalg.norm(o - ref) / np.linalg.norm(ref)
    print(f"  {e:.2e}", flush=True)
    assert e <= 1.65e-7


@pytest.mark.parametrize("BH,L,d", [(1299, 256, 32), (1300, 256, 32), (1300, 257, 32), (1300, 128, 64), (1300, 129, 64)])
def test_one_split_of_many_heads(capi, BH, L, d):
    """Both sides of the rule that leaves them to the long split's kernel."""
    q, k, v = _inputs("bf16", 1, BH, L, d, BH + L)
    o, lse = _run(capi, "bf16", q, k, v)
    ro, rl = orc.attn_decode_f64(q, k, v, 0.125)
    assert orc.max_rel_err(o, ro) <= orc.TOL["bf16"]
    assert orc.max_rel_err(lse.reshape(np.shape(rl)), rl) <= 1e-5


def test_split_without_finite_scores(capi):
    q, k, v = _inputs("f32", 1, 2, 1000, 64, 1)
    q[..., 0] = 1.0
    k[:, :, 128:400, 0] = -np.inf  # whole splits of 128 keys among them
    o, lse = _run(capi, "f32", q, k, v)
    keep = np.r_[0:128, 400:1000]
    ro, rl = orc.attn_decode_f64(q, k[:, :, keep], v[:, :, keep], 0.125)
    assert orc.max_rel_err(o, ro) <= orc.TOL["f32"]
    assert orc.max_rel_err(lse.reshape(np.shape(rl)), rl) <= 1e-5


REFUSED = r"""
import ctypes as C, numpy as np, tt_capi as T
from oracle import attn_oracle as orc
def in_use():
    a, b = C.c_size_t(), C.c_size_t()
    T.lib().call("tt_mem_stats", C.byref(a), C.byref(b))
    return a.value
def bufs(L):
    return [T.DeviceBuffer((1, 8, n, 128), "bf16") for n in (1, L, L, 1)]
r = np.random.default_rng(1)
WARM, L = %r
if WARM:  # allocations 0 .. 4: a call whose heads take long splits, and its partials
    q, k, v, o = bufs(WARM)
    k.fill_normal(1), v.fill_normal(2), q.fill_normal(3)
    T.attn_decode(q, k, v, o, None, 0.125)
b = bufs(L)  # the last allocations before the refusals
x = [orc.bf16_round(r.standard_normal(a.shape).astype(np.float32)) for a in b[:3]]
for d, a in zip(b, x):
    d.upload(a)
T.lib().sync()
before = in_use()
T.attn_decode(*b, None, 0.125)
assert in_use() == before, "the scratch was not refused"
assert orc.max_rel_err(b[3].download(), orc.attn_decode_f64(*x, 0.125)[0]) <= 2e-2
try:
    T.DeviceBuffer((1 << 20,))
except T.TTError as e:
    print("REFUSED", e.code == T.TT_ERR_NOMEM)
"""


@pytest.mark.parametrize("warm,L", [(0, 200), (32768, 8000)])
def test_refused_scratch(capi, warm, L):
    """Without scratch for the short splits: one long split, or the long splits' buffer that is there."""
    env = dict(os.environ, TT_FAIL_ALLOC_AFTER="9" if warm else "4", PYTHONPATH=os.pathsep.join(
        [ROOT, os.path.join(ROOT, "pku-aiprogramming_amd"), os.environ.get("PYTHONPATH", "")]))
    r = subprocess.run([sys.executable, "-c", REFUSED % ((warm, L),)], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "REFUSED True" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("L", [200, 3000])
def test_captured_decode_replays(capi, L):
    """Calls of other sizes on the stream, shorter and longer, leave the graph's scratch alone."""
    st = capi.Stream()

    def bufs(n):
        return [capi.DeviceBuffer(s, "f32") for s in ((1, 4, 1, 128), (1, 4, n, 128), (1, 4, n, 128), (1, 4, 1, 128))]

    b = bufs(L)
    for a in b[:3]:
        a.fill_normal(9)
    capi.lib().sync()
    capi.attn_decode(*b, None, 0.125, stream=st.handle)  # leaves the scratch on the stream
    st.sync()
    with Capture(capi, st.handle) as c:
        capi.attn_decode(*b, None, 0.125, stream=st.handle)
    others = [bufs(n) for n in (100, 700, 9000, 45000)]
    for i, other in enumerate(others):
        x = _inputs("f32", 1, 4, L, 128, i)
        for d, a in zip(b, x):
            d.upload(a)
        y = _inputs("f32", 1, 4, other[1].shape[2], 128, i + 10)
        for d, a in zip(other, y):
            d.upload(a)
        capi.attn_decode(*other, None, 0.125, stream=st.handle)
        c.launch()
        assert orc.max_rel_err(b[3].download(), orc.attn_decode_f64(*x, 0.125)[0]) <= orc.TOL["f32"]
        assert orc.max_rel_err(other[3].download(), orc.attn_decode_f64(*y, 0.125)[0]) <= orc.TOL["f32"]
    c.destroy()
