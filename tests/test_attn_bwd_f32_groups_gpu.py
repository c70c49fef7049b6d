"""GPU tests of the fp32 backward with two groups of waves per workgroup
(csrc/attn_bwd_f32.h, d <= 64): odd and even counts of tiles on either side of
the loop, ragged ends, diagonals, and the sizes on both sides of the rule that
chooses it, against the float64 oracle at the fp32 bar (1e-4, normwise: fp32
products and sums, in another order)."""
import numpy as np
import pytest

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


CASES = [(1, 2, 256, 256, 64, False), (1, 1, 255, 255, 64, True), (1, 3, 257, 257, 64, True), (1, 2, 289, 65, 64, False),
         (1, 2, 65, 321, 64, False), (1, 1, 64, 300, 64, False), (1, 1, 300, 64, 64, False), (2, 8, 353, 480, 64, False),
         (1, 8, 640, 640, 64, True), (1, 2, 512, 512, 32, False), (1, 2, 511, 511, 32, True), (1, 3, 577, 577, 32, True),
         (1, 1, 70, 961, 32, False), (1, 1, 1025, 66, 32, False), (3, 16, 513, 300, 32, False), (3, 12, 513, 513, 32, True)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_backward(capi, case):
    B, H, Lq, Lk, d, causal = case
    rng = np.random.default_rng(Lq + Lk)
    scale = float(np.float32(d ** -0.5))
    x = [rng.standard_normal((B, H, L, d)).astype(np.float32) for L in (Lq, Lk, Lk, Lq)]
    q, k, v, do = (capi.DeviceBuffer.from_numpy(a, "f32") for a in x)
    o, lse = capi.DeviceBuffer((B, H, Lq, d), "f32"), capi.DeviceBuffer((B, H, Lq), "f32")
    grads = [capi.DeviceBuffer((B, H, L, d), "f32") for L in (Lq, Lk, Lk)]
    capi.attn_fwd(q, k, v, o, lse, scale, causal)
    capi.attn_bwd(q, k, v, o, lse, do, *grads, scale, causal)
    for got, ref in zip(grads, orc.attn_bwd_f64(*x, scale, causal)):
        assert orc.max_rel_err(got.download(), ref) <= orc.TOL["f32"]
