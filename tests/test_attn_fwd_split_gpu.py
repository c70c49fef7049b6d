"""GPU tests of the bf16 forward with its keys split over workgroups, or over
two groups of waves of one workgroup (few query tiles, many keys; csrc/attn_fwd.hip), where splits, tiles and diagonals
meet, against the float64 oracle at the bf16 bar (2e-2, normwise).  LSE: the
row sum adds the bf16-rounded weights that the P V product applies, each
within 2^-9 of its value, so it is within log(1 + 2^-9) < 2^-9 of the exact
one, split or not, plus fp32 rounding (1e-5)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    return tt_capi


def _run(capi, q, k, v, scale, causal):
    bufs = [capi.DeviceBuffer.from_numpy(a, "bf16") for a in (q, k, v)]
    o, lse = capi.DeviceBuffer(q.shape, "bf16"), capi.DeviceBuffer(q.shape[:3], "f32")
    capi.attn_fwd(*bufs, o, lse, scale, causal)
    return o.download(), lse.download()


def _inputs(B, H, Lq, Lk, d, seed):
    rng = np.random.default_rng(seed)
    return [orc.bf16_round(rng.standard_normal(s).astype(np.float32)) for s in
            ((B, H, Lq, d), (B, H, Lk, d), (B, H, Lk, d))]


# 16 key tiles is the shortest split (up to 32 query tiles), 32 beyond; unsplit just below
CASES = [(1, 1, 1, 961, 64, False), (1, 1, 5, 960, 32, False), (1, 3, 129, 1500, 128, False), (1, 2, 300, 2049, 64, False),
         (1, 1, 1025, 1025, 64, True), (1, 2, 1000, 1000, 128, True), (1, 1, 4097, 4097, 32, True),
         (1, 8, 1985, 1985, 32, True), (1, 9, 1000, 2047, 32, False),
         # two key groups without a split: an odd and an even count of key tiles, ragged ends, diagonals
         (1, 9, 769, 769, 128, True), (1, 9, 833, 833, 64, True), (2, 17, 896, 896, 32, True),
         (2, 20, 300, 1023, 128, False), (1, 33, 130, 768, 64, False)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_split_forward(capi, case):
    B, H, Lq, Lk, d, causal = case
    q, k, v = _inputs(B, H, Lq, Lk, d, Lq + Lk)
    o, lse = _run(capi, q, k, v, float(np.float32(d ** -0.5)), causal)
    ro, rl = orc.attn_fwd_f64(q, k, v, float(np.float32(d ** -0.5)), causal)
    assert orc.max_rel_err(o, ro) <= orc.TOL["bf16"]
    assert np.abs(lse - rl).max() <= 2.0 ** -9 + 1e-5


def test_split_forward_extreme_scores(capi):
    """Running maxima that differ by hundreds between splits, and a NaN query row."""
    q, k, v = _inputs(1, 2, 40, 2000, 64, 3)
    q *= 8
    k[:, :, 1500:] *= 8  # the last splits hold every row's weight
    q, k = orc.bf16_round(q), orc.bf16_round(k)
    o, _ = _run(capi, q, k, v, 0.125, False)
    assert orc.max_rel_err(o, orc.attn_fwd_f64(q, k, v, 0.125, False)[0]) <= orc.TOL["bf16"]
    q[0, 1, 7, 3] = np.nan
    o2, lse2 = _run(capi, q, k, v, 0.125, False)
    bad = np.zeros(o.shape[:3], bool)
    bad[0, 1, 7] = True
    assert np.isnan(o2[bad]).all() and np.isnan(lse2[bad]).all()
    np.testing.assert_array_equal(o2[~bad], o[~bad])


def test_refused_scratch_runs_unsplit(capi):
    code = (
        "import ctypes as C, numpy as np, tt_capi as T\n"
        "from oracle import attn_oracle as orc\n"
        "r = np.random.default_rng(1)\n"
        "q, k, v = (orc.bf16_round(r.standard_normal((1, 1, n, 64)).astype(np.float32)) for n in (9, 2000, 2000))\n"
        "b = [T.DeviceBuffer.from_numpy(a, 'bf16') for a in (q, k, v)]\n"
        "o, l = T.DeviceBuffer(q.shape, 'bf16'), T.DeviceBuffer(q.shape[:3], 'f32')\n"
        "def in_use():\n"
        "    n = C.c_size_t(); T.lib().call('tt_mem_stats', C.byref(n), None); return n.value\n"
        "before = in_use()\n"
        "T.attn_fwd(*b, o, l, 0.125, False)\n"
        "assert in_use() == before, 'the scratch was not refused'\n"
        "assert orc.max_rel_err(o.download(), orc.attn_fwd_f64(q, k, v, 0.125, False)[0]) <= 2e-2\n"
        "try:\n"
        "    T.DeviceBuffer((1 << 20,))\n"
        "except T.TTError as x:\n"
        "    print('REFUSED', x.code == T.TT_ERR_NOMEM)\n")
    env = dict(os.environ, TT_FAIL_ALLOC_AFTER="5", PYTHONPATH=os.pathsep.join(
        [ROOT, os.path.join(ROOT, "pku-aiprogramming_amd"), os.environ.get("PYTHONPATH", "")]))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "REFUSED True" in r.stdout, r.stdout + r.stderr
