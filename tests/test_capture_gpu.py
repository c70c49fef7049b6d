"""GPU tests of the calls that take scratch only where they can (products,
column sums, convolutions, the bf16 forward, long softmax rows): with the
scratch refused, captured into a graph and replayed on new inputs with eager
work in between, and on one stream while another is being captured (they may
neither end that capture nor join it); and of tt_malloc then.  Each result
against float64 at the bars of the eager tests: 1e-5 normwise where sums and
products are fp32, 2e-2 for bf16 attention."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import attn_oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.gpu

GLOBAL, THREAD_LOCAL = 0, 1  # hipStreamCaptureMode


@pytest.fixture(scope="module")
def capi():
    import tt_capi

    assert tt_capi.lib().device_count() >= 1, "no HIP device visible"
    tt_capi.lib().call("tt_init", 0)
    return tt_capi


class Op:
    """One call: fill(seed) uploads new inputs, run(stream) queues it, check() compares."""

    def __init__(self, capi, name):
        self.T, self.call, self.kind = capi, capi.lib().call, name
        f, h = "f32", "bf16"
        shapes = {  # inputs, outputs
            "gemm": ([((256, 784), f), ((784, 100), f)], [((256, 100), f)]),
            "col_sum": ([((5000, 70), f)], [((70,), f)]),
            "softmax": ([((40, 12291), f)], [((40, 12291), f)]),
            "softmax_aligned": ([((6, 16384), f)], [((6, 16384), f)]),
            "conv": ([((4, 8, 14, 14), f), ((16, 8, 5, 5), f), ((4, 16, 14, 14), f)],
                     [((4, 16, 14, 14), f), ((4, 8, 14, 14), f), ((16, 8, 5, 5), f)]),
            "fwd_bf16": ([((1, 2, 40, 64), h), ((1, 2, 2000, 64), h), ((1, 2, 2000, 64), h)],
                         [((1, 2, 40, 64), h), ((1, 2, 40), f)]),
        }[name]
        self.dts = [dt for _, dt in shapes[0]]
        self.shapes = [s for s, _ in shapes[0]]
        self.inp = [capi.DeviceBuffer(s, dt) for s, dt in shapes[0]]
        self.out = [capi.DeviceBuffer(s, dt) for s, dt in shapes[1]]

    def fill(self, seed):
        rng = np.random.default_rng(seed)
        self.x = [rng.standard_normal(s).astype(np.float32) for s in self.shapes]
        self.x = [orc.bf16_round(a) if dt == "bf16" else a for a, dt in zip(self.x, self.dts)]
        for b, a in zip(self.inp, self.x):
            b.upload(a)
        for b in self.out:
            self.call("tt_elementwise", 2, self.T.TT_BF16 if b.dtype == "bf16" else self.T.TT_F32, b.ptr, None, None,
                      int(np.prod(b.shape)), 77.0, 0.0, 0, None)
        self.T.lib().sync()

    def run(self, st):
        i, o, F32 = [b.ptr for b in self.inp], [b.ptr for b in self.out], self.T.TT_F32
        if self.kind == "gemm":
            self.call("tt_gemm_f32", 0, 0, 256, 100, 784, 1.0, i[0], i[1], 0.0, o[0], st)
        elif self.kind == "col_sum":
            self.call("tt_col_sum", F32, i[0], o[0], 5000, 70, st)
        elif self.kind.startswith("softmax"):
            self.call("tt_softmax_rows_f32", i[0], o[0], *self.shapes[0], st)
        elif self.kind == "conv":
            geo = (4, 8, 14, 14, 16, 5, 5, 2, 2, 1, 1, st)
            self.call("tt_conv_forward", F32, i[0], i[1], o[0], *geo)
            self.call("tt_conv_backward", F32, i[0], i[1], i[2], o[1], o[2], *geo)
        else:
            self.call("tt_attn_fwd_bf16", *i, *o, 1, 2, 40, 2000, 64, 0.125, 0, st)

    def ref(self):
        x = [a.astype(np.float64) for a in self.x]
        if self.kind == "gemm":
            return [x[0] @ x[1]]
        if self.kind == "col_sum":
            return [x[0].sum(0)]
        if self.kind.startswith("softmax"):
            return [orc.softmax_rows_f64(self.x[0])]
        if self.kind == "conv":
            im = np.pad(x[0], ((0, 0), (0, 0), (2, 2), (2, 2)))
            out, gim, gw = np.zeros(x[2].shape), np.zeros(im.shape), np.zeros(x[1].shape)
            for ky in range(5):
                for kx in range(5):
                    at = (slice(None), slice(None), slice(ky, ky + 14), slice(kx, kx + 14))
                    out += np.einsum("oc,ncyx->noyx", x[1][:, :, ky, kx], im[at])
                    gw[:, :, ky, kx] = np.einsum("noyx,ncyx->oc", x[2], im[at])
                    gim[at] += np.einsum("oc,noyx->ncyx", x[1][:, :, ky, kx], x[2])
            return [out, gim[:, :, 2:-2, 2:-2], gw]
        return list(orc.attn_fwd_f64(*self.x, 0.125, False))

    def check(self):
        for b, r in zip(self.out, self.ref()):
            # bf16 attention: also its LSE, whose row sums are of bf16 weights (2^-9 of a log of about 8)
            tol = orc.TOL["bf16"] if self.kind == "fwd_bf16" else 1e-5
            assert orc.max_rel_err(b.download().reshape(r.shape), r) <= tol, self.kind


OPS = ["gemm", "col_sum", "softmax", "softmax_aligned", "conv", "fwd_bf16"]


class Capture:
    """`with Capture(capi, stream, mode) as c:` captures; c.launch() replays."""

    def __init__(self, capi, stream, mode=THREAD_LOCAL):
        self.hip, self.stream, self.mode = capi.lib().lib, C.c_void_p(stream), mode  # its HIP runtime's symbols
        self.graph, self.exec = C.c_void_p(), C.c_void_p()

    def __enter__(self):
        assert self.hip.hipStreamBeginCapture(self.stream, self.mode) == 0
        return self

    def __exit__(self, *exc):
        rc = self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph))
        assert exc[0] is not None or rc == 0, rc

    def launch(self):
        if not self.exec:
            assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)) == 0
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0
        assert self.hip.hipStreamSynchronize(self.stream) == 0

    def destroy(self):
        if self.exec:
            self.hip.hipGraphExecDestroy(self.exec)
        if self.graph:
            self.hip.hipGraphDestroy(self.graph)


REFUSED = """
import ctypes as C
import tt_capi as T
from test_capture_gpu import Op

def in_use():
    n = C.c_size_t()
    T.lib().call("tt_mem_stats", C.byref(n), None)
    return n.value

op = Op(T, "%s")
op.fill(0)
before = in_use()
op.run(None)
assert in_use() == before, "the scratch was not refused"
op.check()
try:
    T.DeviceBuffer((1 << 20,))
except T.TTError as e:
    print("REFUSED", e.code == T.TT_ERR_NOMEM)
"""


@pytest.mark.parametrize("kind", OPS)
def test_refused_scratch_runs_unsplit(capi, kind):
    """Every allocation after the operands' fails: the call's scratch is the first of them."""
    op = Op(capi, kind)
    env = dict(os.environ, TT_FAIL_ALLOC_AFTER=str(len(op.inp) + len(op.out)), PYTHONPATH=os.pathsep.join(
        [ROOT, os.path.join(ROOT, "tests"), os.path.join(ROOT, "pku-aiprogramming_amd"),
         os.environ.get("PYTHONPATH", "")]))
    r = subprocess.run([sys.executable, "-c", REFUSED % kind], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "REFUSED True" in r.stdout, r.stdout + r.stderr


def test_scratch_is_taken_where_it_is_there(capi):
    """The operations above do split: each leaves its workspace behind."""
    n = C.c_size_t()
    for kind in OPS:
        op, st = Op(capi, kind), capi.Stream()
        op.fill(0)
        capi.lib().call("tt_mem_stats", C.byref(n), None)
        before = n.value
        op.run(st.handle)
        st.sync()
        capi.lib().call("tt_mem_stats", C.byref(n), None)
        assert n.value > before, kind
        st.destroy()


@pytest.mark.parametrize("kind", OPS)
def test_captured_calls_replay(capi, kind):
    op, other, st = Op(capi, kind), Op(capi, kind), capi.Stream()
    op.fill(0)
    with Capture(capi, st.handle) as c:
        op.run(st.handle)
    for seed in (1, 2, 3):
        op.fill(seed)
        c.launch()
        op.check()
        other.fill(seed + 10)  # eager work on the same stream between replays
        other.run(st.handle)
        st.sync()
        other.check()
    c.destroy()


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL])
@pytest.mark.parametrize("kind", OPS)
def test_calls_beside_a_capture(capi, kind, mode):
    """On a new stream, so that the scratch is a new allocation."""
    op, captured, st = Op(capi, kind), capi.Stream(), capi.Stream()
    op.fill(4)
    capi.lib().call("tt_empty_cache")
    with Capture(capi, captured.handle, mode) as c:
        op.run(st.handle)
    st.sync()
    op.check()
    c.destroy()


@pytest.mark.parametrize("kind", OPS)
def test_calls_beside_a_capture_of_the_library_stream(capi, kind):
    """They run at once and do not become part of the graph."""
    op, st = Op(capi, kind), capi.Stream()
    op.fill(5)
    capi.lib().call("tt_empty_cache")
    with Capture(capi, capi.lib().lib.tt_stream()) as c:
        op.run(st.handle)
    st.sync()
    op.check()
    c.destroy()


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL])
def test_malloc_of_a_freed_tensors_block_beside_a_capture(capi, mode):
    import myTensor as mt

    L = capi.lib()
    L.call("tt_empty_cache")
    n = 300000
    t = mt.Tensor_float([n], "gpu").ones()
    captured, p = capi.Stream(), C.c_void_p()
    del t  # its block now waits for the library stream
    with Capture(capi, captured.handle, mode) as c:
        L.check(L.lib.tt_malloc(C.byref(p), 4 * n), "tt_malloc")
    L.call("tt_free", p)
    c.destroy()


def test_captured_fp32_forward_keeps_its_scratch(capi):
    """The key splits of a later, larger bf16 forward on the stream take another buffer."""
    st = capi.Stream()

    def fwd(dt, Lq, Lk):
        x = [orc.bf16_round(np.random.default_rng(Lk).standard_normal((1, 2, n, 64)).astype(np.float32))
             for n in (Lq, Lk, Lk)]
        b = [capi.DeviceBuffer.from_numpy(a, dt) for a in x] + [capi.DeviceBuffer((1, 2, Lq, 64), dt)]
        return b, orc.attn_fwd_f64(*x, 0.125, False)[0]

    f32, ref = fwd("f32", 100, 300)
    capi.attn_fwd(*f32, None, 0.125, False, stream=st.handle)  # leaves the scratch on the stream
    st.sync()
    with Capture(capi, st.handle) as c:
        capi.attn_fwd(*f32, None, 0.125, False, stream=st.handle)
    held = []
    for Lk in (2000, 8000):
        b16, ref16 = fwd("bf16", 200, Lk)
        capi.attn_fwd(*b16, None, 0.125, False, stream=st.handle)
        held += [capi.DeviceBuffer((n,), "f32") for n in (100000, 400000, 1600000)]  # what a replaced buffer would become
        for h in held:
            h.zero()
        c.launch()
        assert orc.max_rel_err(f32[3].download(), ref) <= orc.TOL["f32"]
        assert orc.max_rel_err(b16[3].download(), ref16) <= orc.TOL["bf16"]
        assert not any(h.download().any() for h in held)
    c.destroy()
