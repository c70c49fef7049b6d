"""The work this framework is timed on: attention training steps, prefill and
decode, row softmax and GEMM through the C-ABI binding (tt_capi), and whole
MLP / CNN training steps through myTensor and myLayer.

A case is a dict of plain values with a "kind":

  step     attention forward + backward (q, k, v, dO -> o, lse, dq, dk, dv)
  fwd      attention forward (prefill, cross attention)
  decode   one query per head against a K/V cache
  softmax  row softmax, fp32
  gemm     C = op(A) op(B)
  mlp      one training step of a two-layer perceptron on 28 x 28 images
  cnn      one training step of a small convolutional network

The C-ABI calls take plain device pointers; the tensors here are torch's and
the work runs on the library stream.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pku-aiprogramming_amd")
for _p in (_PKG, os.path.join(_PKG, "optimizer")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import tt_capi  # noqa: E402

DEV = "cuda"
IMG = 28  # image side of the mlp and cnn cases
CLASSES = 10
GRID = 2048  # first-layer weights are multiples of 1 / GRID (see _first_layer)


def listed():
    def step(name, dtype, B, H, L, d, causal, std=1.0):
        return dict(name=name, kind="step", dtype=dtype, B=B, H=H, Lq=L, Lk=L, d=d, causal=causal, std=std)

    return [
        # one small head, forward and backward: launch latency and the serial chain of one workgroup
        step("step_f32_tiny", "f32", 1, 1, 64, 32, False),
        # the repository's fp32 training configuration: a chip half full, fp32 matrix units
        step("step_f32_256", "f32", 8, 8, 256, 64, False),
        # its short-sequence bf16 training configuration
        step("step_bf16_1024", "bf16", 16, 16, 1024, 64, True, 0.5),
        # its long-sequence bf16 training configuration, the largest call
        step("step_bf16_4096", "bf16", 4, 32, 4096, 128, True),
        # a single prompt of odd length run through one layer's heads
        dict(name="prefill_bf16_1531", kind="fwd", dtype="bf16", B=1, H=32, Lq=1531, Lk=1531, d=128, causal=True,
             std=1.0),
        # few queries against a long context, no mask (cross attention): odd lengths on both sides
        dict(name="cross_bf16_77x4099", kind="fwd", dtype="bf16", B=2, H=16, Lq=77, Lk=4099, d=64, causal=False,
             std=1.0),
        # decoding with a full batch: the K/V cache read at memory speed
        dict(name="decode_bf16_batch64", kind="decode", dtype="bf16", B=64, H=32, Lk=8192, d=128),
        # decoding for one user: a token's latency
        dict(name="decode_bf16_batch1", kind="decode", dtype="bf16", B=1, H=32, Lk=4097, d=128),
        # class probabilities over a long odd row
        dict(name="softmax_10007", kind="softmax", rows=8192, cols=10007),
        # the repository's large bf16 product
        dict(name="gemm_bf16_8192", kind="gemm", dtype="bf16", m=8192, n=8192, k=8192, ta=False, tb=False),
        # a training step of the 784-100-10 perceptron
        dict(name="mlp_784_100_10", kind="mlp", batch=256, hidden=100),
        # a training step of a two-convolution network on 28 x 28 images
        dict(name="cnn_28x28", kind="cnn", batch=64, c1=8, c2=16),
    ]


# ------------------------------------------------------------------ drawing

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, unit):
    """Log-uniform in [lo, hi]; half of the time a multiple of `unit`, else any value."""
    x = _log(rng, lo, hi)
    if rng.random() < 0.5:
        x = max(unit, (x + unit // 2) // unit * unit)
    return max(lo, min(hi, x))


def draw(rng):
    kind = rng.choice(["step", "step", "fwd", "fwd", "decode", "decode", "softmax", "gemm", "gemm", "mlp", "cnn"])
    if kind in ("step", "fwd"):
        dtype = rng.choice(["bf16", "bf16", "f32"])
        d, causal = rng.choice([32, 64, 128]), rng.random() < 0.6
        Lq = _size(rng, 16, 4096, 64)
        Lk = Lq if causal or kind == "step" else _size(rng, 16, 8192, 64)
        most = (1.6e12 if dtype == "bf16" else 6e10) / (12.0 * Lq * Lk * d)  # heads
        heads = _log(rng, 1, max(1, min(512, most, 2 ** 26 / (max(Lq, Lk) * d))))
        H = rng.choice([1, 8, 16, 32])
        H = H if H <= heads else 1
        return dict(kind=kind, dtype=dtype, B=max(1, heads // H), H=H, Lq=Lq, Lk=Lk, d=d, causal=causal, std=1.0)
    if kind == "decode":
        d, Lk = rng.choice([32, 64, 128]), _size(rng, 64, 32768, 256)
        H = rng.choice([8, 16, 32])
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), B=_log(rng, 1, max(1, min(64, 2 ** 30 / (H * Lk * d)))),
                    H=H, Lk=Lk, d=d)
    if kind == "softmax":
        cols = _size(rng, 10, 262144, 64)
        return dict(kind=kind, rows=_log(rng, 1, max(1, min(65536, 2 ** 27 / cols))), cols=cols)
    if kind == "gemm":
        dtype = rng.choice(["bf16", "f32"])
        m, n, k = (_size(rng, 16, 8192 if dtype == "bf16" else 4096, 64) for _ in range(3))
        while 2.0 * m * n * k > 2.8e11:
            m, n, k = (m + 1) // 2, (n + 1) // 2, (k + 1) // 2
        return dict(kind=kind, dtype=dtype, m=m, n=n, k=k, ta=rng.random() < 0.5, tb=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind=kind, batch=_size(rng, 16, 2048, 32), hidden=_size(rng, 32, 1024, 16))
    return dict(kind="cnn", batch=_size(rng, 8, 128, 16), c1=rng.randint(4, 16), c2=rng.randint(6, 32))


# ------------------------------------------------------------------ inputs

_T = {"bf16": torch.bfloat16, "f32": torch.float32}


def _scale(d):
    return float(np.float32(1.0 / math.sqrt(d)))


def _normal(g, shape, dtype, std=1.0):
    x = torch.empty(shape, dtype=_T[dtype], device=DEV)
    return x.normal_(0.0, std, generator=g)


def _inputs(case, seed):
    """The device inputs of the C-ABI kinds, from the seed alone."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    if kind in ("step", "fwd", "decode"):
        B, H, d, Lk = case["B"], case["H"], case["d"], case["Lk"]
        Lq, std = case.get("Lq", 1), case.get("std", 1.0)
        x = {"q": _normal(g, (B, H, Lq, d), case["dtype"], std), "k": _normal(g, (B, H, Lk, d), case["dtype"], std),
             "v": _normal(g, (B, H, Lk, d), case["dtype"], std)}
        if kind == "step":
            x["do"] = _normal(g, (B, H, Lq, d), case["dtype"])
        return x
    if kind == "softmax":
        return {"x": _normal(g, (case["rows"], case["cols"]), "f32", 3.0)}
    m, n, k = case["m"], case["n"], case["k"]
    return {"a": _normal(g, (k, m) if case["ta"] else (m, k), case["dtype"]),
            "b": _normal(g, (n, k) if case["tb"] else (k, n), case["dtype"])}


def _first_layer(rng, shape, fan_in):
    """Weights in +-1/sqrt(fan_in) on a grid of 1 / GRID.  With 8-bit pixels
    the first layer's sums are then exact in fp32, so that ReLU and the
    pooling behind it pick the same elements whatever the order of the sums;
    every later layer takes ordinary fp32 values."""
    lim = 1.0 / math.sqrt(fan_in)
    return (np.round(rng.uniform(-lim, lim, shape) * GRID) / GRID).astype(np.float32)


def _layer(rng, shape, fan_in):
    lim = 1.0 / math.sqrt(fan_in)
    return rng.uniform(-lim, lim, shape).astype(np.float32)


def _images(rng, batch):
    """8-bit gray images, most pixels background."""
    px = rng.integers(0, 256, (batch, 1, IMG, IMG)) * (rng.random((batch, 1, IMG, IMG)) < 0.25)
    return (px / 256.0).astype(np.float32)


def _net(case, seed):
    """The host values of an mlp or cnn case, from the seed alone."""
    rng = np.random.default_rng(int(seed))
    b = case["batch"]
    x = {"images": _images(rng, b), "labels": rng.integers(0, CLASSES, b).astype(np.int32)}
    if case["kind"] == "mlp":
        h = case["hidden"]
        x["images"] = x["images"].reshape(b, IMG * IMG)
        x.update(w1=_first_layer(rng, (IMG * IMG, h), IMG * IMG), b1=_first_layer(rng, (h,), IMG * IMG),
                 w2=_layer(rng, (h, CLASSES), h), b2=_layer(rng, (CLASSES,), h))
    else:
        c1, c2 = case["c1"], case["c2"]
        x.update(w1=_first_layer(rng, (c1, 1, 5, 5), 25), w2=_layer(rng, (c2, c1, 5, 5), 25 * c1),
                 w3=_layer(rng, (c2 * 49, CLASSES), c2 * 49), b3=_layer(rng, (CLASSES,), c2 * 49))
    return x


# ------------------------------------------------------------------ prepare, run

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("mlp", "cnn"):
        import myTensor as mt

        x = _net(case, seed)
        s = {n: mt.Tensor_float(a, "gpu") for n, a in x.items() if n != "labels"}
        s["labels"] = mt.Tensor_int(x["labels"].reshape(1, -1), "gpu")
        return {"case": case, "t": s}
    s = {"case": case, "lib": tt_capi.lib(), **_inputs(case, seed)}
    if kind in ("step", "fwd"):
        s["o"] = torch.empty_like(s["q"])
        s["lse"] = torch.empty(s["q"].shape[:3], dtype=torch.float32, device=DEV)
        if kind == "step":
            for n in ("q", "k", "v"):
                s["d" + n] = torch.empty_like(s[n])
    elif kind == "decode":
        s["o"] = torch.empty_like(s["q"])
    elif kind == "softmax":
        s["y"] = torch.empty_like(s["x"])
    else:
        s["c"] = torch.empty((case["m"], case["n"]), dtype=_T[case["dtype"]], device=DEV)
    torch.cuda.synchronize()  # torch filled these on its own stream
    return s


def _run_mlp(case, t):
    import myLayer as ml
    import myTensor as mt

    def new():
        return mt.Tensor_float([1], "gpu")

    h, z, p, loss, gz = new(), new(), new(), new(), new()
    ml.FcForward(t["images"], h, t["w1"], t["b1"])
    a = h.ReluForward()
    ml.FcForward(a, z, t["w2"], t["b2"])
    ml.SoftmaxForward(z, p)
    ml.CrossEntropyLoss(p, t["labels"], loss)
    ml.CrossEntropyLossBackward(p, t["labels"], gz)
    gz.mults(1.0 / case["batch"])
    ga, gw2, gb2, gx, gw1, gb1 = new(), new(), new(), new(), new(), new()
    ml.FcBackward(a, z, t["w2"], t["b2"], ga, gz, gw2, gb2)
    gh = h.ReluBackward(ga)
    ml.FcBackward(t["images"], h, t["w1"], t["b1"], gx, gh, gw1, gb1)
    return {"p": p.numpy(), "loss": loss.numpy(), "gw1": gw1.numpy(), "gb1": gb1.numpy(), "gw2": gw2.numpy(),
            "gb2": gb2.numpy()}


def _run_cnn(case, t):
    import myLayer as ml
    import myTensor as mt

    def new():
        return mt.Tensor_float([1], "gpu")

    h1, m1, mask, h2, z, p, loss, gz = (new() for _ in range(8))
    ml.ConvForward(t["images"], h1, t["w1"], 2, 2, 1, 1)
    a1 = h1.ReluForward()
    ml.MaxPoolingForward(a1, m1, mask, [2, 2], 0, 0, 2, 2)
    ml.ConvForward(m1, h2, t["w2"], 2, 2, 2, 2)
    a2 = h2.SigmoidForward()
    f = a2.flatten()
    ml.FcForward(f, z, t["w3"], t["b3"])
    ml.SoftmaxForward(z, p)
    ml.CrossEntropyLoss(p, t["labels"], loss)
    ml.CrossEntropyLossBackward(p, t["labels"], gz)
    gz.mults(1.0 / case["batch"])
    gf, gw3, gb3, gm, gw2, ga1, gx, gw1 = (new() for _ in range(8))
    ml.FcBackward(f, z, t["w3"], t["b3"], gf, gz, gw3, gb3)
    gf.resize(h2.get_shape())
    gh2 = h2.SigmoidBackward(gf)
    ml.ConvBackward(m1, h2, t["w2"], gm, gh2, gw2, 2, 2, 2, 2)
    ml.MaxPoolingBackward(gm, mask, ga1, [IMG, IMG], [2, 2], 0, 0, 2, 2)
    gh1 = h1.ReluBackward(ga1)
    ml.ConvBackward(t["images"], h1, t["w1"], gx, gh1, gw1, 2, 2, 1, 1)
    return {"p": p.numpy(), "loss": loss.numpy(), "gw1": gw1.numpy(), "gw2": gw2.numpy(), "gw3": gw3.numpy(),
            "gb3": gb3.numpy()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mlp":
        return _run_mlp(case, state["t"])
    if kind == "cnn":
        return _run_cnn(case, state["t"])
    call, s = state["lib"].call, state
    if kind in ("step", "fwd"):
        dims = (case["B"], case["H"], case["Lq"], case["Lk"], case["d"], _scale(case["d"]), int(case["causal"]), None)
        qkv = (s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(), s["lse"].data_ptr())
        call("tt_attn_fwd_" + case["dtype"], *qkv, *dims)
        if kind == "fwd":
            return {"o": s["o"], "lse": s["lse"]}
        call("tt_attn_bwd_" + case["dtype"], *qkv, s["do"].data_ptr(), s["dq"].data_ptr(), s["dk"].data_ptr(),
             s["dv"].data_ptr(), *dims)
        return {n: s[n] for n in ("o", "lse", "dq", "dk", "dv")}
    if kind == "decode":
        call("tt_attn_decode_" + case["dtype"], s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
             s["o"].data_ptr(), None, case["B"], case["H"], case["Lk"], case["d"], _scale(case["d"]), None)
        return s["o"]
    if kind == "softmax":
        call("tt_softmax_rows_f32", s["x"].data_ptr(), s["y"].data_ptr(), case["rows"], case["cols"], None)
        return s["y"]
    call("tt_gemm_" + case["dtype"], int(case["ta"]), int(case["tb"]), case["m"], case["n"], case["k"], 1.0,
         s["a"].data_ptr(), s["b"].data_ptr(), 0.0, s["c"].data_ptr(), None)
    return s["c"]


# ------------------------------------------------------------------ work, tolerance

def work(case):
    kind = case["kind"]
    e = 2 if case.get("dtype") == "bf16" else 4
    if kind in ("step", "fwd", "decode"):
        bh, Lq, Lk, d = case["B"] * case["H"], case.get("Lq", 1), case["Lk"], case["d"]
        rows, keys = bh * Lq * d * e, bh * Lk * d * e
        # forward: scores and P V; backward: dV, dP, dQ, dK (no recomputation counted)
        fwd = 4.0 * bh * Lq * Lk * d * (0.5 if case.get("causal") else 1.0)
        if kind == "step":
            return {"bytes": 4 * rows + 4 * keys + 4 * bh * Lq, "flops": 3 * fwd}
        return {"bytes": 2 * rows + 2 * keys + (4 * bh * Lq if kind == "fwd" else 0), "flops": fwd}
    if kind == "softmax":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 4.0 * case["rows"] * case["cols"]}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": e * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    b = case["batch"]
    if kind == "mlp":
        h, px = case["hidden"], IMG * IMG
        w = px * h + h + h * CLASSES + CLASSES
        # forward, weight gradients, and the hidden layer's gradient
        return {"bytes": 4 * (b * px + 2 * w + b * (CLASSES + 1) + 1),
                "flops": 2.0 * b * (2 * px * h + 3 * h * CLASSES)}
    c1, c2 = case["c1"], case["c2"]
    conv1, conv2, fc = c1 * 25 * IMG * IMG, c2 * c1 * 25 * 49, c2 * 49 * CLASSES
    w = 25 * c1 + 25 * c1 * c2 + c2 * 49 * CLASSES + CLASSES
    return {"bytes": 4 * (b * IMG * IMG + 2 * w + b * (CLASSES + 1) + 1),
            "flops": 2.0 * b * (2 * conv1 + 3 * conv2 + 3 * fc)}


def tolerance(case):
    # about four times the largest errors against exact() that the path shows
    # (bf16 products 1.7e-3, bf16 attention 2.5e-3; fp32 sums up to 5e-7 at the
    # listed sizes and several times that over the longest sums drawn)
    if case["kind"] in ("mlp", "cnn"):
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] == "softmax":
        return {"rel": 1e-6, "max": 1e-4}
    if case.get("dtype") == "bf16":
        if case["kind"] == "gemm":
            return {"rel": 7e-3, "max": 0.05}
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------------------ 64-bit results

def _attn64(case, x):
    B, H, Lk, d = case["B"], case["H"], case["Lk"], case["d"]
    Lq, causal, sc = case.get("Lq", 1), case.get("causal", False), _scale(case["d"])
    step = case["kind"] == "step"
    out = {"o": torch.empty(x["q"].shape, dtype=torch.float64, device=DEV),
           "lse": torch.empty((B, H, Lq), dtype=torch.float64, device=DEV)}
    if step:
        for n in ("q", "k", "v"):
            out["d" + n] = torch.empty(x[n].shape, dtype=torch.float64, device=DEV)
    mask = torch.ones(Lq, Lk, dtype=torch.bool, device=DEV).triu(1) if causal else None
    for b in range(B):
        for h in range(H):
            q, k, v = (x[n][b, h].double() for n in ("q", "k", "v"))
            s = (q @ k.t().contiguous()) * sc
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            lse = torch.logsumexp(s, 1)
            p = torch.exp_(s.sub_(lse[:, None]))
            o = p @ v
            out["o"][b, h], out["lse"][b, h] = o, lse
            if step:
                do = x["do"][b, h].double()
                out["dv"][b, h] = p.t().contiguous() @ do
                ds = (do @ v.t().contiguous()).sub_((do * o).sum(1, keepdim=True)).mul_(p).mul_(sc)
                out["dq"][b, h] = ds @ k
                out["dk"][b, h] = ds.t().contiguous() @ q
    return out


def _net64(case, seed):
    x = {n: torch.from_numpy(a) for n, a in _net(case, seed).items()}
    w = {n: a.double().requires_grad_() for n, a in x.items() if n[0] in "wb"}
    img, lab = x["images"].double(), x["labels"].long()
    if case["kind"] == "mlp":
        z = torch.relu(img @ w["w1"] + w["b1"]) @ w["w2"] + w["b2"]
    else:
        F = torch.nn.functional
        a1 = F.max_pool2d(torch.relu(F.conv2d(img, w["w1"], padding=2)), 2)
        a2 = torch.sigmoid(F.conv2d(a1, w["w2"], padding=2, stride=2))
        z = a2.flatten(1) @ w["w3"] + w["b3"]
    logp = torch.log_softmax(z, 1)
    loss = -logp[torch.arange(len(lab)), lab].sum()
    (loss / case["batch"]).backward()
    return {"p": logp.detach().exp(), "loss": loss.detach().reshape(1), **{"g" + n: a.grad for n, a in w.items()}}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mlp", "cnn"):
        return _net64(case, seed)
    x = _inputs(case, seed)
    if kind in ("step", "fwd"):
        return _attn64(case, x)
    if kind == "decode":
        return _attn64(case, x)["o"]
    if kind == "softmax":
        return torch.softmax(x["x"].double(), 1)
    a = x["a"].double().t().contiguous() if case["ta"] else x["a"].double()
    b = x["b"].double().t().contiguous() if case["tb"] else x["b"].double()
    return a @ b
