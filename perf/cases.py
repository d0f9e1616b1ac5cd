"""The work that this framework is used for, as cases that can be timed and checked.

Each case is one forward pass and its backward through public entry points: the device calls of
dreamcompiler_amd.hip on tensors that are on the GPU, and (kind "mlp") the runtime builtins of
dreamcompiler_amd.runtime on host tensors, as a compiled program calls them.

  listed()              the named cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   inputs, made from the seed, and the buffers that a program keeps
  run(state)            one pass; returns every output and gradient
  work(case)            bytes and floating-point operations that a pass cannot do without
  tolerance(case)       how far another correct implementation may be from this one
  exact(case, seed)     the same outputs in 64 bits by plain torch
"""
import ctypes
import math

import numpy as np
import torch

from dreamcompiler_amd import hip
from dreamcompiler_amd import runtime as rt

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f64": torch.float64}
BYTES = {"f32": 4, "bf16": 2, "f64": 8}


def listed():
    return [
        # A training step of a small classifier as a compiled program issues it: builtins on
        # host tensors, so the copies over PCIe and the host's own loops are part of it.
        dict(name="mlp_step", kind="mlp", batch=4096, inp=784, hidden=257, out=10),
        # The hidden layer of that classifier alone, on the device: fused bias and ReLU, a bias
        # gradient, two gradients of products whose sides are no multiple of a tile.
        dict(name="linear_relu_layer", kind="linear", rows=4096, inp=784, out=257),
        # `@` in the default precision at an ordinary size, with the products of its backward.
        dict(name="matmul_f32", kind="matmul", dtype="f32", M=1024, N=1024, K=1024),
        # `@` in reduced precision at the largest size in use.
        dict(name="matmul_bf16_large", kind="matmul", dtype="bf16", M=8192, N=8192, K=8192),
        # `@` in reduced precision with odd sides: rows that are not 16-byte aligned.
        dict(name="matmul_bf16_ragged", kind="matmul", dtype="bf16", M=1023, N=2050, K=1537),
        # `@` below the size from which the runtime leaves double precision.
        dict(name="matmul_f64", kind="matmul", dtype="f64", M=511, N=511, K=511),
        # The attention block of a character-level model: the smallest flash call.
        dict(name="flash_f32_small", kind="flash", dtype="f32", BH=24, S=256, D=64, causal=True),
        # Attention of a long context in reduced precision: the largest flash call.
        dict(name="flash_bf16_large", kind="flash", dtype="bf16", BH=128, S=4096, D=128,
             causal=True),
        # Attention of an encoder over a sequence that ends inside a tile.
        dict(name="flash_bf16_ragged", kind="flash", dtype="bf16", BH=32, S=1000, D=64,
             causal=False),
        # Attention with a head dimension above 128, which the runtime computes in fp64.
        dict(name="attention_f64", kind="attention", BH=16, S=1024, D=256, causal=True),
        # A 3x3 layer of a convolutional network.
        dict(name="conv3x3", kind="conv", N=64, Cin=64, H=56, W=56, Cout=64, KH=3, KW=3, pad=1,
             stride=1),
        # The log-softmax of a wide classification head.
        dict(name="log_softmax_wide", kind="rows", op="log_softmax", R=4096, C=5000),
    ]


# --------------------------------------------------------------------------- drawing

def _size(rng, lo, hi):
    """A size of lo..hi, even over its logarithm: half of them a multiple of 16 (where that
    fits), half as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= 16:
        v = v // 16 * 16
    return max(lo, min(hi, v))


def _seconds(case):
    """A rough upper estimate of a pass: keeps drawn cases below the largest listed one."""
    w = work(case)
    rate = {"bf16": 500e12, "f32": 50e12, "f64": 15e12}[case.get("dtype", "f64" if case["kind"] == "attention" else "f32")]
    return w["flops"] / rate + w["bytes"] / 2e12


def _draw(rng):
    kind = rng.choice(("mlp", "linear", "matmul", "matmul", "matmul", "flash", "flash",
                       "attention", "conv", "conv", "rows"))
    if kind == "mlp":
        return dict(kind=kind, batch=_size(rng, 64, 4096), inp=_size(rng, 16, 1024),
                    hidden=_size(rng, 16, 512), out=_size(rng, 2, 128))
    if kind == "linear":
        return dict(kind=kind, rows=_size(rng, 64, 16384), inp=_size(rng, 32, 4096),
                    out=_size(rng, 32, 4096))
    if kind == "matmul":
        dtype = rng.choice(("f32", "bf16", "f64"))
        if dtype == "f64":   # below the runtime's threshold of 512 * 512 results
            M = _size(rng, 32, 2048)
            return dict(kind=kind, dtype=dtype, M=M, N=_size(rng, 16, min(2048, 262143 // M)),
                        K=_size(rng, 32, 2048))
        return dict(kind=kind, dtype=dtype, M=_size(rng, 128, 8192), N=_size(rng, 128, 8192),
                    K=_size(rng, 64, 8192))
    if kind == "flash":
        return dict(kind=kind, dtype=rng.choice(("f32", "bf16")), BH=_size(rng, 4, 128),
                    S=_size(rng, 128, 4096), D=rng.choice((32, 64, 128)),
                    causal=rng.random() < 0.6)
    if kind == "attention":
        return dict(kind=kind, BH=_size(rng, 1, 16), S=_size(rng, 64, 1024),
                    D=_size(rng, 129, 256), causal=rng.random() < 0.6)
    if kind == "conv":
        k = rng.choice((1, 3, 3, 5))
        side = _size(rng, 7, 112)
        return dict(kind=kind, N=_size(rng, 4, 64), Cin=rng.choice((3, _size(rng, 16, 256))),
                    H=side, W=side, Cout=_size(rng, 16, 256), KH=k, KW=k, pad=k // 2,
                    stride=rng.choice((1, 1, 2)))
    return dict(kind="rows", op=rng.choice(("softmax", "log_softmax", "layer_norm")),
                R=_size(rng, 256, 16384), C=_size(rng, 64, 16384))


def draw(rng):
    while True:
        case = _draw(rng)
        if _seconds(case) < 2.0e-3:
            return case


# --------------------------------------------------------------------------- inputs

def _normal(seed, *specs):
    """One tensor for each (shape, dtype, scale), from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(torch.randn(shape, generator=g, device="cuda",
                         dtype=torch.float64 if dt == "f64" else torch.float32) * scale)
            .to(TORCH[dt]) for shape, dt, scale in specs]


def _out_side(c):
    return ((c["H"] + 2 * c["pad"] - c["KH"]) // c["stride"] + 1,
            (c["W"] + 2 * c["pad"] - c["KW"]) // c["stride"] + 1)


def _inputs(c, seed):
    """The tensors that a pass reads, by name."""
    k = c["kind"]
    if k == "mlp":
        r = np.random.default_rng(seed)
        B, I, H, O = c["batch"], c["inp"], c["hidden"], c["out"]
        t = dict(X=r.uniform(0, 1, (B, I)), W1=r.standard_normal((H, I)) * math.sqrt(2 / I),
                 b1=r.standard_normal((1, H)) * 0.1,
                 W2=r.standard_normal((O, H)) * math.sqrt(2 / H),
                 b2=r.standard_normal((1, O)) * 0.1, G=r.standard_normal((B, O)))
        # A hidden unit within rounding of zero may fall on either side of the ReLU, so the
        # samples that have one carry no loss.
        t["G"][(np.abs(t["X"] @ t["W1"].T + t["b1"]) < 1e-5).any(axis=1)] = 0.0
        return t
    if k == "linear":
        R, I, O = c["rows"], c["inp"], c["out"]
        X, W, b, dY = _normal(seed, ((R, I), "f32", 1.0), ((O, I), "f32", math.sqrt(2 / I)),
                              ((O,), "f32", 0.1), ((R, O), "f32", 1.0))
        # A unit within rounding of zero may fall on either side of the ReLU: no gradient there.
        dY[(X.double() @ W.double().t() + b).abs() < 1e-5] = 0.0
        return dict(X=X, W=W, b=b, dY=dY)
    if k == "matmul":
        M, N, K, dt = c["M"], c["N"], c["K"], c["dtype"]
        return dict(zip(("A", "B", "dC"), _normal(
            seed, ((M, K), dt, 1.0), ((K, N), dt, 1.0), ((M, N), dt, 1.0))))
    if k in ("flash", "attention"):
        shape, dt = (c["BH"], c["S"], c["D"]), c.get("dtype", "f64")
        s = 1.0 if dt == "bf16" else 0.5
        return dict(zip(("Q", "K", "V", "dO"), _normal(
            seed, (shape, dt, s), (shape, dt, s), (shape, dt, s), (shape, dt, 1.0))))
    if k == "conv":
        OH, OW = _out_side(c)
        fan = c["Cin"] * c["KH"] * c["KW"]
        return dict(zip(("X", "Kn", "b", "dY"), _normal(
            seed, ((c["N"], c["Cin"], c["H"], c["W"]), "f32", 1.0),
            ((c["Cout"], fan), "f32", math.sqrt(2 / fan)), ((c["Cout"],), "f32", 0.1),
            ((c["N"], c["Cout"], OH, OW), "f32", 1.0))))
    return dict(zip(("X", "dY"), _normal(seed, ((c["R"], c["C"]), "f32", 2.0),
                                         ((c["R"], c["C"]), "f32", 1.0))))


def _like(x, dtype=None):
    return torch.empty(x.shape, dtype=dtype or x.dtype, device="cuda")


class State:
    """A case's inputs and output buffers; `p` holds the device address of each."""

    def __init__(self, case, seed):
        self.case = case
        self.t = _inputs(case, seed)
        c, k, t = case, case["kind"], self.t
        if k == "linear":
            t["Y"], t["dX"], t["dW"], t["db"] = _like(t["dY"]), _like(t["X"]), _like(t["W"]), _like(t["b"])
        elif k == "matmul":
            dt = torch.float64 if c["dtype"] == "f64" else torch.float32
            t["C"], t["dA"], t["dB"] = _like(t["dC"], dt), _like(t["A"], dt), _like(t["B"], dt)
        elif k in ("flash", "attention"):
            t["O"] = _like(t["Q"])
            if k == "flash":
                t["LSE"] = torch.empty((c["BH"], c["S"]), device="cuda")
            for n in "QKV":
                t["d" + n] = _like(t["Q"], torch.float64 if k == "attention" else torch.float32)
        elif k == "conv":
            t["Y"], t["dX"], t["dK"] = _like(t["dY"]), _like(t["X"]), _like(t["Kn"])
            if c["stride"] > 1:   # the data gradient of a strided layer: a product and col2im
                OH, OW = _out_side(c)
                cols = c["N"] * OH * OW
                t["g"] = torch.empty((c["Cout"], cols), device="cuda")
                t["col"] = torch.empty((c["Cin"] * c["KH"] * c["KW"], cols), device="cuda")
        elif k == "rows":
            t["Y"], t["dX"] = _like(t["X"]), _like(t["X"])
        self.p = {n: x.data_ptr() for n, x in t.items()}
        torch.cuda.synchronize()   # the library has a stream of its own


class MlpState:
    """A small classifier's tensors in the runtime, and the log-probabilities of the last pass."""

    def __init__(self, case, seed):
        self.case = case
        self.t = {n: rt.tensor(x) for n, x in _inputs(case, seed).items()}
        self.last = None

    def __del__(self):
        rt.release(self.last, *self.t.values())


def prepare(case, seed):
    return MlpState(case, seed) if case["kind"] == "mlp" else State(case, seed)


# --------------------------------------------------------------------------- one pass

def _host(state, ptr, rows, size):
    """A runtime tensor's values as an array, without a copy; it keeps the tensor's state."""
    a = (ctypes.c_double * size).from_address(ctypes.addressof(ptr.contents))
    a.state = state
    return np.frombuffer(a).reshape(rows, -1)


def _run_mlp(s):
    L, t = rt.load(), s.t
    params = ("X", "W1", "b1", "W2", "b2")
    for n in params:
        rt.release(L.zero_grad(t[n]))
    rt.release(s.last)
    h = L.dream_linear_relu(t["X"], t["W1"], t["b1"])
    y = L.dream_linear(h, t["W2"], t["b2"])
    lp = L.dream_log_softmax(y)
    m = L.tensor_mul(lp, t["G"])
    loss = L.sum(m)
    r = L.backward(loss)
    rt.release(r, loss, m, y, h)
    s.last = lp
    out = {"logp": _host(s, lp.contents.data, lp.contents.d0, lp.contents.size)}
    for n in params:
        c = t[n].contents
        out["d" + n] = _host(s, c.grad, c.d0, c.size)
    return out


def run(s):
    c, k = s.case, s.case["kind"]
    if k == "mlp":
        return _run_mlp(s)
    t, p = s.t, s.p
    if k == "linear":
        R, I, O = c["rows"], c["inp"], c["out"]
        hip.gemm_ex("f32", 0, 1, R, O, I, p["X"], I, 0, p["W"], I, 0, 0.0, p["Y"], O, 0,
                    bias=p["b"], relu=True)
        hip.linear_bias_grad(p["Y"], p["dY"], p["db"], R, O, relu=True)
        hip.gemm_f32(0, 0, R, I, O, p["dY"], O, p["W"], I, 0.0, p["dX"], I)
        hip.gemm_f32(1, 0, O, I, R, p["dY"], O, p["X"], I, 0.0, p["dW"], I)
        return [t[n] for n in ("Y", "dY", "db", "dX", "dW")]
    if k == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        f = {"f32": hip.gemm_f32, "bf16": hip.gemm_bf16, "f64": hip.gemm_f64}[c["dtype"]]
        f(0, 0, M, N, K, p["A"], K, p["B"], N, 0.0, p["C"], N)
        f(0, 1, M, K, N, p["dC"], N, p["B"], N, 0.0, p["dA"], K)
        f(1, 0, K, N, M, p["A"], K, p["dC"], N, 0.0, p["dB"], N)
        return [t[n] for n in ("C", "dA", "dB")]
    if k == "flash":
        dt = hip.F32 if c["dtype"] == "f32" else hip.BF16
        a = (dt, c["BH"], c["S"], c["D"], 1.0 / math.sqrt(c["D"]), c["causal"], p["Q"], p["K"],
             p["V"])
        hip.flash_fwd(*a, p["O"], p["LSE"])
        hip.flash_bwd(*a, p["O"], p["dO"], p["LSE"], p["dQ"], p["dK"], p["dV"], 0)
        return [t[n] for n in ("O", "LSE", "dQ", "dK", "dV")]
    if k == "attention":
        a = (c["BH"], c["S"], c["D"], 1.0 / math.sqrt(c["D"]), c["causal"], p["Q"], p["K"], p["V"])
        hip.attention_f64_fwd(*a, p["O"])
        hip.attention_f64_bwd(*a, p["dO"], p["dQ"], p["dK"], p["dV"], 0)
        return [t[n] for n in ("O", "dQ", "dK", "dV")]
    if k == "conv":
        N, Cin, H, W, Cout, KH, KW, pad, stride = shape = [c[n] for n in (
            "N", "Cin", "H", "W", "Cout", "KH", "KW", "pad", "stride")]
        hip.conv2d_fwd(p["X"], p["Kn"], p["b"], p["Y"], *shape)
        if stride == 1:
            hip.conv2d_bwd_data(p["dY"], p["Kn"], p["dX"], *shape)
        else:
            OH, OW = _out_side(c)
            cols, fan = N * OH * OW, Cin * KH * KW
            hip.nct_to_cnt(p["dY"], p["g"], N, Cout, OH * OW)
            hip.gemm_f32(1, 0, fan, cols, Cout, p["Kn"], fan, p["g"], cols, 0.0, p["col"], cols)
            hip.col2im(p["col"], p["dX"], N, Cin, H, W, KH, KW, pad, stride)
        hip.conv2d_bwd_filter(p["dY"], p["X"], p["dK"], *shape)
        return [t[n] for n in ("Y", "dX", "dK")]
    R, C = c["R"], c["C"]
    if c["op"] == "layer_norm":
        hip.layer_norm(p["X"], p["Y"], R, C)
        hip.layer_norm_bwd(p["X"], p["Y"], p["dY"], p["dX"], R, C)
    else:
        log = c["op"] == "log_softmax"
        hip.row_softmax(p["X"], p["Y"], R, C, log=log)
        hip.row_softmax_bwd(p["Y"], p["dY"], p["dX"], R, C, log=log)
    return [t[n] for n in ("Y", "dX")]


# --------------------------------------------------------------------------- what a pass needs

def work(c):
    k = c["kind"]
    if k == "mlp":   # host tensors: the bytes are those of the arrays read and written there
        B, I, H, O = c["batch"], c["inp"], c["hidden"], c["out"]
        params = H * I + H + O * H + O
        return {"bytes": 8 * (2 * B * I + 2 * B * O + 2 * params), "flops": 6 * B * (I * H + H * O)}
    if k == "linear":
        R, I, O = c["rows"], c["inp"], c["out"]
        return {"bytes": 4 * (2 * R * I + 2 * O * I + 2 * O + 3 * R * O), "flops": 6 * R * I * O}
    if k == "matmul":
        M, N, K, e = c["M"], c["N"], c["K"], BYTES[c["dtype"]]
        n = M * K + K * N + M * N
        return {"bytes": n * (e + (8 if c["dtype"] == "f64" else 4)), "flops": 6 * M * N * K}
    if k in ("flash", "attention"):
        n, e = c["BH"] * c["S"] * c["D"], BYTES[c.get("dtype", "f64")]
        pairs = c["S"] * (c["S"] + 1) // 2 if c["causal"] else c["S"] * c["S"]
        # forward two products over the visible pairs, backward five
        return {"bytes": n * (5 * e + 3 * max(e, 4)), "flops": 14 * c["BH"] * pairs * c["D"]}
    if k == "conv":
        OH, OW = _out_side(c)
        x, y = c["N"] * c["Cin"] * c["H"] * c["W"], c["N"] * c["Cout"] * OH * OW
        kn = c["Cout"] * c["Cin"] * c["KH"] * c["KW"]
        return {"bytes": 4 * (2 * x + 2 * y + 2 * kn), "flops": 6 * c["N"] * OH * OW * kn}
    n = c["R"] * c["C"]
    return {"bytes": 4 * 4 * n, "flops": 16 * n}


def tolerance(c):
    """About four times the error against exact() at the largest sizes of the ranges: 2.5e-3
    where probabilities and results are rounded to bf16, 1.2e-6 for fp32 sums over 8192 terms
    (bf16 products too: they are exact in fp32 and summed there), 1.5e-15 in fp64."""
    if c["kind"] == "flash" and c["dtype"] == "bf16":
        return {"rel": 1e-2}
    if c["kind"] == "attention" or c.get("dtype") == "f64":
        return {"rel": 1e-14}
    return {"rel": 5e-6}


# --------------------------------------------------------------------------- in 64 bits

def _exact_attention(c, t):
    Q, K, V, dO = (t[n].double() for n in ("Q", "K", "V", "dO"))
    scale = 1.0 / math.sqrt(c["D"])
    S = c["S"]
    hidden = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1) if c["causal"] else None
    O, dQ, dK, dV = (torch.empty_like(Q) for _ in range(4))
    LSE = torch.empty((c["BH"], S), dtype=torch.float64, device="cuda")
    for b in range(c["BH"]):
        s = (Q[b] @ K[b].t()) * scale
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        LSE[b] = torch.logsumexp(s, dim=1)
        P = torch.exp(s - LSE[b][:, None])
        O[b] = P @ V[b]
        dV[b] = P.t() @ dO[b]
        dS = P * (dO[b] @ V[b].t() - (dO[b] * O[b]).sum(1, keepdim=True))
        dQ[b] = scale * (dS @ K[b])
        dK[b] = scale * (dS.t() @ Q[b])
    return [O, LSE, dQ, dK, dV] if c["kind"] == "flash" else [O, dQ, dK, dV]


def _exact_conv(c, t):
    """Per tap, so that no matrix of windows is built."""
    OH, OW = _out_side(c)
    N, Cin, Cout, st, pad = c["N"], c["Cin"], c["Cout"], c["stride"], c["pad"]
    X = torch.nn.functional.pad(t["X"].double(), (pad, pad, pad, pad))
    Kn = t["Kn"].double().reshape(Cout, Cin, c["KH"], c["KW"])
    dY = t["dY"].double().permute(1, 0, 2, 3).reshape(Cout, -1)
    Y = torch.zeros((Cout, N * OH * OW), dtype=torch.float64, device="cuda")
    dX, dK = torch.zeros_like(X), torch.empty_like(Kn)
    for i in range(c["KH"]):
        for j in range(c["KW"]):
            at = (slice(None), slice(None), slice(i, i + st * (OH - 1) + 1, st),
                  slice(j, j + st * (OW - 1) + 1, st))
            win = X[at].permute(1, 0, 2, 3).reshape(Cin, -1)
            w = Kn[:, :, i, j].contiguous()
            Y += w @ win
            dK[:, :, i, j] = dY @ win.t()
            dX[at] += (w.t() @ dY).reshape(Cin, N, OH, OW).permute(1, 0, 2, 3)
    Y = Y.reshape(Cout, N, OH, OW).permute(1, 0, 2, 3) + t["b"].double()[None, :, None, None]
    dX = dX[:, :, pad:pad + c["H"], pad:pad + c["W"]]
    return [Y.contiguous(), dX.contiguous(), dK.reshape(Cout, -1)]


def exact(c, seed):
    k, t = c["kind"], _inputs(c, seed)
    if k == "mlp":
        X, W1, b1, W2, b2, G = (torch.from_numpy(t[n]) for n in ("X", "W1", "b1", "W2", "b2", "G"))
        h = torch.relu(X @ W1.t() + b1)
        lp = torch.log_softmax(h @ W2.t() + b2, dim=1)
        dy = G - lp.exp() * G.sum(1, keepdim=True)
        dh = (dy @ W2) * (h > 0)
        return {"logp": lp, "dX": dh @ W1, "dW1": dh.t() @ X, "db1": dh.sum(0, keepdim=True),
                "dW2": dy.t() @ h, "db2": dy.sum(0, keepdim=True)}
    if k == "linear":
        X, W, b, dY = (t[n].double() for n in ("X", "W", "b", "dY"))
        Y = torch.relu(X @ W.t() + b)
        dY = dY * (Y > 0)
        return [Y, dY, dY.sum(0), dY @ W, dY.t() @ X]
    if k == "matmul":
        A, B, dC = (t[n].double() for n in ("A", "B", "dC"))
        return [A @ B, dC @ B.t(), A.t() @ dC]
    if k in ("flash", "attention"):
        return _exact_attention(c, t)
    if k == "conv":
        return _exact_conv(c, t)
    X, dY = t["X"].double(), t["dY"].double()
    if c["op"] == "layer_norm":
        inv = 1.0 / torch.sqrt(X.var(1, unbiased=False, keepdim=True) + 1e-5)
        Y = (X - X.mean(1, keepdim=True)) * inv
        return [Y, inv * (dY - dY.mean(1, keepdim=True) - Y * (dY * Y).mean(1, keepdim=True))]
    if c["op"] == "softmax":
        Y = torch.softmax(X, dim=1)
        return [Y, Y * (dY - (dY * Y).sum(1, keepdim=True))]
    Y = torch.log_softmax(X, dim=1)
    return [Y, dY - Y.exp() * dY.sum(1, keepdim=True)]
