"""Performance cases of the Dense library, through its public entry points.

A case is one of seven kinds of call that programs make of the library:

  forward   one mounted Dense layer on device buffers
            (welvet_hip_dense_forward_device): decode, small-batch serving,
            prefill
  volume    the forward of a whole grid of Dense cells on device buffers
            (welvet_hip_volume_forward_device)
  swiglu    a mounted SwiGLU layer on device buffers
  train     several training steps of a grid on device buffers and then the
            checkpoint of every cell's native bytes into pinned host memory
  leaf      the one-shot NormalBP call of the reference's C ABI on host
            buffers (encode, forward, MSE, backward, SGD, decode)
  execute   a mounted layer called on host buffers (welvet_dense_execute)
  codec     a mounted store re-encoded from new host values, its native bytes
            and its decoded values read back

over the storage types that programs use in earnest (Float32, the two half
types, FP8, Int8 / Uint8, Int4, NF4, FP4).  Weights are drawn as values that
the storage type holds exactly, so exact() knows what the store decodes to
without this repository's codec.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "welvet.metal_amd"))
import pywelvet  # noqa: E402

DEV = "cuda:0"
DTYPES = ("float32", "float16", "bfloat16", "fp8e4m3", "fp8e5m2", "int8", "uint8", "int4", "nf4", "fp4")
TRAINED = DTYPES[:-1]  # FP4 stores have no scale: layers of its values (up to 6) do not train
FLOATS = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16,
          "fp8e4m3": torch.float8_e4m3fn, "fp8e5m2": torch.float8_e5m2}
# QLoRA's normal-float quantiles and the E2M1 values, as the library stores them
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
       -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
       0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
       0.7229568362236023, 1.0)
FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def listed():
    return [
        # one small layer, the reference's own first configuration: a launch's latency
        {"name": "volume_f32_512x512_b1", "kind": "volume", "dtype": "float32", "widths": "512-512",
         "batch": 1, "act": "tanh"},
        # single-token decode of an LLM's up projection in FP8 (the headline metric's shape)
        {"name": "forward_e4m3_4096x11008_b1", "kind": "forward", "dtype": "fp8e4m3", "inn": 4096, "out": 11008,
         "batch": 1, "act": "linear", "bias": False},
        # an MLP block decoding a handful of sequences in NF4
        {"name": "swiglu_nf4_4096x11008_b8", "kind": "swiglu", "dtype": "nf4", "inn": 4096, "inter": 11008,
         "batch": 8},
        # batched serving (the headline metric's batched shape)
        {"name": "forward_e4m3_4096x11008_b64", "kind": "forward", "dtype": "fp8e4m3", "inn": 4096, "out": 11008,
         "batch": 64, "act": "linear", "bias": False},
        # prefill of one prompt through an MLP block in FP4
        {"name": "swiglu_fp4_4096x11008_b512", "kind": "swiglu", "dtype": "fp4", "inn": 4096, "inter": 11008,
         "batch": 512},
        # a long prefill in half-precision weights, with bias and activation: the largest
        {"name": "forward_bf16_4096x11008_b2048", "kind": "forward", "dtype": "bfloat16", "inn": 4096, "out": 11008,
         "batch": 2048, "act": "silu", "bias": True},
        # a small network's layer whose sizes are nothing's multiple
        {"name": "forward_f32_1001x777_b100", "kind": "forward", "dtype": "float32", "inn": 1001, "out": 777,
         "batch": 100, "act": "relu", "bias": True},
        # training a two-layer MLP on a large batch in Int8
        {"name": "train_int8_2048_8192_2048_b256", "kind": "train", "dtype": "int8", "widths": "2048-8192-2048",
         "batch": 256, "steps": 8},
        # training a deep narrow volume on a small batch in FP8
        {"name": "train_e4m3_32x1024_b16", "kind": "train", "dtype": "fp8e4m3",
         "widths": "-".join(["1024"] * 33), "batch": 16, "steps": 8},
        # the reference's one-shot training leaf on host buffers
        {"name": "leaf_f16_1024x1024_b32", "kind": "leaf", "dtype": "float16", "inn": 1024, "out": 1024,
         "batch": 32, "act": "gelu"},
        # a drop-in caller of the reference's resident session: host buffers in and out
        {"name": "execute_int4_2048x5504_b16", "kind": "execute", "dtype": "int4", "inn": 2048, "out": 5504,
         "batch": 16, "act": "relu", "bias": True},
        # new values for a resident store, and its bytes and decoded values back
        {"name": "codec_nf4_2048x8192", "kind": "codec", "dtype": "nf4", "inn": 2048, "out": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A width: half of them multiples of 64, a quarter of 4, a quarter any."""
    n = _log(rng, lo, hi)
    r = rng.random()
    return max(lo, n // 64 * 64) if r < 0.5 else max(lo, n // 4 * 4) if r < 0.75 else n


def _aligned(case):
    """Whether every row of the case's layers starts on a 16-byte (sub-byte types: a 32-code) boundary."""
    bits = pywelvet.DTYPE_BITS[pywelvet.DTYPE[case["dtype"]]]
    per = 32 if bits <= 6 else 128 // bits
    return all(i % per == 0 for i, _ in _layers(case))


def draw(rng):
    kind = rng.choices(("forward", "volume", "swiglu", "train", "leaf", "execute", "codec"),
                       (40, 8, 12, 16, 8, 8, 8))[0]
    while True:
        c = {"kind": kind, "dtype": rng.choice(TRAINED if kind in ("train", "leaf") else DTYPES)}
        if kind == "forward":
            c.update(inn=_size(rng, 256, 11008), out=_size(rng, 256, 11008), batch=_log(rng, 1, 2048),
                     act=rng.choice(("linear", "relu", "silu", "gelu", "tanh")), bias=rng.random() < 0.5)
        elif kind == "swiglu":
            c.update(inn=_size(rng, 256, 4096), inter=_size(rng, 512, 11008), batch=_log(rng, 1, 1024))
        elif kind == "volume":
            c.update(widths="-".join(str(_size(rng, 256, 4096)) for _ in range(rng.randint(2, 6))),
                     batch=_log(rng, 1, 256), act=rng.choice(("relu", "tanh")))
        elif kind == "train":
            c.update(widths="-".join(str(_size(rng, 128, 2048)) for _ in range(rng.randint(3, 9))),
                     batch=_log(rng, 4, 512), steps=rng.randint(4, 8))
        elif kind == "codec":
            c.update(inn=_size(rng, 256, 4096), out=_size(rng, 256, 4096))
        else:
            c.update(inn=_size(rng, 128, 2048), out=_size(rng, 128, 2048), batch=_log(rng, 1, 256),
                     act=rng.choice(("relu", "gelu", "linear")))
            if kind == "execute":
                c.update(bias=rng.random() < 0.5)
        # no costlier than the largest listed case; rows that start off a
        # 16-byte boundary belong to small networks and small batches
        if work(c)["flops"] <= (1.8e11 if _aligned(c) else 1.5e9):
            return c


def _layers(case):
    """(in, out) of the case's Dense layers."""
    if case["kind"] == "swiglu":
        return [(case["inn"], case["inter"])] * 2 + [(case["inter"], case["inn"])]
    if "widths" in case:
        w = [int(v) for v in case["widths"].split("-")]
        return list(zip(w[:-1], w[1:]))
    return [(case["inn"], case["out"])]


def work(case):
    bits = pywelvet.DTYPE_BITS[pywelvet.DTYPE[case["dtype"]]]
    layers, b = _layers(case), case.get("batch", 0)
    n = sum(i * o for i, o in layers)
    packed = n * bits / 8
    first, last = layers[0][0], layers[-1][1]
    if case["kind"] == "codec":  # values in, bytes out, decoded values out; a compare and a divide each
        return {"bytes": 8 * n + packed, "flops": 2 * n}
    if case["kind"] == "train":
        # forward, dX of every layer but the first, dW; the weights read once
        # and written once each step, and written once more as the checkpoint
        i0, o0 = layers[0]
        s = case["steps"]
        return {"bytes": s * (2 * packed + 4 * b * (first + last)) + packed,
                "flops": s * (2 * b * (3 * n - i0 * o0) + 2 * n)}
    if case["kind"] == "leaf":  # W in, dW and W_after out; x and target in, pre, post and dX out
        return {"bytes": 12 * n + 4 * b * (2 * first + 3 * last), "flops": 6 * b * n + 2 * n}
    if case["kind"] == "swiglu":
        return {"bytes": packed + 4 * b * (2 * case["inn"] + case["inter"]), "flops": 2 * b * n}
    if case["kind"] == "volume":
        return {"bytes": packed + 4 * b * (first + last), "flops": 2 * b * n}
    return {"bytes": packed + 4 * b * (first + 2 * last), "flops": 2 * b * n}


# ----------------------------------------------------------------- inputs
def _weights(dtype, out, inn, std, gen):
    """f32 values [out][inn] about N(0, std) that `dtype` stores exactly: the
    scaled types on power-of-two steps with the extreme codes present, so the
    library's per-tensor scale is that step."""
    w = torch.randn((out, inn), generator=gen, device=DEV) * std
    if dtype == "float32":
        return w
    if dtype == "bfloat16":
        return w.to(torch.bfloat16).float()
    if dtype == "float16":  # the library's half encoder flushes subnormals
        w = w.half().float()
        return torch.where(w.abs() < 2.0 ** -14, 0.0, w)
    if dtype in ("fp8e4m3", "fp8e5m2"):  # a zero exponent field decodes to zero
        e4 = dtype == "fp8e4m3"
        w = w.to(torch.float8_e4m3fn if e4 else torch.float8_e5m2).float()
        return torch.where(w.abs() < (2.0 ** -6 if e4 else 2.0 ** -14), 0.0, w)
    if dtype == "fp4":  # unscaled E2M1: the values carry their own magnitude
        t = torch.tensor(FP4, device=DEV)
        v = torch.randint(0, 8, (out, inn), generator=gen, device=DEV)
        s = torch.randint(0, 2, (out, inn), generator=gen, device=DEV) * 2 - 1
        return torch.where(v == 0, 0.0, t[v] * s)
    flat = w.view(-1)
    if dtype == "nf4":
        scale = 2.0 ** round(math.log2(4 * std))
        t = torch.tensor(NF4, device=DEV)
        flat = t[torch.bucketize(flat / scale, (t[1:] + t[:-1]) / 2)] * scale
        flat[0] = scale
    elif dtype == "uint8":
        step = 2.0 ** round(math.log2(8 * std / 255))
        flat = (torch.round(flat / step) + 128).clamp(0, 255)
        flat[0], flat[-1] = 0, 255
        flat = (flat - 128) * step
    else:
        top = 127 if dtype == "int8" else 7
        step = 2.0 ** round(math.log2(4 * std / top))
        flat = torch.round(flat / step).clamp(-top, top)
        flat[0] = top
        flat = torch.where(flat == 0, 0.0, flat * step)
    return flat.view(out, inn)


def _inputs(case, seed):
    """Every input of a case from the seed: weights per layer, bias, x, target."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    d = case["dtype"]
    layers = _layers(case)
    deep = case["kind"] in ("train", "volume")
    std = [math.sqrt(2.0 / i) if deep else 0.05 if d.startswith("fp8") else 0.02 for i, _ in layers]
    W = [_weights(d, o, i, s, gen) for (i, o), s in zip(layers, std)]
    first, last = layers[0][0], layers[-1][1]
    b = case.get("batch", 1)
    x = torch.randn((b, first), generator=gen, device=DEV)
    if d == "fp4":  # the unscaled weights are near 3: activations of a scaled program
        x = x * 0.01
    t = torch.randn((b, last), generator=gen, device=DEV) * 4
    bias = torch.randn(last, generator=gen, device=DEV, dtype=torch.float64) * 0.1 if case.get("bias") else None
    return W, bias, x, t


def _rate(case):
    """SGD rate, of an MSE over batch * out values: deep networks take small steps."""
    layers = len(_layers(case))
    return 0.5 if layers <= 2 else 0.5 / layers ** 2


class _Layer(pywelvet.Session):
    """pywelvet.Session mounted from device memory."""

    def __init__(self, W, batch, act, dtype, bias):
        self.h = None
        self.out, self.inn = W.shape
        self.batch, self.dtype = batch, dtype
        b = None if bias is None else bias.cpu().numpy()
        h = ctypes.c_void_p()
        torch.cuda.synchronize()
        pywelvet.check(pywelvet.lib().welvet_hip_dense_mount_device(
            batch, self.inn, self.out, act, dtype, ctypes.c_void_p(W.data_ptr()),
            None if b is None else b.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 0 if b is None else b.size,
            ctypes.byref(h)))
        self.h = h


class _Swiglu(pywelvet.SwigluSession):
    def __del__(self):
        self.close()


def _acts(case):
    """Activation of each layer: a grid's hidden ones are ReLU (or the case's), its last linear."""
    n = len(_layers(case))
    if case["kind"] == "train":
        return ["relu"] * (n - 1) + ["linear"]
    if case["kind"] == "volume":
        return [case["act"]] * (n if n == 1 else n - 1) + ([] if n == 1 else ["linear"])
    return [case.get("act", "linear")] * n


def _grid(case, W):
    layers = len(W)
    # 32 cells as the deep configuration lays them out, else one cell a layer
    dims = (2, 2, 2, 4) if layers == 32 else (1, 1, 1, layers)
    g = pywelvet.Grid(*dims, case["batch"])
    coords = [(z, y, x, k) for z in range(dims[0]) for y in range(dims[1]) for x in range(dims[2])
              for k in range(dims[3])]
    for at, w, a in zip(coords, W, _acts(case)):
        g.bind_dense(at, w.cpu().numpy(), act=pywelvet.ACT[a], dtype=pywelvet.DTYPE[case["dtype"]])
    return g, coords


def prepare(case, seed):
    W, bias, x, t = _inputs(case, seed)
    kind, dt = case["kind"], pywelvet.DTYPE[case["dtype"]]
    act = pywelvet.ACT[case.get("act", "linear")]
    s = {"kind": kind, "case": case, "stream": torch.cuda.current_stream().cuda_stream}
    b = case.get("batch", 1)
    last = _layers(case)[-1][1]
    if kind == "forward":
        s.update(h=_Layer(W[0], b, act, dt, bias), x=x, pre=torch.zeros((b, last), device=DEV),
                 post=torch.zeros((b, last), device=DEV))
    elif kind == "swiglu":
        torch.cuda.synchronize()
        s.update(h=_Swiglu(*(w.cpu().numpy() for w in W), b, dt), x=x,
                 pre=torch.zeros((b, case["inter"]), device=DEV), post=torch.zeros((b, last), device=DEV))
    elif kind == "volume":
        g, _ = _grid(case, W)
        s.update(h=g, x=x, y=torch.zeros((b, last), device=DEV))
    elif kind == "train":
        g, coords = _grid(case, W)
        bits = pywelvet.DTYPE_BITS[dt]
        room = [torch.zeros((i * o * bits + 7) // 8 + 4, dtype=torch.uint8).pin_memory() for i, o in _layers(case)]
        s.update(h=g, x=x, t=t, coords=coords, room=room, lr=_rate(case))
    elif kind == "leaf":
        s.update(W=W[0].cpu().numpy(), x=x.cpu().numpy(), t=t.cpu().numpy(), act=act, dt=dt, lr=_rate(case))
    elif kind == "execute":
        s.update(h=_Layer(W[0], b, act, dt, bias), x=x.cpu().numpy())
    else:
        new = _inputs(case, seed + 7919)[0][0]
        s.update(h=_Layer(W[0], 1, -1, dt, None), values=new.cpu().numpy())
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "forward":
        s["h"].forward_device(s["x"].data_ptr(), s["pre"].data_ptr(), s["post"].data_ptr(), s["stream"])
        return {"pre": s["pre"], "post": s["post"]}
    if kind == "swiglu":
        pywelvet.check(s["h"].forward_device(s["x"].data_ptr(), s["pre"].data_ptr(), s["post"].data_ptr(),
                                             s["stream"]))
        return {"pre": s["pre"], "post": s["post"]}
    if kind == "volume":
        x, y = s["x"], s["y"]
        pywelvet.check(pywelvet.lib().welvet_hip_volume_forward_device(
            s["h"].h, x.data_ptr(), x.shape[1], y.data_ptr(), y.shape[1], s["stream"]))
        return {"y": y}
    if kind == "train":
        return _train(s)
    if kind == "leaf":
        return pywelvet.normalbp(s["W"], s["x"], s["t"], 1, s["lr"], act=s["act"], dtype=s["dt"])
    if kind == "execute":
        pre, post = s["h"].execute(s["x"])
        return {"pre": pre, "post": post}
    s["h"].repack(s["values"])
    raw, scale = s["h"].native()
    return {"native": raw, "scale": scale, "values": s["h"].export_f32()}


def _train(s):
    lib, g, x, t = pywelvet.lib(), s["h"], s["x"], s["t"]
    loss, losses = ctypes.c_double(), []
    for _ in range(s["case"]["steps"]):
        pywelvet.check(lib.welvet_hip_volume_train_step_device(
            g.h, x.data_ptr(), x.shape[1], t.data_ptr(), t.shape[1], s["lr"], ctypes.byref(loss), s["stream"]))
        losses.append(loss.value)
    n, scale, saved = ctypes.c_size_t(), ctypes.c_float(), []
    kind = FLOATS.get(s["case"]["dtype"])
    for at, room in zip(s["coords"], s["room"]):
        pywelvet.check(lib.welvet_hip_grid_native(
            g.h, *at, ctypes.cast(room.data_ptr(), ctypes.POINTER(ctypes.c_uint8)), room.numel(), ctypes.byref(n),
            ctypes.byref(scale)))
        raw = room[:n.value]
        saved.append(raw if kind is None else raw.view(kind))
    return {"loss": losses, "weights": saved}


# ------------------------------------------------------------ expectations
def tolerance(case):
    """Four times what two routes of one product differ by (fp32 sums of up to
    11008 products in other orders and splits: rel 2e-6, max 2e-5).  A weight
    whose update falls next to a rounding boundary is stored one code off
    after such a difference: few of a leaf's decoded W_after, and more over
    the steps of a training run, where each one moves the next step (two
    routes after 16 steps: rel 2.2e-3, 0.4% of integer codes)."""
    if case["kind"] == "codec":
        return "exact"
    if case["kind"] == "train" and case["dtype"] != "float32":
        return {"rel": 1e-2, "max": 0.99, "differ": 1e-2}
    if case["kind"] == "leaf" and case["dtype"] != "float32":
        return {"rel": 1e-3, "max": 0.9}
    return {"rel": 8e-6, "max": 1e-4}


def _act(v, name):
    if name == "relu":
        return v.clamp(min=0)
    if name == "silu":
        return v * torch.sigmoid(v)
    if name == "gelu":
        return 0.5 * v * (1 + torch.tanh(math.sqrt(2 / math.pi) * (v + 0.044715 * v ** 3)))
    return torch.tanh(v) if name == "tanh" else v


def exact(case, seed):
    kind = case["kind"]
    if kind == "codec":  # bytes and table values: bit for bit, nothing to compute
        return None
    W, bias, x, t = _inputs(case, seed)
    W = [w.double() for w in W]
    x, t = x.double(), t.double()
    if kind in ("forward", "execute"):
        pre = x @ W[0].t()
        if bias is not None:
            pre = pre + bias
        r = {"pre": pre, "post": _act(pre, case["act"])}
        return r if kind == "forward" else {k: v.cpu().numpy() for k, v in r.items()}
    if kind == "swiglu":
        h = _act(x @ W[0].t(), "silu") * (x @ W[1].t())
        return {"pre": h, "post": h @ W[2].t()}
    acts = _acts(case)
    if kind == "volume":
        for w, a in zip(W, acts):
            x = _act(x @ w.t(), a)
        return {"y": x}
    if kind == "train":
        # the first step's loss (the later ones follow re-encoded weights);
        # a Float32 network's weights are not re-encoded: all of its losses
        # and its weights
        known = case["dtype"] == "float32"
        losses = []
        for _ in range(case["steps"] if known else 1):
            ins, v = [], x
            for w, a in zip(W, acts):
                ins.append(v)
                v = _act(v @ w.t(), a)
            losses.append(float(((v - t) ** 2).mean()))
            if not known:
                break
            g = 2 * (v - t) / t.numel()
            for k in range(len(W) - 1, -1, -1):
                below = g @ W[k]
                W[k] = W[k] - _rate(case) * (g.t() @ ins[k])
                g = below * (ins[k] > 0) if k else None
        losses += [None] * (case["steps"] - len(losses))
        return {"loss": losses, "weights": [w.view(-1).cpu() if known else None for w in W]}
    w = W[0].requires_grad_()
    x.requires_grad_()
    pre = x @ w.t()
    post = _act(pre, case["act"])
    loss = ((post - t) ** 2).mean()
    loss.backward()
    r = {"pre": pre, "post": post, "dX": x.grad, "dW": w.grad,
         "W_after": w - _rate(case) * w.grad if case["dtype"] == "float32" else None}
    r = {k: None if v is None else v.detach().cpu().numpy() for k, v in r.items()}
    r["loss"] = float(loss)
    return r
