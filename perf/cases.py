"""The work that a user of this layer has it do, as cases that can be measured.

A case names a layer (widths, experts, data type, router mode), a batch and what is done with it:
  forward   one layer forward (MoELayer.forward): serving, decode and prefill
  block     the FFN half of a transformer block (MoELayer.forward_block): out = x + layer(rmsnorm(x))
  grads     forward and backward in training mode, then every parameter gradient into buffers of the caller: one
            worker of a data-parallel job, which all-reduces them and steps its own optimiser
  adamw     one training step of the block form: forward, backward, clipping by the global norm, AdamW, and the updated
            weights into buffers of the caller (what it checkpoints or sends to its serving replicas)
  sgd       one training step of a layer without an updater: forward, backward, w -= lr * gradient, the updated weights
            into buffers of the caller
Weights, tokens and output gradients are drawn on the device by the library's own seeded generator with the standard
deviations of omega-ai_amd/configs.py; `zipf` is the exponent of the gate bias that makes some experts hot and others
empty.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

P = importlib.import_module("omega-ai_amd")
L = importlib.import_module("omega-ai_amd._lib")
C = P.configs

STREAM_DOUT = 900      # generator stream of the output gradient
DOUT_STD = 1e-3        # per element, the order of a mean loss's gradient
CLIP_NORM = 1.0
ADAMW_LR = 1e-6        # a fine-tuning step: thousands of passes leave the weights what they are
SGD_LR = 1e-3


def _case(name, do, T, d, E, K, H, Es=0, renorm=True, dtype="bf16", zipf=0.0, router="exact"):
    return dict(name=name, do=do, T=T, d=d, E=E, K=K, H=H, Es=Es, renorm=renorm, dtype=dtype, zipf=zipf, router=router)


def listed():
    mixtral = dict(d=4096, E=8, K=2, H=14336)
    fine = dict(d=2048, E=64, K=6, H=1408, Es=2, renorm=False)
    return [
        # the smallest call: the fp32 configuration that the reference's users know (latency and launches)
        _case("tiny_f32", "forward", T=256, d=128, E=8, K=2, H=256, dtype="f32"),
        # one user's decode step
        _case("decode_one", "forward", T=1, **mixtral),
        # a decode step of 64 sequences
        _case("decode_batch", "forward", T=64, **mixtral),
        # the same with many small experts: most of them get a few rows
        _case("decode_finegrained", "forward", T=48, **fine),
        # a chunk of a prompt, no multiple of anything, through the block form
        _case("prefill_chunk", "block", T=777, **mixtral),
        # prompts of 8 x 512 tokens
        _case("prefill_mixtral", "forward", T=4096, **mixtral),
        # one longer prompt, gate sums in the fast mode
        _case("prefill_fast_router", "forward", T=1500, router="fast", **fine),
        # many small experts and shared ones, a large batch
        _case("prefill_finegrained", "forward", T=8192, **fine),
        # the largest batch, hot and empty experts
        _case("prefill_skewed", "forward", T=16384, d=2048, E=128, K=8, H=768, zipf=1.2),
        # fp32 training, the data type of the reference
        _case("train_f32", "sgd", T=4096, d=1024, E=8, K=2, H=3584, dtype="f32"),
        # bf16 training with the updater, a ragged batch
        _case("train_adamw", "adamw", T=3000, d=2048, E=16, K=4, H=1408, Es=1),
        # data-parallel bf16 training at the widths of the prefill case
        _case("train_grads", "grads", T=4096, **mixtral),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cost(case):
    """Rough seconds of a pass, to keep drawn cases within the largest listed one."""
    w = work(case)
    rate = (2e13 if case["do"] == "sgd" else 6e13) if case["dtype"] == "f32" else 8e14
    return w["flops"] / rate + w["bytes"] / 3e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        do = rng.choices(["forward", "block", "grads", "adamw", "sgd"], [55, 15, 10, 10, 10])[0]
        f32 = do == "sgd" or (do == "forward" and rng.random() < 0.2)
        E = _spread(rng, 2, 16) if f32 or do == "grads" else _spread(rng, 4, 128)
        c = dict(do=do, E=E, K=rng.randint(1, min(8, E)), renorm=rng.random() < 0.7, dtype="f32" if f32 else "bf16",
                 Es=rng.choice([0, 0, 0, 1, 2]), zipf=1.2 if E >= 16 and rng.random() < 0.25 else 0.0,
                 router="fast" if rng.random() < 0.15 else "exact")
        if f32:
            c.update(T=_spread(rng, 1, 4096), d=_spread(rng, 64, 1024), H=_spread(rng, 64, 3584))
        else:  # bf16 layers take widths d % 256 == 0 and H % 128 == 0
            c.update(T=_spread(rng, 1 if do in ("forward", "block") else 32, 16384 if do in ("forward", "block") else 4096),
                     d=256 * _spread(rng, 4, 16), H=128 * _spread(rng, 4, 112))
        n = 3 * c["d"] * c["H"] * (c["E"] + c["Es"])
        if n <= (4e8 if do == "adamw" else 1.45e9) and c["T"] * c["K"] * max(c["d"], c["H"]) <= 1e9 and _cost(c) <= most:
            return c


_ctx = None


def _context():
    """One context (device and stream) for the program, as a user's program has."""
    global _ctx
    if _ctx is None:
        _ctx = P.Context(0)
    return _ctx


class _Held:
    """A layer and the buffers of its caller, given back with the last tensor that looks at them."""

    def __init__(self, layer):
        self.layer, self.buffers = layer, []

    def buffer(self, shape, dtype):
        b = P.DeviceBuffer(self.layer.ctx, shape, dtype)
        self.buffers.append(b)
        return b

    def __del__(self):
        for b in self.buffers:
            b.free()
        self.layer.close()


class _Memory:
    def __init__(self, held, buf):
        self.held = held
        self.__cuda_array_interface__ = {"version": 2, "shape": tuple(buf.shape), "data": (buf.ptr.value, False),
                                         "typestr": "<i2" if buf.dtype == "bf16" else "<f4", "strides": None}


def _tensor(held, buf):
    """The device buffer as a tensor, without a copy."""
    t = torch.as_tensor(_Memory(held, buf), device="cuda")
    return t.view(torch.bfloat16) if buf.dtype == "bf16" else t


def prepare(case, seed):
    cfg = C.MoEConfig("case", T=case["T"], d=case["d"], E=case["E"], K=case["K"], H=case["H"], Es=case["Es"],
                      renorm=case["renorm"], dtype=case["dtype"], zipf_bias=case["zipf"])
    layer = P.MoELayer(cfg.d, cfg.H, cfg.E, cfg.K, renorm=cfg.renorm, nShared=cfg.Es, bias=cfg.has_gate_bias, ctx=_context(),
                       dtype=cfg.dtype, router_mode=case["router"], T_max=cfg.T)
    held = _Held(layer)
    layer.init_synthetic(seed, C, cfg)
    x = held.buffer((cfg.T, cfg.d), cfg.dtype)
    x.fill_normal(seed, C.STREAM_X, C.tensor_std(cfg, "x"))
    s = {"do": case["do"], "held": held, "layer": layer, "x": x, "step": 0, "tensors": {}}
    if case["do"] in ("grads", "adamw", "sgd"):
        layer.set_training(True)
        s["dout"] = held.buffer((cfg.T, cfg.d), cfg.dtype)
        s["dout"].fill_normal(seed, STREAM_DOUT, DOUT_STD)
        # where the caller takes gradients (fp32) or updated weights (the layer's type), the experts' one after the other
        dt, G = "f32" if case["do"] == "grads" else cfg.dtype, cfg.E + cfg.Es
        s["params"] = {"Wg": held.buffer((cfg.E, cfg.d), dt), "W1": held.buffer((G, cfg.H, cfg.d), dt),
                       "W3": held.buffer((G, cfg.H, cfg.d), dt), "W2": held.buffer((G, cfg.d, cfg.H), dt)}
    layer.ctx.sync()
    return s


def _fetch(s, what):
    """Every parameter's gradient or weight into the caller's buffers (device to device)."""
    layer, lib = s["layer"], s["layer"].lib
    get = lib.omega_moe_get_grad if what == "grads" else lib.omega_moe_get_weights
    for name, which in (("Wg", L.W_GATE), ("W1", L.W_W1), ("W3", L.W_W3), ("W2", L.W_W2)):
        buf = s["params"][name]
        n = 1 if name == "Wg" else buf.shape[0]
        for g in range(n):
            layer.ctx.check(get(layer.handle, which, g, ctypes.c_void_p(buf.ptr.value + g * (buf.nbytes // n)), 1))


def run(s):
    layer, do = s["layer"], s["do"]
    got = {"out": layer.forward_block(s["x"]) if do in ("block", "adamw") else layer.forward(s["x"])}
    if do in ("grads", "sgd"):
        got["dx"] = layer.back(s["dout"])
    elif do == "adamw":
        got["dx"] = layer.back_block(s["dout"])
        layer.clipGradNorm(CLIP_NORM)
        s["step"] += 1
        layer.updateAdamW(ADAMW_LR, s["step"])
    if do == "sgd":
        layer.update(SGD_LR)
    if do in ("grads", "adamw", "sgd"):
        _fetch(s, do)
        got.update(s["params"])
    views = s["tensors"]
    for name, buf in got.items():
        if name not in views:
            views[name] = _tensor(s["held"], buf)
    return dict(views)


def _experts_used(case):
    """Routed experts that get at least one token: from a sample of gate logits with the configuration's spread."""
    T, E, K = case["T"], case["E"], case["K"]
    r = np.random.default_rng(1)
    z = r.normal(0.0, 0.02 * math.sqrt(case["d"]), (min(T, 4096), E))
    if case["zipf"]:
        p = np.arange(1, E + 1) ** -case["zipf"]
        z = z + 2 * np.log(p / p.sum())
    return len(np.unique(np.argpartition(-z, K - 1, axis=1)[:, :K]))


def work(case):
    T, d, H, E, K, Es = (case[k] for k in ("T", "d", "H", "E", "K", "Es"))
    b = 2 if case["dtype"] == "bf16" else 4
    rows = T * (K + Es)
    n_used, n_all = 3 * d * H * (_experts_used(case) + Es), 3 * d * H * (E + Es)
    gate = E * d
    if case["do"] in ("forward", "block"):
        # the tokens in and out, the weights of the experts that are used
        return {"bytes": 2 * T * d * b + (n_used + gate) * b, "flops": 6 * d * H * rows + 2 * T * gate}
    # tokens and output gradient in, output and input gradient out; forward once, input and weight gradients
    r = {"bytes": 4 * T * d * b + (n_used + gate) * b, "flops": 18 * d * H * rows + 6 * T * gate}
    if case["do"] == "grads":
        r["bytes"] += (n_all + gate) * 4      # the gradients
    elif case["do"] == "adamw":
        # weights out; master weights and two moments in and out
        r["bytes"] += (n_all + gate) * (b + 24)
    else:
        r["bytes"] += (n_used + gate) * b     # the updated weights
    return r


def tolerance(case):
    # About four times what the path differs from float64 and from fp32 sums in another order with the same rounding
    # points: fp32 rel 1.4e-6, max 8.7e-6; bf16 rel 4.3e-4 (the output), max 1.5e-2 (a gradient element one of whose
    # bf16 factors rounds the other way); fast against exact gate sums rel 1.4e-5.
    if case["dtype"] == "f32":
        return {"rel": 6e-6, "max": 4e-5}
    return {"rel": 2e-3, "max": 6e-2}
