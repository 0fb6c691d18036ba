"""What this library is timed on: the calls that a model runtime makes through the public entry points, from one token of
one narrow layer to the prefill and the training step of wide ones.

Every case is a dict with a "kind"; the kinds are the ways a runtime uses the library:

* linear   one device-resident call, `linear_a8` (per-token int8 activations) or `linear_float`;
* layer    the projections of one decoder layer in a decoder's order: q,k,v behind the attention norm as one group, o with
           its residual add, gate,up behind the FFN norm as one group, down with its residual add;
* group    one grouped launch over the resident layers of a stack (continuous batching, given inputs);
* forward  `TernaryLinear.forward` on host slices, what a host-side model calls per layer;
* salt     block-scale additive planes (`linear_salt`), decode and prompt;
* salt_v2  the exact forward over a SALT V2 codec payload;
* vjp      the training step's three gradients of one layer (`projected_vjp`).

Sizes are those of the benchmark's configurations (hidden 2560 / 5120, FFN 6912 / 17408, K=2048 N=8192) and ragged ones
between and around them.
"""
import ctypes
import math

import numpy as np
import torch

import tritium_amd as T

MAX_TOKENS = 4096
MAX_OPS = 2.2e12           # 2*M*N*K*planes of the largest listed case
ZEROS = (0.4, 0.7, 0.85, 0.85)   # share of zero trits, plane by plane
EPS = 1e-5

_DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "bf16": 2}


def listed():
    return [
        # one token of a square projection: the smallest call a decoder makes, all latency
        {"name": "token", "kind": "linear", "contract": "a8", "m": 1, "n": 2560, "k": 2560, "planes": 1, "act": "bf16", "out": "bf16"},
        # one layer of interactive decoding: four dependent calls
        {"name": "layer 1", "kind": "layer", "m": 1, "hidden": 2560, "kv": 640, "ffn": 6912},
        # the same layer with a batch of sequences in flight
        {"name": "layer 32", "kind": "layer", "m": 32, "hidden": 2560, "kv": 640, "ffn": 6912},
        # a stack of two-plane layers on float activations, small batch: weights stream from memory
        {"name": "stack float 8", "kind": "group", "contract": "float", "m": 8, "n": 8192, "k": 2048, "planes": 2, "copies": 48,
         "act": "bf16", "out": "f32"},
        # continuous batching of 64 sequences on wide three-plane layers: up projections of a stack
        {"name": "stack a8 64", "kind": "group", "contract": "a8", "m": 64, "n": 17408, "k": 5120, "planes": 3, "copies": 8,
         "act": "bf16", "out": "bf16"},
        # prefill of 2048 tokens through one up projection
        {"name": "prefill 2048", "kind": "linear", "contract": "a8", "m": 2048, "n": 6912, "k": 2560, "planes": 1, "act": "bf16", "out": "bf16"},
        # a long prompt on a wide three-plane layer: the largest product
        {"name": "prefill 4096", "kind": "linear", "contract": "a8", "m": 4096, "n": 17408, "k": 5120, "planes": 3, "act": "bf16", "out": "bf16"},
        # a short prompt on float activations, nothing a multiple of anything
        {"name": "prompt float", "kind": "linear", "contract": "float", "m": 333, "n": 5003, "k": 2050, "planes": 2, "act": "f32", "out": "f32"},
        # a host-side model: slices in, slices out
        {"name": "forward 48", "kind": "forward", "m": 48, "n": 6912, "k": 2560},
        # a prompt through block-scale planes
        {"name": "salt 128", "kind": "salt", "m": 128, "n": 8192, "k": 2048, "planes": 2, "act": "bf16", "out": "f32"},
        # a small batch through a codec payload
        {"name": "salt v2 8", "kind": "salt_v2", "m": 8, "n": 4096, "k": 4096, "codec": "B3", "scale_group": 128},
        # the backward step of the 2048-token prefill layer
        {"name": "vjp 2048", "kind": "vjp", "m": 2048, "n": 6912, "k": 2560},
    ]


# ---- cases of the same ranges ------------------------------------------------------------------

def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi):
    """A layer width: mostly whole blocks of 256 or 128 as models have them, sometimes ragged."""
    step = rng.choice((256, 256, 256, 128, 128, 64, 1))
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("linear",) * 5 + ("layer", "layer", "group", "group", "forward", "salt", "salt_v2", "vjp"))
    if kind == "linear":
        c = {"kind": kind, "contract": rng.choice(("a8", "a8", "float")), "m": _log(rng, 1, MAX_TOKENS), "n": _width(rng, 512, 17408),
             "k": _width(rng, 512, 17408), "planes": rng.choice((1, 1, 2, 3)), "act": rng.choice(("bf16", "bf16", "f32"))}
        c["out"] = c["act"]
        rows = 4 if c["contract"] == "float" else 1   # a float token costs about four int8 ones
        while 2.0 * c["m"] * c["n"] * c["k"] * c["planes"] * rows > MAX_OPS:
            c["m"] = (c["m"] + 1) // 2
        return c
    if kind == "layer":
        hidden = max(1024, _log(rng, 1024, 5120) // 128 * 128)
        return {"kind": kind, "m": _log(rng, 1, 64), "hidden": hidden, "kv": hidden // 4 // 64 * 64,
                "ffn": int(hidden * rng.uniform(2.5, 3.5)) // 64 * 64}
    if kind == "group":
        c = {"kind": kind, "contract": rng.choice(("a8", "a8", "float")), "n": _width(rng, 1024, 17408), "k": _width(rng, 1024, 6912),
             "planes": rng.choice((1, 2, 3)), "act": "bf16", "out": rng.choice(("bf16", "f32"))}
        c["m"] = _log(rng, 1, 64 if c["contract"] == "a8" else 16)
        per = c["planes"] * c["n"] * c["k"] / 4
        c["copies"] = max(2, min(48, round(rng.uniform(1.5e8, 4e8) / per)))   # more weights than the last-level cache holds, where 48 layers do
        return c
    if kind == "forward":
        return {"kind": kind, "m": _log(rng, 1, 256), "n": _width(rng, 512, 8192), "k": _width(rng, 512, 8192)}
    if kind == "salt":
        return {"kind": kind, "m": _log(rng, 1, 1024), "n": _width(rng, 1024, 8192), "k": _width(rng, 1024, 8192), "planes": rng.choice((1, 2, 3)),
                "act": rng.choice(("bf16", "f32")), "out": "f32"}
    if kind == "salt_v2":
        return {"kind": kind, "m": _log(rng, 1, 64), "n": 2 * _log(rng, 256, 4096), "k": max(512, _log(rng, 512, 4096) // 128 * 128),
                "codec": rng.choice(("D2", "B3", "S34")), "scale_group": rng.choice((64, 128))}
    return {"kind": kind, "m": _log(rng, 64, 2048), "n": _width(rng, 512, 6912), "k": _width(rng, 512, 2560)}


# ---- inputs ------------------------------------------------------------------------------------

_backend = None


def backend():
    global _backend
    if _backend is None:
        _backend = T.Mi355xBackend(torch.cuda.current_device())
    return _backend


class Buffer:
    """A torch tensor and the library's view of it."""

    def __init__(self, tensor):
        self.tensor = tensor
        dt = {torch.float32: "f32", torch.bfloat16: "bf16", torch.int8: "i8"}[tensor.dtype]
        self.array = T.DeviceArray(backend(), ctypes.c_void_p(tensor.data_ptr()), tensor.numel(), T.backend.DTYPES[dt])


class Source:
    """Random inputs of one seed, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)

    def normal(self, m, k, dtype):
        return Buffer(torch.randn(m, k, generator=self.gen, device="cuda").to(_DTYPE[dtype]))

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def codes(self, n, k, p_zero):
        """[n,k] trit codes 0..2 (trit + 1), uint8."""
        u = torch.rand(n, k, generator=self.gen, device="cuda")
        half = (1.0 - p_zero) / 2
        return (u > half).to(torch.uint8) + (u > half + p_zero).to(torch.uint8)

    def tq2_rows(self, n, k, p_zero, block_scales=None):
        """Packed TQ2_0 rows as a model file holds them: 64 code bytes and an f16 scale per 256 trits."""
        nb = (k + 255) // 256
        c = torch.full((n, nb * 256), 1, dtype=torch.uint8, device="cuda")
        c[:, :k] = self.codes(n, k, p_zero)
        c = c.view(n, nb, 2, 4, 32)
        packed = torch.empty(n, nb, 66, dtype=torch.uint8, device="cuda")
        packed[:, :, :64] = (c[:, :, :, 0] | c[:, :, :, 1] << 2 | c[:, :, :, 2] << 4 | c[:, :, :, 3] << 6).reshape(n, nb, 64)
        scale = torch.ones(n, nb, device="cuda") if block_scales is None else block_scales
        packed[:, :, 64:] = scale.half().view(torch.uint8).view(n, nb, 2)
        return packed.cpu().numpy()

    def linear(self, n, k, planes):
        """A resident additive-plane layer with U(0.01, 0.1) channel scales."""
        bufs = [backend().upload_weights(self.tq2_rows(n, k, ZEROS[p]), T.GemmShape(0, n, k), T.TernaryFormat.Tq2_0) for p in range(planes)]
        scales = [Buffer(self.uniform(0.01, 0.1, n)) for _ in range(planes)]
        layer = T.Linear(backend(), bufs, [s.array for s in scales])
        layer.keep = scales
        return layer


class State:
    """What a runtime keeps between calls; groups are given back with it."""

    def __init__(self, case):
        self.case, self.groups = case, []

    def group(self, *args, **kw):
        g = backend().group(*args, **kw)
        self.groups.append(g)
        return g

    def __del__(self):
        for g in self.groups:
            g.destroy()


def _empty(m, n, dtype):
    return Buffer(torch.empty(m, n, dtype=_DTYPE[dtype], device="cuda"))


def prepare(case, seed):
    src, s, be = Source(seed), State(case), backend()
    kind, m = case["kind"], case["m"]
    if kind == "layer":
        h, kv, f = case["hidden"], case["kv"], case["ffn"]
        widths = {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (f, h), "up": (f, h), "down": (h, f)}
        s.lin = {name: src.linear(n, k, 1) for name, (n, k) in widths.items()}
        s.norms = [Buffer(src.uniform(0.5, 1.5, h)) for _ in range(2)]
        # the residual stream, the attention's output and the gated FFN activation come from the runtime's other kernels
        s.x, s.attended, s.gated = src.normal(m, h, "bf16"), src.normal(m, h, "bf16"), src.normal(m, f, "bf16")
        s.out = {name: _empty(m, n, "bf16") for name, (n, _) in widths.items()}
        s.qkv = s.group([(s.lin[p], s.x.array, m, s.out[p].array) for p in "qkv"], 1, "bf16", "bf16",
                        norms=[(s.norms[0].array, EPS, False)] * 3)
        s.gate_up = s.group([(s.lin[p], s.out["o"].array, m, s.out[p].array) for p in ("gate", "up")], 1, "bf16", "bf16",
                            norms=[(s.norms[1].array, EPS, False)] * 2)
        torch.cuda.synchronize()
        return s
    n, k = case["n"], case["k"]
    if kind == "linear":
        s.layer, s.x, s.out = src.linear(n, k, case["planes"]), src.normal(m, k, case["act"]), _empty(m, n, case["out"])
    elif kind == "group":
        s.layers = [src.linear(n, k, case["planes"]) for _ in range(case["copies"])]
        s.x = src.normal(m, k, case["act"])
        s.outs = [_empty(m, n, case["out"]) for _ in s.layers]
        s.members = s.group([(layer, s.x.array, m, o.array) for layer, o in zip(s.layers, s.outs)], int(case["contract"] == "a8"),
                            case["act"], case["out"])
    elif kind == "forward":
        trits = (src.codes(n, k, ZEROS[0]).to(torch.int8) - 1).cpu().numpy()
        s.layer = T.TernaryLinear.with_row_scales(be, trits, n, k, src.uniform(0.01, 0.1, n).cpu().numpy())
        s.x = torch.randn(m, k, generator=src.gen, device="cuda").cpu().numpy()
        s.out = np.zeros((m, n), np.float32)
    elif kind == "salt":
        nb = (k + 255) // 256
        s.planes = [be.upload_weights_scaled(src.tq2_rows(n, k, ZEROS[p], src.uniform(0.02, 1.0, n, nb) * 0.5 ** p), T.GemmShape(0, n, k))
                    for p in range(case["planes"])]
        s.x, s.out = src.normal(m, k, case["act"]), _empty(m, n, case["out"])
    elif kind == "salt_v2":
        s.matrix = _salt_v2(src, case)
        s.x, s.out = src.normal(m, k, "f32"), _empty(m, n, "f32")
    else:
        s.layer = src.linear(n, k, 1)
        s.x, s.up = src.normal(m, k, "f32"), Buffer(torch.randn(m, n, generator=src.gen, device="cuda") / math.sqrt(n))
        s.grad_x, s.grad_w, s.grad_b = _empty(m, k, "f32"), _empty(n, k, "f32"), _empty(1, n, "f32")
    torch.cuda.synchronize()
    return s


def _salt_v2(src, case):
    """Two planes in every allocation tile of 256 coefficients, one f16 scale per plane and scale group."""
    n, k, group = case["n"], case["k"], case["scale_group"]
    tiles = n * k // 256
    codec = {"D2": T.SALT_V2_D2, "B3": T.SALT_V2_B3, "S34": T.SALT_V2_S34}[case["codec"]]
    planes = []
    for p in range(2):
        if case["codec"] == "S34":   # four coefficients with one zero in five bits: every bit pattern is one
            planes.append(torch.randint(0, 256, (tiles, 40), generator=src.gen, device="cuda", dtype=torch.uint8))
            continue
        c = src.codes(tiles, 256, ZEROS[p])
        if case["codec"] == "D2":
            c = c.view(tiles, 64, 4)
            planes.append(c[:, :, 0] | c[:, :, 1] << 2 | c[:, :, 2] << 4 | c[:, :, 3] << 6)
        else:                        # five trits to a byte, the first the least significant; the last byte is filled with zero trits
            c = torch.cat([c, torch.ones(tiles, 4, dtype=torch.uint8, device="cuda")], 1).view(tiles, 52, 5)
            planes.append(c[:, :, 0] + 3 * c[:, :, 1] + 9 * c[:, :, 2] + 27 * c[:, :, 3] + 81 * c[:, :, 4])
    payload = torch.stack(planes, 1).reshape(-1).cpu().numpy()
    scales = src.uniform(0.02, 1.0, tiles * 2 * (256 // group)).half().cpu().numpy().view(np.uint16)
    return backend().salt_v2_upload(codec, group, payload, scales, np.full(tiles, 2, np.uint8), n, k)


# ---- one pass ----------------------------------------------------------------------------------

def run(s):
    c, be = s.case, backend()
    kind, m = c["kind"], c["m"]
    if kind == "linear":
        (be.linear_a8 if c["contract"] == "a8" else be.linear_float)(s.layer, s.x.array, m, s.out.array)
        return s.out.tensor
    if kind == "layer":
        s.qkv.launch()
        be.linear_a8_residual(s.lin["o"], s.attended.array, m, s.x.array, s.out["o"].array)
        s.gate_up.launch()
        be.linear_a8_residual(s.lin["down"], s.gated.array, m, s.out["o"].array, s.out["down"].array)
        return {name: o.tensor for name, o in s.out.items()}
    if kind == "group":
        s.members.launch()
        return [o.tensor for o in s.outs]
    if kind == "forward":
        s.layer.forward(be, s.x, m, s.out)
        return s.out
    if kind == "salt":
        be.linear_salt(s.planes, s.x.array, m, s.out.array)
        return s.out.tensor
    if kind == "salt_v2":
        s.matrix.forward(s.x.array, m, s.out.array)
        return s.out.tensor
    be.projected_vjp(s.layer.planes[0], s.layer.scales[0], s.x.array, s.up.array, m, s.grad_x.array, s.grad_w.array, s.grad_b.array)
    return [s.grad_x.tensor, s.grad_w.tensor, s.grad_b.tensor]


# ---- what a pass cannot do without -------------------------------------------------------------

def _codes(n, k, planes=1):
    """Bytes of 2-bit codes and channel scales."""
    return planes * (n * k / 4 + 4 * n)


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "layer":
        h, kv, f = case["hidden"], case["kv"], case["ffn"]
        shapes = ((h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f))
        return {"bytes": sum(_codes(n, k) + 2 * m * n for n, k in shapes) + 2 * m * (2 * h + f) + 8 * h,
                "flops": sum(2.0 * m * n * k for n, k in shapes)}
    n, k = case["n"], case["k"]
    ops = 2.0 * m * n * k
    if kind == "linear":
        return {"bytes": _codes(n, k, case["planes"]) + m * k * _SIZE[case["act"]] + m * n * _SIZE[case["out"]], "flops": ops * case["planes"]}
    if kind == "group":
        return {"bytes": case["copies"] * (_codes(n, k, case["planes"]) + m * n * _SIZE[case["out"]]) + m * k * _SIZE[case["act"]],
                "flops": ops * case["planes"] * case["copies"]}
    if kind == "forward":
        return {"bytes": _codes(n, k) + 4 * m * (n + k), "flops": ops}
    if kind == "salt":
        return {"bytes": case["planes"] * n * k * (66 / 256) + m * k * _SIZE[case["act"]] + m * n * 4, "flops": ops * case["planes"]}
    if kind == "salt_v2":
        per = {"D2": 64, "B3": 52, "S34": 40}[case["codec"]]
        return {"bytes": 2 * n * k * (per / 256 + 2 / case["scale_group"]) + 4 * m * (n + k), "flops": 2 * ops}
    return {"bytes": _codes(n, k) + 4 * (2 * m * k + m * n + n * k + n), "flops": 2 * ops}


def tolerance(case):
    """The int8 contract, SALT V2 and the gradients promise the bits of the CPU's order. Sums of float activations in
    another order (an f32 fold over k or over blocks against a float64 product, K = 512 .. 17408) differ by up to 1.7e-6;
    a bf16 result additionally rounds to the other neighbour where the two lie on either side of a tie."""
    if case["kind"] == "salt" or case.get("contract") == "float":
        return {"rel": 5e-6} if case["out"] == "f32" else {"rel": 3e-4, "max": 1e-2}
    return "exact"
