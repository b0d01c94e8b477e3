"""Workloads of the quantized linear layers, as a program that serves a model runs them: what one step of an engine asks of
the library, through its public entry points, from one token of one request to a whole prompt chunk.

Kinds of case (a case is a dict of plain values):

* "decode": the projections of `layers` decoder layers over `rows` tokens, every weight a trellis (EXL3) tensor of `bits`
  bits: q, k, v of one input in a group, o with the residual added, then the MLP block with the residual added. 1 row is
  one request, 2..16 rows are speculative verification or a few requests, up to 64 a decode batch. `act` is the type of the
  activations on both sides.
* "x3_prompt": the MLP block over a prompt of `rows` tokens when the trellis is the only form of the weights.
* "mixed": one step of continuous batching, the MLP block over `dec` decode rows (trellis) and `rows` - `dec` prompt rows
  (NVFP4, gate and up fused with SwiGLU). dec = 0 is a prompt chunk alone.
* "fp4": the MLP block of a checkpoint that holds NVFP4 weights only, `rows` tokens: gate and up fused into one linear, SwiGLU,
  down with the residual added.
* "fp8": two e4m3 linears of the prompt path, one after the other, `rows` tokens.
* "bf16": the MLP block over plain bf16 weights, `rows` tokens of which the first `dec` are decode rows.

hidden, kv and inter are the layer's widths: the 5120 / 1024 / 17408 layer of the library's benchmark, half of it as one of
two tensor-parallel ranks holds it, and smaller or odd ones.
"""
import math

import torch

from ferrite_amd import bf16, exl3, fp4, route

B, F = exl3.Dtype.Bf16, exl3.Dtype.F32


def listed():
    full = {"hidden": 5120, "kv": 1024, "inter": 17408}
    mlp = {"hidden": 5120, "inter": 17408}
    return [
        # one request, token by token: the case that the whole format is for
        {"name": "decode 1 row 4 bits", "kind": "decode", "rows": 1, "bits": 4, **full, "layers": 2, "act": "bf16"},
        # a small draft model: nothing but latency, launches and host time
        {"name": "decode 1 row small", "kind": "decode", "rows": 1, "bits": 3, "hidden": 1024, "kv": 256, "inter": 2816, "layers": 1, "act": "bf16"},
        # a verify step of speculative decoding
        {"name": "decode 7 rows 5 bits", "kind": "decode", "rows": 7, "bits": 5, **full, "layers": 1, "act": "bf16"},
        # a decode batch of many requests
        {"name": "decode 40 rows 4 bits", "kind": "decode", "rows": 40, "bits": 4, **full, "layers": 1, "act": "bf16"},
        # a long prompt, and a short one of odd length, straight from the trellis
        {"name": "trellis prompt 2048", "kind": "x3_prompt", "rows": 2048, "bits": 4, **mlp},
        {"name": "trellis prompt 203", "kind": "x3_prompt", "rows": 203, "bits": 3, **mlp},
        # a prompt chunk through the NVFP4 weights, and a step with decode rows in front of a short prompt
        {"name": "nvfp4 prompt 2048", "kind": "mixed", "rows": 2048, "dec": 0, "bits": 4, **mlp},
        {"name": "mixed 5 + 390 rows", "kind": "mixed", "rows": 395, "dec": 5, "bits": 4, **mlp},
        # decode on NVFP4 weights
        {"name": "nvfp4 decode 1 row", "kind": "fp4", "rows": 1, **mlp},
        # the e4m3 linears of a prompt
        {"name": "fp8 prompt 777", "kind": "fp8", "rows": 777, **mlp},
        # unquantized layers: a small decode batch, a prompt
        {"name": "bf16 decode 12 rows", "kind": "bf16", "rows": 12, "dec": 12, **mlp},
        {"name": "bf16 prompt 1000", "kind": "bf16", "rows": 1000, "dec": 0, **mlp},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "x3_prompt", "x3_prompt", "mixed", "mixed", "fp4", "fp4", "fp8", "bf16", "bf16"])
    # widths in blocks of 128, the formats' own granularity
    hidden, inter = rng.choice([(5120, 17408), (5120, 8704), (128 * _log(rng, 8, 40), 128 * _log(rng, 22, 136))])
    case = {"kind": kind, "hidden": hidden, "inter": inter}
    bits = rng.choice([2, 3, 3, 4, 4, 4, 5, 5, 6, 8])
    if kind == "decode":
        case.update(rows=_log(rng, 1, 64), bits=bits, kv=128 * rng.randint(1, 8), layers=rng.randint(1, 2), act=rng.choice(["bf16"] * 5 + ["f32"]))
    elif kind == "x3_prompt":
        case.update(rows=_log(rng, 65, 2048), bits=bits)
    elif kind == "mixed":
        dec = rng.choice([0, _log(rng, 1, 64)])
        case.update(dec=dec, rows=dec + _log(rng, 17, 1984), bits=bits)
    elif kind == "fp4":
        case.update(rows=_log(rng, 1, 2048))
    elif kind == "fp8":
        case.update(rows=_log(rng, 17, 2048))
    else:
        dec = rng.choice([0, _log(rng, 1, 64)])
        rows = dec + rng.choice([0, _log(rng, 17, 1984)])
        case.update(rows=rows or _log(rng, 1, 16), dec=dec)
    return case


# ---- weights and inputs ---------------------------------------------------------------------------------------------------

_kern = {}


def _kernels(mod):
    """The loaded kernels of one weight form: a program loads them once."""
    if mod not in _kern:
        _kern[mod] = mod.Kernels.load()
    return _kern[mod]


class _Maker:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=dtype)

    def activations(self, rows, k, dtype=torch.bfloat16):
        """N(0, 1) with 1 % outlier channels twenty times as large."""
        x = self.normal(rows, k, dtype=torch.float32)
        ch = torch.randperm(k, generator=self.g, device="cuda")[: max(1, k // 100)]
        x[:, ch] *= 20.0
        return x.to(dtype)

    def signs_scales(self, n, scale):
        s = torch.randint(0, 2, (n,), generator=self.g, device="cuda") * 2 - 1
        return (s * (1.0 + 0.05 * self.normal(n, dtype=torch.float32)) * scale).to(torch.float16)

    def trellis(self, k, n, bits, name):
        """A trellis linear: any words are a valid code stream; the scales bring its outputs to the size of its inputs."""
        words = torch.randint(-(1 << 31), 1 << 31, (k * n // 32 * bits,), generator=self.g, device="cuda", dtype=torch.int32)
        suh, svh = self.signs_scales(k, 1.0), self.signs_scales(n, 1.0 / (1.24 * math.sqrt(k)))
        view = exl3.Exl3View(k, n, bits, words.data_ptr(), suh.data_ptr(), svh.data_ptr(), True)
        lin = exl3.Linear.from_view(_kernels(exl3), name, view, exl3.Linear.plan_for(k, n, bits, exl3.default_blocks(exl3.cu_count())))
        lin.keep = (words, suh, svh)
        return lin

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)

    def nvfp4_part(self, n, k, name, input_scale):
        """Codes and block scales of one NVFP4 tensor: codes uniform, scales |N(0, 1)| * 0.1 as e4m3."""
        s = (self.normal(n, k // 16, dtype=torch.float32).abs() * 0.1).clamp(2.0 ** -9, 448.0).to(torch.float8_e4m3fn)
        return (name, self.bytes(n, k // 2).cpu().numpy(), s.view(torch.uint8).cpu().numpy(), 1.0 / (0.29 * math.sqrt(k)), input_scale)

    def fp8_linear(self, n, k, name):
        w = (self.normal(n, k, dtype=torch.float32) * 32.0).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return fp4.HostLinear.fuse_fp8([(name, w.view(torch.uint8).cpu().numpy(), 1.0 / (32.0 * math.sqrt(k)), 0.25)]).upload()

    def weight(self, n, k):
        return self.normal(n, k) * (1.0 / math.sqrt(k))


def _empty(*shape, dtype=torch.bfloat16):
    return torch.zeros(shape, device="cuda", dtype=dtype)


def prepare(case, seed):
    m, kind, rows, h, i = _Maker(seed), case["kind"], case["rows"], case["hidden"], case["inter"]
    s = {"kind": kind, "rows": rows, "hidden": h, "inter": i}
    if kind == "decode":
        t, bits, kv = torch.float32 if case["act"] == "f32" else torch.bfloat16, case["bits"], case["kv"]
        s["x_type"], s["add"] = (F, exl3.Dtype.F32Add) if case["act"] == "f32" else (B, exl3.Dtype.Bf16Add)
        s["layers"], lins = [], []
        for n in range(case["layers"]):
            qkv = [m.trellis(h, h, bits, "q"), m.trellis(h, kv, bits, "k"), m.trellis(h, kv, bits, "v")]
            o, gate, up, down = m.trellis(h, h, bits, "o"), m.trellis(h, i, bits, "gate"), m.trellis(h, i, bits, "up"), m.trellis(i, h, bits, "down")
            s["layers"].append({
                "qkv": qkv, "o": o, "gate": gate, "up": up, "down": down, "x": m.activations(rows, h, t), "attn": m.normal(rows, h, dtype=t),
                "xn": m.activations(rows, h, t), "y": [_empty(rows, l.n, dtype=t) for l in qkv], "resid": m.normal(rows, h, dtype=t),
                "yg": _empty(rows, i), "yu": _empty(rows, i)})
            lins += qkv + [o, gate, up, down]
        s["ws"] = exl3.Workspace(lins, rows)
        return s
    s["x"] = m.normal(rows, h)
    s["xn"] = m.activations(rows, h)
    if kind == "fp8":
        s["up"], s["down"] = m.fp8_linear(i, h, "up"), m.fp8_linear(h, i, "down")
        s["ws"], s["mid"] = fp4.Workspace(rows, max(h, i)), _empty(rows, i)
        return s
    s["big"], s["act"] = _empty(rows, 2 * i), _empty(rows, i)
    if kind == "fp4":
        gate, up = m.nvfp4_part(i, h, "gate", 1.0), m.nvfp4_part(i, h, "up", 1.0)
        s["gate_up"] = fp4.HostLinear.fuse([gate, up]).upload()
        s["down"] = fp4.HostLinear.fuse([m.nvfp4_part(h, i, "down", 1.0)]).upload()
        s["ws"] = fp4.Workspace(rows, max(h, i))
        return s
    q, w, p, x3, f4 = [None] * 3, [None] * 3, None, None, None
    s["swiglu"] = s["act_ws"] = s["swiglu_w"] = None
    if kind in ("x3_prompt", "mixed"):
        bits = case["bits"]
        q = [m.trellis(h, i, bits, "gate"), m.trellis(h, i, bits, "up"), m.trellis(i, h, bits, "down")]
        x3 = (_kernels(exl3), exl3.Workspace(q, rows if kind == "x3_prompt" else 64))
    if kind == "mixed":
        host = fp4.HostLinear.fuse([m.nvfp4_part(i, h, "gate", 1.0), m.nvfp4_part(i, h, "up", 1.0)])
        s["swiglu"] = host.into_swiglu().upload()
        p = fp4.HostLinear.fuse([m.nvfp4_part(h, i, "down", 1.0)]).upload()
        f4, s["act_ws"] = (_kernels(fp4), fp4.Workspace(rows, max(h, i))), fp4.Workspace(rows, i)
    if kind == "bf16":
        w = [m.weight(i, h), m.weight(i, h), m.weight(h, i)]
        s["swiglu_w"] = bf16.interleave_gu(_kernels(bf16), w[0], w[1])
    s["ctx"] = route.LinCtx(x3=x3, fp4=f4)
    if kind == "bf16":
        s["ctx"].set_bf16(_kernels(bf16))
    s["ctx"].dec = case.get("dec", 0)
    s["gate_up"] = route.Proj([(route.Linear("gate", i, h, q=q[0], w=w[0]), [i]), (route.Linear("up", i, h, q=q[1], w=w[1]), [i])])
    s["down"] = route.Linear("down", h, i, q=q[2], p=p, w=w[2])
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------------

def run(s):
    rows, kind = s["rows"], s["kind"]
    if kind == "decode":
        t, ws = s["x_type"], s["ws"]
        for l in s["layers"]:
            exl3.forward_group(l["qkv"], l["x"], t, l["y"], t, rows, ws)
            l["o"].forward(l["attn"], t, l["resid"], s["add"], rows, ws)
            exl3.mlp_forward(l["gate"], l["up"], l["down"], l["xn"], t, l["yg"], l["yu"], l["resid"], s["add"], rows, ws)
        return [l["y"] + [l["yg"], l["yu"], l["resid"]] for l in s["layers"]]
    h, i, x, xn = s["hidden"], s["inter"], s["x"], s["xn"]
    if kind == "fp8":
        s["up"].forward(_kernels(fp4), s["ws"], s["mid"], i, xn, h, rows)
        s["down"].forward(_kernels(fp4), s["ws"], x, h, s["mid"], i, rows, res=x)
        return [s["mid"], x]
    if kind == "fp4":
        big, act = s["big"], s["act"]
        s["gate_up"].forward(_kernels(fp4), s["ws"], big, 2 * i, xn, h, rows)
        route.silu_mul(act, big.data_ptr(), big.data_ptr() + 2 * i, 2 * i, i, rows)
        s["down"].forward(_kernels(fp4), s["ws"], x, h, act, i, rows, res=x)
        return [big, act, x]
    route.mlp_forward(s["ctx"], s["gate_up"], s["down"], x, xn, s["big"], s["act"], rows, h, i, swiglu=s["swiglu"],
                      act_ws=s["act_ws"], swiglu_w=s["swiglu_w"])
    return [x]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def work(case):
    """Each weight form that the rows need read once, inputs read once, outputs written once (the residual both)."""
    rows, h, i, kind = case["rows"], case["hidden"], case["inter"], case["kind"]
    mlp_weights, mlp_io = 3 * h * i, rows * 2 * (h + 2 * h)  # xn in, x in and out
    flops = 2 * rows * mlp_weights
    if kind == "decode":
        kv, e = case["kv"], 4 if case["act"] == "f32" else 2
        weights = 2 * h * h + 2 * h * kv + mlp_weights
        scales = 2 * (4 * h + 2 * h + 2 * kv + 2 * (h + i) + i + h)
        io = rows * (e * (h + h + 2 * kv + h + h + 2 * h) + 2 * 2 * i)
        return {"bytes": case["layers"] * (weights * case["bits"] // 8 + scales + io), "flops": case["layers"] * 2 * rows * weights}
    if kind == "x3_prompt":
        return {"bytes": mlp_weights * case["bits"] // 8 + mlp_io, "flops": flops}
    if kind == "mixed":
        trellis = mlp_weights * case["bits"] // 8 if case["dec"] else 0
        return {"bytes": trellis + mlp_weights * 9 // 16 + mlp_io, "flops": flops}
    if kind == "fp4":
        return {"bytes": mlp_weights * 9 // 16 + mlp_io + rows * 2 * 3 * i, "flops": flops}
    if kind == "fp8":
        return {"bytes": 2 * h * i + rows * 2 * (3 * h + i), "flops": 2 * rows * 2 * h * i}
    return {"bytes": 2 * mlp_weights + mlp_io, "flops": flops}


def tolerance(case):
    """bf16 results of f32 sums: another order of the sums moves a value by one bf16 step where it lies between two, and the
    MLP block's inner values, which are bf16 too, by the same. Where activations are quantized to 4 or 8 bits between two
    linears, such a step can move a code."""
    if case["kind"] in ("mixed", "fp4", "fp8"):
        return {"rel": 1e-2, "max": 6e-2}
    return {"rel": 4e-3, "max": 2e-2}
