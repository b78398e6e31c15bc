"""The work this framework is used for, as cases to time and to check: decode projections and MLPs of 1 to 32 rows,
prefill projections and MLPs of up to 2048 rows, and MoE blocks in both directions, in the weight formats a model
carries. Every pass goes through the C ABI (splash_q4's binding of it) with the plan, weights and buffers that a
serving program holds.

Weights are native MLX affine tensors or GGUF blocks made from the seed, repacked at preparation as a loader does;
`exact` dequantises the same native tensors in 64 bits with plain torch.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "splash-desktop_amd"))

import splash_q4 as sq  # noqa: E402

FORMATS = {"af4g32": sq.FMT_AF4G32, "af4g64": sq.FMT_AF4G64, "af4g128": sq.FMT_AF4G128, "af8g64": sq.FMT_AF8G64,
           "q4_k": sq.FMT_Q4K, "q5_k": sq.FMT_Q5K, "q6_k": sq.FMT_Q6K, "q8_0": sq.FMT_Q80}
AFFINE = {"af4g32": (4, 32), "af4g64": (4, 64), "af4g128": (4, 128), "af8g64": (8, 64)}
RMS_EPSILON = 1e-6


# ---------------------------------------------------------------- cases

def listed():
    return [
        # One token through one square projection: the smallest call, a single short dispatch.
        {"name": "row1_proj", "kind": "proj", "rows": 1, "k": 4096, "n": 4096, "fmt": "af4g64", "residual": False},
        # Two rows (a draft step) through an MLP: norm, one gate/up pair, down onto the residual stream.
        {"name": "row2_mlp", "kind": "mlp", "rows": 2, "h": 4096, "i": 14336, "fmt": "af4g64", "down": "af4g64"},
        # One verify lane of eight rows through the 27B model's MLP.
        {"name": "verify8_mlp", "kind": "mlp", "rows": 8, "h": 5120, "i": 17408, "fmt": "af4g64", "down": "af4g64"},
        # Two lanes through a fused q|k|v of two formats, one dispatch.
        {"name": "verify16_qkv", "kind": "qkv", "rows": 16, "k": 5120, "q": 6144, "kv": 1024, "fmt": "q4_k",
         "vfmt": "q6_k"},
        # Four lanes, the most rows a decode step has, through an MLP of GGUF's usual mix (Q4_K, Q6_K down).
        {"name": "verify32_mlp", "kind": "mlp", "rows": 32, "h": 5120, "i": 17408, "fmt": "q4_k", "down": "q6_k"},
        # The output head of a verify lane: the largest single tensor, fp32 logits.
        {"name": "head8", "kind": "head", "rows": 8, "k": 5120, "n": 131072, "fmt": "q6_k"},
        # A short prompt of an odd length through an attention output projection onto the residual stream.
        {"name": "prefill77_proj", "kind": "proj", "rows": 77, "k": 6144, "n": 5120, "fmt": "q4_k", "residual": True},
        # A middling chunk through an 8-bit projection.
        {"name": "prefill500_proj", "kind": "proj", "rows": 500, "k": 4096, "n": 14336, "fmt": "q8_0",
         "residual": False},
        # A full chunk through an MLP: the largest case.
        {"name": "prefill2048_mlp", "kind": "mlp", "rows": 2048, "h": 4096, "i": 14336, "fmt": "af4g64",
         "down": "af4g64"},
        # One verify lane through the 35B model's MoE block (Q4_K gate/up, Q5_K down, a gated Q8_0 shared expert).
        {"name": "moe_decode8", "kind": "moe", "rows": 8, "h": 2048, "i": 512, "experts": 256, "top_k": 8,
         "fmt": "q4_k", "down": "q5_k", "shared": 1, "sfmt": "q8_0"},
        # A chunk of 512 rows through 128 routed experts alone, MLX 4-bit.
        {"name": "moe_prefill512", "kind": "moe", "rows": 512, "h": 2048, "i": 768, "experts": 128, "top_k": 8,
         "fmt": "af4g64", "down": "af4g64", "shared": 0, "sfmt": ""},
        # A nearly full chunk of an odd length through the 35B model's MoE block.
        {"name": "moe_prefill1999", "kind": "moe", "rows": 1999, "h": 2048, "i": 512, "experts": 256, "top_k": 8,
         "fmt": "q4_k", "down": "q5_k", "shared": 1, "sfmt": "q8_0"},
    ]


def draw(rng):
    def spread(lo, hi, step=1):
        """lo..hi, a multiple of step, spread over the logarithm."""
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return max(lo, min(hi, int(round(v / step)) * step))

    fmt, down = rng.choice(sorted(FORMATS)), rng.choice(sorted(FORMATS))
    kind = rng.choice(["proj", "proj", "prefill", "prefill", "mlp", "mlp", "prefill_mlp", "qkv", "head", "moe", "moe",
                       "moe_prefill", "moe_prefill"])
    if kind == "proj":
        return {"kind": "proj", "rows": spread(1, 32), "k": spread(1024, 14336, 256), "n": spread(512, 28672, 64),
                "fmt": fmt, "residual": rng.random() < 0.5}
    if kind == "prefill":
        return {"kind": "proj", "rows": spread(33, 2048), "k": spread(1024, 14336, 256), "n": spread(512, 14336, 64),
                "fmt": fmt, "residual": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": "mlp", "rows": spread(1, 32), "h": spread(1024, 5120, 256), "i": spread(2048, 17408, 256),
                "fmt": fmt, "down": down}
    if kind == "prefill_mlp":
        return {"kind": "mlp", "rows": spread(33, 2048), "h": spread(1024, 4096, 256), "i": spread(2048, 14336, 256),
                "fmt": fmt, "down": down}
    if kind == "qkv":
        return {"kind": "qkv", "rows": spread(1, 32), "k": spread(1024, 5120, 256), "q": spread(1024, 8192, 64),
                "kv": spread(256, 2048, 64), "fmt": fmt, "vfmt": down}
    if kind == "head":
        return {"kind": "head", "rows": spread(1, 8), "k": spread(1024, 4096, 256), "n": spread(32768, 131072, 64),
                "fmt": rng.choice(["q6_k", "q8_0", "q4_k", "af4g64", "af8g64"])}
    shared = rng.choice([0, 1])
    return {"kind": "moe", "rows": spread(1, 32) if kind == "moe" else spread(33, 1999),
            "h": spread(1024, 2048, 256), "i": rng.choice([256, 512, 768]), "experts": rng.choice([64, 128, 256]),
            "top_k": rng.choice([4, 6, 8]), "fmt": rng.choice(["af4g32", "af4g64", "af4g128", "q4_k", "q5_k", "q8_0"]),
            "down": rng.choice(["af4g64", "q4_k", "q5_k", "q6_k"]), "shared": shared,
            "sfmt": rng.choice(["q8_0", "af8g64"]) if shared else ""}


# ---------------------------------------------------------------- weights

def uniform(gen, shape, lo, hi):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=gen)


def codes_of(gen, shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)


class Affine:
    """MLX affine tensors: little-endian packed codes, a bf16 scale and bias a group; w = s q + z."""

    def __init__(self, gen, fmt, n, k):
        self.fmt, self.n, self.k = fmt, n, k
        bits, group = AFFINE[fmt]
        self.codes = codes_of(gen, (n, k * bits // 8))
        sigma = 0.005 if bits == 4 else 0.005 / 16
        scales = torch.randn((n, k // group), device="cuda", generator=gen).abs_().add_(0.2).mul_(sigma)
        self.scales = scales.to(torch.bfloat16)
        self.biases = (self.scales.float() * -float(1 << (bits - 1))).to(torch.bfloat16)

    def planes(self):
        p0, meta = sq.plane_bytes(FORMATS[self.fmt], self.n, self.k)
        plane0 = torch.empty(p0, dtype=torch.uint8, device="cuda")
        words = torch.empty(meta, dtype=torch.uint8, device="cuda")
        sq.mlx_repack(FORMATS[self.fmt], self.n, self.k, self.codes, self.scales, self.biases, plane0, words)
        return plane0, None, words

    def values(self, lo, hi):
        bits, group = AFFINE[self.fmt]
        c = self.codes[lo:hi]
        q = c if bits == 8 else torch.stack([c & 15, c >> 4], -1).reshape(hi - lo, self.k)
        q = q.double().reshape(hi - lo, -1, group)
        w = q * self.scales[lo:hi, :, None].double() + self.biases[lo:hi, :, None].double()
        return w.reshape(hi - lo, self.k)


def half_bytes(values):
    """float [blocks] -> the two bytes of each one's fp16."""
    return values.to(torch.float16).view(torch.uint8).reshape(-1, 2)


class Gguf:
    """GGUF blocks of 256 (Q8_0: 32) elements with scales a model's blocks have."""
    BYTES = {"q4_k": 144, "q5_k": 176, "q6_k": 210, "q8_0": 34}

    def __init__(self, gen, fmt, n, k):
        self.fmt, self.n, self.k = fmt, n, k
        blocks = n * k // (32 if fmt == "q8_0" else 256)
        raw = codes_of(gen, (blocks, self.BYTES[fmt]))
        if fmt == "q8_0":
            raw[:, :2] = half_bytes(uniform(gen, blocks, 1e-4, 4e-4))
        elif fmt == "q6_k":
            scales = torch.randint(32, 128, (blocks, 16), dtype=torch.int16, device="cuda", generator=gen)
            signs = torch.randint(0, 2, (blocks, 16), dtype=torch.int16, device="cuda", generator=gen) * 2 - 1
            raw[:, 192:208] = (scales * signs).to(torch.int8).view(torch.uint8)
            raw[:, 208:] = half_bytes(uniform(gen, blocks, 5e-6, 2e-5))
        else:
            middle = 7.5 if fmt == "q4_k" else 15.5
            d = uniform(gen, blocks, 6e-5, 1.5e-4) * (7.5 / middle)
            raw[:, :2], raw[:, 2:4] = half_bytes(d), half_bytes(d * middle)
            sc = torch.randint(18, 60, (blocks, 8), dtype=torch.int16, device="cuda", generator=gen)
            mn = sc + torch.randint(-3, 4, (blocks, 8), dtype=torch.int16, device="cuda", generator=gen)
            raw[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
            raw[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
            raw[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
        self.raw = raw

    def planes(self):
        f, n, k = FORMATS[self.fmt], self.n, self.k
        p0, meta = sq.plane_bytes(f, n, k)
        p1 = n * (k // 32) * sq.FORMATS[f][5]
        dst = torch.empty(p0 + p1 + meta, dtype=torch.uint8, device="cuda")
        sq.gguf_repack(self.raw, dst, n, k, f, self.raw.numel() // n, p0 + p1, dst_plane1=p0 if p1 else 0)
        return dst[:p0], dst[p0:p0 + p1] if p1 else None, dst[p0 + p1:]

    def values(self, lo, hi):
        per = self.raw.shape[0] // self.n
        b = self.raw[lo * per:hi * per]

        def half(at):
            return b[:, at:at + 2].contiguous().view(torch.float16).double()

        if self.fmt == "q8_0":
            return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(hi - lo, self.k)
        if self.fmt == "q6_k":
            out = []
            for part in range(2):
                ql, qh = b[:, 64 * part:64 * part + 64], b[:, 128 + 32 * part:160 + 32 * part]
                lo4, hi4 = ql & 15, ql >> 4
                for i, four in enumerate((lo4[:, :32], lo4[:, 32:], hi4[:, :32], hi4[:, 32:])):
                    out.append(four.double() + ((qh >> (2 * i)) & 3).double() * 16 - 32)
            q = torch.stack(out, 1).reshape(-1, 16, 16)
            s = half(208) * b[:, 192:208].contiguous().view(torch.int8).double()
            return (q * s[:, :, None]).reshape(hi - lo, self.k)
        s12 = b[:, 4:16].to(torch.int16)
        a, m, c = s12[:, :4], s12[:, 4:8], s12[:, 8:]
        sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], 1).double()
        mn = torch.cat([m & 63, (c >> 4) | ((m >> 6) << 4)], 1).double()
        qs = b[:, 16:144] if self.fmt == "q4_k" else b[:, 48:176]
        qs = qs.reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        if self.fmt == "q5_k":
            fifth = torch.stack([(b[:, 16:48] >> i) & 1 for i in range(8)], 1)
            q = q + 16 * fifth.double()
        w = q * (half(0) * sc)[:, :, None] - (half(2) * mn)[:, :, None]
        return w.reshape(hi - lo, self.k)


def weight(gen, fmt, n, k):
    return (Affine if fmt in AFFINE else Gguf)(gen, fmt, n, k)


def weight_bytes(fmt, n, k):
    if fmt in AFFINE:
        bits, group = AFFINE[fmt]
        return n * k * (bits / 8 + 4 / group)
    return n * k * Gguf.BYTES[fmt] / (32 if fmt == "q8_0" else 256)


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def stream_rows(gen, rows, width):
    """A residual stream: N(0, 1) with eight channels of twenty times the size."""
    x = torch.randn((rows, width), device="cuda", generator=gen)
    x[:, torch.randperm(width, device="cuda", generator=gen)[:8]] *= 20
    return x.to(torch.bfloat16)


def inputs(case, gen):
    """Everything `prepare` and `exact` share: the activations and native weights of the case."""
    kind, rows = case["kind"], case["rows"]
    normal = lambda r, w: torch.randn((r, w), device="cuda", generator=gen).to(torch.bfloat16)  # noqa: E731
    d = {}
    if kind in ("proj", "head"):
        d["x"] = normal(rows, case["k"])
        d["w"] = weight(gen, case["fmt"], case["n"], case["k"])
        if case.get("residual"):
            d["residual"] = stream_rows(gen, rows, case["n"])
    elif kind == "qkv":
        d["x"] = normal(rows, case["k"])
        d["w"] = [weight(gen, f, n, case["k"]) for f, n in ((case["fmt"], case["q"]), (case["fmt"], case["kv"]),
                                                            (case["vfmt"], case["kv"]))]
    elif kind == "mlp":
        d["x"] = stream_rows(gen, rows, case["h"])
        d["norm"] = (1 + 0.1 * torch.randn(case["h"], device="cuda", generator=gen)).to(torch.bfloat16)
        d["gate"], d["up"] = (weight(gen, case["fmt"], case["i"], case["h"]) for _ in range(2))
        d["down"] = weight(gen, case["down"], case["h"], case["i"])
    else:
        e, h, i, s = case["experts"], case["h"], case["i"], case["shared"]
        d["x"], d["residual"] = normal(rows, h), stream_rows(gen, rows, h)
        d["router"] = torch.randn((e, h), device="cuda", generator=gen) * (1.5 / math.sqrt(h))
        d["gate"], d["up"] = (weight(gen, case["fmt"], e * i, h) for _ in range(2))
        d["down"] = weight(gen, case["down"], e * h, i)
        d["slots"] = torch.randperm(e, device="cuda", generator=gen)   # an expert store's slot of each expert
        if s:
            d["shared_gate"], d["shared_up"] = (weight(gen, case["sfmt"], s * i, h) for _ in range(2))
            d["shared_down"] = weight(gen, case["sfmt"], s * h, i)
            d["scalar"] = torch.randn(h, device="cuda", generator=gen) * 0.05
    return d


# ---------------------------------------------------------------- passes

def segment_of(w, column_offset=0):
    """(the planes, to keep; the segment) of a native weight."""
    plane0, plane1, meta = w.planes()
    return (plane0, plane1, meta), sq.segment(FORMATS[w.fmt], w.n, w.k, plane0, meta, column_offset, plane1)


def workload(n, k, rows, epilogue):
    return (sq.decode_workload if rows <= 32 else sq.prefill_workload)(n, k, rows, epilogue)


def empty(rows, width, dtype=torch.bfloat16):
    return torch.empty((rows, width), dtype=dtype, device="cuda")


def prepare_proj(case, d, keep):
    rows = case["rows"]
    if case["kind"] == "qkv":
        segments, at = [], 0
        for w in d["w"]:
            planes, s = segment_of(w, at)
            keep.append(planes)
            segments.append(s)
            at += w.n
        proj = sq.projection(segments)
    else:
        planes, s = segment_of(d["w"])
        keep.append(planes)
        proj = sq.projection(s, destination=sq.OUTPUT_F32 if case["kind"] == "head" else sq.OUTPUT_BF16)
    residual = d.get("residual")
    epilogue = sq.EPILOGUE_RESIDUAL if residual is not None else sq.EPILOGUE_NONE
    plan = sq.plan_for(workload(proj.output_size, proj.input_size, rows, epilogue), proj)
    scratch = sq.Scratch(plan)
    out = empty(plan.storage_rows, proj.output_size, torch.float32 if case["kind"] == "head" else torch.bfloat16)
    x, r = padded(d["x"], plan.storage_rows), padded(residual, plan.storage_rows)
    buffers = sq.LinearBuffers(sq.view(x), sq.view(out), sq.view(r), sq.view(None), scratch.struct())
    keep += [scratch, x, r, buffers, proj, plan]
    calls = [("sq_linear_add", sq.stream_handle(), ctypes.byref(buffers), ctypes.byref(proj), ctypes.byref(plan), None)]
    return calls, [out[:rows]]


def padded(x, rows):
    """The rows of storage a plan binds (a prefill's are whole tiles): the live rows first."""
    if x is None or x.shape[0] >= rows:
        return x
    return torch.cat([x, torch.zeros((rows - x.shape[0], x.shape[1]), dtype=x.dtype, device="cuda")])


def prepare_mlp(case, d, keep):
    rows, h, i = case["rows"], case["h"], case["i"]
    projections = {}
    for name in ("gate", "up", "down"):
        planes, s = segment_of(d[name])
        projections[name] = sq.projection(s)
        keep.append(planes)
    gate, up, down = (projections[n] for n in ("gate", "up", "down"))
    storage = rows if rows <= 32 else (rows + 127) // 128 * 128
    x = padded(d["x"], storage)
    normal, inner, out = empty(storage, h), empty(storage, i), empty(storage, h)
    norm = sq.NormWeights(sq.view(d["norm"]), 0)
    stream = sq.stream_handle()
    calls = [("sq_norm_add_rms", stream, sq.view(x), ctypes.byref(norm), sq.view(normal), h, rows, None,
              sq.LINEAR_INPUT_PLAIN, None)]
    if rows <= 32:
        pair = sq.plan_for(sq.decode_workload(i, h, rows, sq.EPILOGUE_GATE_UP), up, gate)
        last = sq.plan_for(sq.decode_workload(h, i, rows, sq.EPILOGUE_RESIDUAL), down)
        ps, ls = sq.Scratch(pair), sq.Scratch(last)
        b1 = sq.LinearBuffers(sq.view(normal), sq.view(inner), sq.view(None), sq.view(ps.gate), ps.struct())
        b2 = sq.LinearBuffers(sq.view(inner), sq.view(out), sq.view(x), sq.view(None), ls.struct())
        keep += [pair, last, ps, ls, b1, b2]
        calls += [("sq_linear_add", stream, ctypes.byref(b1), ctypes.byref(up), ctypes.byref(pair), ctypes.byref(gate)),
                  ("sq_linear_add", stream, ctypes.byref(b2), ctypes.byref(down), ctypes.byref(last), None)]
    else:
        # One scratch for the layer's projections, as an engine sizes it: the largest of each part.
        plans = [sq.plan_for(sq.prefill_workload(i, h, rows), up), sq.plan_for(sq.prefill_workload(h, i, rows), down)]
        sizes = [sq.scratch_size(p)[0] for p in plans]
        parts = [torch.zeros(max(getattr(s, f) for s in sizes) // 4 + 1, dtype=torch.int32, device="cuda")
                 for f in ("input", "sums", "partials", "counters")]
        scratch = sq.LinearScratch(*[sq.view(p) for p in parts], sq.view(None))
        gated, device = empty(storage, i), sq.device()
        keep += [parts, scratch, gated, device]
        calls.append(("sq_linear_add_prefill_swiglu", ctypes.byref(device), stream, ctypes.byref(gate),
                      ctypes.byref(up), ctypes.byref(down), sq.view(normal), sq.view(gated), sq.view(inner),
                      ctypes.byref(scratch), sq.view(x), sq.view(out), rows))
    keep += [projections, x, norm, d["norm"]]
    return calls, [normal[:rows], inner[:rows], out[:rows]]


def prepare_moe(case, d, keep):
    rows, h, i, e, s = case["rows"], case["h"], case["i"], case["experts"], case["shared"]
    shape = sq.MoeShape(h, e, case["top_k"], i, FORMATS[case["fmt"]], sq.ROUTER_SOFTMAX, s, 1 if s else 0)
    plan = sq.MoePlan()
    if rows <= 32:
        sq.call("sq_moe_decode_rows_plan", ctypes.byref(shape), rows, ctypes.byref(plan))
    else:
        sq.call("sq_moe_prefill_plan", ctypes.byref(shape), rows, None, ctypes.byref(plan))

    # Expert x's planes sit in slot slots[x]: the native rows are in slot order.
    table = d["slots"].to(torch.int32)

    def part(name):
        if name not in d:
            return sq.Segment()
        planes, seg = segment_of(d[name])
        keep.append(planes)
        return seg

    router = sq.Segment(sq.view(d["router"]), sq.view(None), sq.view(None), e, h, 0, sq.FLOAT32_ROWS)
    weights = sq.MoeWeights(part("gate"), part("up"), part("down"), sq.view(table), e, part("shared_gate"),
                            part("shared_up"), part("shared_down"), sq.view(d.get("scalar")), router)
    scratch, fields = sq.MoeScratch(), [f[0] for f in sq.MoeWorkspace._fields_]
    for f in fields:
        t = torch.zeros(getattr(plan.workspace, f) // 4 + 4, dtype=torch.int32, device="cuda")
        keep.append(t)
        setattr(scratch, f, sq.view(t))
    out = empty(rows, h)
    buffers = sq.MoeBuffers(sq.view(d["x"]), sq.view(d["residual"]), sq.view(out), scratch, sq.view(None))
    keep += [shape, plan, table, weights, scratch, buffers, d["x"], d["residual"], d["router"], d.get("scalar")]
    return [("sq_moe_add", sq.stream_handle(), ctypes.byref(buffers), ctypes.byref(weights), ctypes.byref(plan))], [out]


def prepare(case, seed):
    d, keep = inputs(case, generator(seed)), []
    make = {"mlp": prepare_mlp, "moe": prepare_moe}.get(case["kind"], prepare_proj)
    calls, outputs = make(case, d, keep)
    return {"calls": calls, "outputs": outputs, "keep": keep}


def run(state):
    for c in state["calls"]:
        sq.call(*c)
    return state["outputs"]


# ---------------------------------------------------------------- the same in 64 bits

def rounded(x):
    return x.to(torch.bfloat16).double()


def product(x, w, lo=0, hi=None):
    """x (fp64) times rows lo..hi of a native weight, transposed."""
    hi = w.n if hi is None else hi
    step = max(64, (1 << 27) // w.k)
    return torch.cat([x @ w.values(a, min(hi, a + step)).T for a in range(lo, hi, step)], 1)


def swiglu(x, gate, up, lo=0, hi=None):
    """The gated product of two projections, before its bf16 rounding (the projections round to bf16)."""
    g, u = rounded(product(x, gate, lo, hi)), rounded(product(x, up, lo, hi))
    return u * g * torch.sigmoid(g)


def exact(case, seed):
    d = inputs(case, generator(seed))
    x = d["x"].double()
    kind = case["kind"]
    if kind == "qkv":
        return [torch.cat([product(x, w) for w in d["w"]], 1)]
    if kind in ("proj", "head"):
        y = product(x, d["w"])
        return [y + d["residual"].double() if "residual" in d else y]
    if kind == "mlp":
        normal = x * torch.rsqrt(x.square().mean(1, keepdim=True) + RMS_EPSILON) * d["norm"].double()
        inner = swiglu(rounded(normal), d["gate"], d["up"])
        return [normal, inner, x + product(rounded(inner), d["down"])]
    e, h, i, k = case["experts"], case["h"], case["i"], case["top_k"]
    scores, chosen = (x @ d["router"].double().T).topk(k, dim=1)
    share = torch.softmax(scores, 1)
    out = d["residual"].double()

    def expert(rows, part, slot):
        inner = rounded(swiglu(rows, d[part + "gate"], d[part + "up"], slot * i, slot * i + i))
        return rounded(product(inner, d[part + "down"], slot * h, slot * h + h))

    for x_id, slot in enumerate(d["slots"].tolist()):
        row, rank = (chosen == x_id).nonzero(as_tuple=True)
        if row.numel():
            out.index_add_(0, row, share[row, rank, None] * expert(x[row], "", slot))
    for s in range(case["shared"]):
        out += torch.sigmoid(x @ d["scalar"].double())[:, None] * expert(x, "shared_", s)
    return [out]


# ---------------------------------------------------------------- work and tolerance

def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind in ("proj", "head"):
        n, k = case["n"], case["k"]
        out = rows * n * (4 if kind == "head" else 2) + (rows * n * 2 if case.get("residual") else 0)
        return {"bytes": weight_bytes(case["fmt"], n, k) + rows * k * 2 + out, "flops": 2 * rows * n * k}
    if kind == "qkv":
        n, k = case["q"] + 2 * case["kv"], case["k"]
        return {"bytes": weight_bytes(case["fmt"], case["q"] + case["kv"], k) + weight_bytes(case["vfmt"], case["kv"], k)
                + rows * (k + n) * 2, "flops": 2 * rows * n * k}
    if kind == "mlp":
        # The input, and each of the three outputs once.
        h, i = case["h"], case["i"]
        return {"bytes": 2 * weight_bytes(case["fmt"], i, h) + weight_bytes(case["down"], h, i) + rows * (3 * h + i) * 2,
                "flops": 6 * rows * h * i}
    h, i, e, k, s = case["h"], case["i"], case["experts"], case["top_k"], case["shared"]
    live = e * (1 - (1 - k / e) ** rows)   # the experts that some row is expected to choose
    each = 2 * weight_bytes(case["fmt"], i, h) + weight_bytes(case["down"], h, i)
    shared = s * 3 * weight_bytes(case["sfmt"], i, h) if s else 0
    return {"bytes": live * each + shared + e * h * 4 + rows * h * 6,
            "flops": 2 * rows * (3 * (k + s) * h * i + e * h)}


def tolerance(case):
    # Measured against `exact`: 0.0014 to 0.0021 of the norm wherever outputs round to bf16 (2^-9 at most, and an MLP's
    # intermediate rounds before its last sum), 4e-7 to 8e-7 for the head's fp32 logits (sums in another order).
    if case["kind"] == "head":
        return {"rel": 3e-6, "max": 3e-5}
    return {"rel": 8e-3, "max": 5e-2}
