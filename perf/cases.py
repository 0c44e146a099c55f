"""The work that a program has this library do, as cases that can be timed and compared.

Four kinds of call, each through the public entry points of `beglin_amd`:

  linear   one bgl_matmul_dev / bgl_matmul_group_dev call: a projection, or q/k/v or gate+up fused
  mlp      one bgl_mlp_dev call: gate+up, SwiGLU, down
  step     the projections of one decoding step over several layers (fused q/k/v, o, the MLP block
           per layer), captured once into a HIP graph and replayed, as a serving loop does
  moe      one bgl_moe_layer_dev call: router, top-K, the routed experts, the shared experts
  pack     load time: one fp32 tensor packed on the device (bgl_quantize_dev) and read back decoded

Weights are N(0, 0.02) rounded to nearest in the engine's byte layouts and bound with bgl_bind, as
the engine's blobs are; activations are N(0, 1).  `exact` decodes the same bytes in 64 bits.
"""
import math
import random

import torch

import beglin_amd as B

KINDS = {"q4g64": B.K_Q4G64, "q8g64": B.K_Q8G64, "g256sf": B.K_Q4G256SF, "qng64": B.K_QNG64, "q4g32h": B.K_Q4G32H,
         "q4g64a": B.K_Q4G64A}
ACTS = {"f32": B.ACT_F32, "w4a8": B.ACT_W4A8}

# The per-expert formats of a mixed-precision routed layer: int4 group-32, int8 and qNg64 n = 7..15.
MIXED = [("q4g32h", 4), ("q8g64", 8)] + [("qng64", n) for n in range(7, 16)]


# ---------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one int4 projection of one token (Qwen2.5-1.5B's gate, 8960 x 1536)
        dict(name="linear_int4_token", call="linear", kind="q4g32h", bits=4, act="f32", rows="8960", cols=1536, m=1),
        # decoding one sequence: Qwen2.5-1.5B's projections, g256sf weights, int8 activations
        dict(name="step_g256sf_token", call="step", kind="g256sf", bits=4, act="w4a8", mlp_kind="g256sf", mlp_bits=4,
             hidden=1536, kv=256, inner=8960, layers=14, m=1),
        # the same model serving eight sequences at once
        dict(name="step_g256sf_batch8", call="step", kind="g256sf", bits=4, act="w4a8", mlp_kind="g256sf", mlp_bits=4,
             hidden=1536, kv=256, inner=8960, layers=14, m=8),
        # one token through an 8B-sized MLP block in bit planes (qNg64), fp32 activations
        dict(name="mlp_qng64_token", call="mlp", kind="qng64", bits=6, act="f32", hidden=4096, inner=14336, m=1),
        # checking a few speculated tokens: the fused gate+up pair, int4, fp32 activations
        dict(name="linear_q4g64_spec5", call="linear", kind="q4g64", bits=4, act="f32", rows="14336,14336", cols=4096, m=5),
        # 32 sequences of an 8B model (Llama-3.1-8B's shapes): int8 attention, int4 MLP, fp32 activations
        dict(name="step_mixed_batch32", call="step", kind="q8g64", bits=8, act="f32", mlp_kind="q4g32h", mlp_bits=4,
             hidden=4096, kv=1024, inner=14336, layers=2, m=32),
        # a prompt chunk of 64 tokens through the 8B MLP block, int4 weights and int8 activations
        dict(name="mlp_q4g64_chunk64", call="mlp", kind="q4g64", bits=4, act="w4a8", hidden=4096, inner=14336, m=64),
        # a routed layer (DeepSeek-V2-Lite: 64 experts, top 6, two shared) in mixed precision:
        # one token, a small batch, a prompt chunk
        dict(name="moe_mixed_token", call="moe", fmt="mixed", experts=64, top=6, hidden=2048, inner=1408, shared=2816, m=1),
        dict(name="moe_mixed_batch8", call="moe", fmt="mixed", experts=64, top=6, hidden=2048, inner=1408, shared=2816, m=8),
        dict(name="moe_mixed_chunk64", call="moe", fmt="mixed", experts=64, top=6, hidden=2048, inner=1408, shared=2816, m=64),
        # the same layer in affine int4, the format that the name-keyed MoE boundary binds by default
        dict(name="moe_affine_batch16", call="moe", fmt="q4g64a", experts=64, top=6, hidden=2048, inner=1408, shared=2816, m=16),
        # load time: one 8B-sized fp32 tensor packed to int4 with error feedback and decoded
        dict(name="pack_q4g64", call="pack", kind="q4g64", bits=4, rows="14336", cols=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(2 ** rng.uniform(math.log2(lo), math.log2(hi))))


def _width(rng, lo, hi, unit):
    """A multiple of `unit`, log-uniform in [lo, hi]: the widths that the weight groups allow, odd multiples among them."""
    return max(1, int(round(_log_int(rng, lo, hi) / unit))) * unit


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        call = rng.choice(["linear", "linear", "mlp", "step", "moe", "moe", "pack"])
        m = _log_int(rng, 1, 64)
        act = rng.choice(["f32", "w4a8"])
        kind = rng.choice(["q4g64", "q8g64", "g256sf"] if act == "w4a8" else ["q4g64", "q8g64", "q4g32h", "qng64"])
        bits = {"q8g64": 8, "qng64": rng.randint(2, 15)}.get(kind, 4)
        unit = 256 if kind == "g256sf" else 64
        if call == "linear":
            rows = ",".join(str(_log_int(rng, 200, 14336)) for _ in range(rng.choice([1, 2, 3])))
            c = dict(call=call, kind=kind, bits=bits, act=act, rows=rows, cols=_width(rng, 512, 14336, unit), m=m)
        elif call == "mlp":
            c = dict(call=call, kind=kind, bits=bits, act=act, hidden=_width(rng, 768, 4096, unit),
                     inner=_width(rng, 2048, 14336, unit), m=m)
        elif call == "step":
            c = dict(call=call, kind=kind, bits=bits, act=act, mlp_kind=kind, mlp_bits=bits, hidden=_width(rng, 768, 4096, unit),
                     kv=_width(rng, 128, 1024, 64), inner=_width(rng, 2048, 14336, unit), layers=rng.randint(1, 12), m=m)
            if act == "f32" and rng.random() < 0.5:
                c["mlp_kind"], c["mlp_bits"] = rng.choice([("q4g32h", 4), ("q4g64", 4), ("q8g64", 8), ("qng64", rng.randint(2, 15))])
        elif call == "moe":
            e = rng.choice([8, 16, 32, 64])
            c = dict(call=call, fmt=rng.choice(["mixed", "mixed", "q4g64", "q4g64a"]), experts=e, top=rng.randint(1, min(e, 8)),
                     hidden=_width(rng, 512, 2880, 64), inner=_width(rng, 256, 2880, 64),
                     shared=rng.choice([0, _width(rng, 256, 2816, 64)]), m=m)
        else:
            kind = rng.choice(["q4g64", "q8g64", "qng64", "q4g32h", "g256sf"])
            c = dict(call=call, kind=kind, bits={"q8g64": 8, "qng64": rng.randint(5, 15)}.get(kind, 4),
                     rows=str(_log_int(rng, 256, 14336)), cols=_width(rng, 512, 4096, 256))
        if _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------- weights as byte layouts
def _wbytes(kind, bits, out, inn):
    """Bytes of one tensor's codes and scales."""
    n = out * inn
    return {"q4g64": n / 2 + n / 16, "q8g64": n + n / 16, "g256sf": n / 2 + n / 64 + n / 64, "qng64": n * bits / 8 + n / 16,
            "q4g32h": n / 2 + n / 16, "q4g64a": n / 2 + n / 8}[kind]


def _normal(gen, out, inn, sigma=0.02):
    return torch.randn((out, inn), generator=gen, device="cuda").mul_(sigma)


def _pack4(codes, out, inn):
    c = codes.reshape(out, inn // 2, 2).to(torch.uint8)
    return c[..., 0] | (c[..., 1] << 4)


def _round(w, group, top, lo, hi):
    g = w.reshape(w.shape[0], -1, group)
    s = g.abs().amax(-1).clamp_min_(1e-12) / top
    return torch.round(g / s[..., None]).clamp_(lo, hi), s


def _pack(kind, bits, w):
    """(packed, scales, sub) of fp32 weights in the engine's layout, on the device."""
    out, inn = w.shape
    if kind == "q4g64":
        q, s = _round(w, 64, 7.0, -8, 7)
        return _pack4(q + 8, out, inn), s, None
    if kind == "q4g32h":
        g = w.reshape(out, -1, 32)
        s = (g.abs().amax(-1) / 7.0).half()
        q = torch.round(g / s.float().clamp_min(1e-7)[..., None]).clamp_(-8, 7)
        return _pack4(q + 8, out, inn), s, None
    if kind == "q8g64":
        q, s = _round(w, 64, 127.0, -127, 127)
        return q.reshape(out, inn).to(torch.int8), s, None
    if kind == "g256sf":
        need = w.reshape(out, -1, 4, 64).abs().amax(-1) / 7.0                     # [out][in/256][4]
        super_ = need.amax(-1).clamp_min_(1e-12)
        sub = torch.ceil(need / super_[..., None] * 63.0).clamp_(1, 63)
        eff = super_[..., None] * sub / 63.0
        q = torch.round(w.reshape(out, -1, 4, 64) / eff[..., None]).clamp_(-8, 7)
        return _pack4(q + 8, out, inn), super_, sub.to(torch.uint8).reshape(out, -1)
    if kind == "qng64":
        half = 1 << (bits - 1)
        q, s = _round(w, 64, float(half - 1), -half, half - 1)
        u = (q + half).to(torch.int32).reshape(out, -1, 8, 8)                     # bit p % 8 of byte p / 8
        place = (1 << torch.arange(8, device=w.device, dtype=torch.int32))
        planes = [(((u >> j) & 1) * place).sum(-1).to(torch.uint8) for j in range(bits)]
        return torch.stack(planes, dim=2).reshape(out, -1), s, None
    g = w.reshape(out, -1, 64)                                                    # q4g64a: nib * s + b
    b = g.amin(-1)
    s = ((g.amax(-1) - b) / 15.0).clamp_min_(1e-12)
    q = torch.round((g - b[..., None]) / s[..., None]).clamp_(0, 15)
    return _pack4(q, out, inn), s, b


def _decode(kind, bits, packed, scales, sub, out, inn):
    """The weights that these bytes stand for, in 64 bits."""
    if kind == "q8g64":
        return (packed.double().reshape(out, -1, 64) * scales.double()[..., None]).reshape(out, inn)
    if kind == "qng64":
        p = packed.reshape(out, -1, bits, 8, 1).int()
        place = torch.arange(8, device=p.device, dtype=torch.int32)
        weight = (1 << torch.arange(bits, device=p.device, dtype=torch.int32)).reshape(1, 1, bits, 1, 1)
        u = (((p >> place) & 1) * weight).sum(2)
        return ((u.double().reshape(out, -1, 64) - (1 << (bits - 1))) * scales.double()[..., None]).reshape(out, inn)
    nib = torch.stack([packed & 15, packed >> 4], dim=-1).reshape(out, inn).double()
    if kind == "q4g64a":
        return (nib.reshape(out, -1, 64) * scales.double()[..., None] + sub.double()[..., None]).reshape(out, inn)
    if kind == "g256sf":
        eff = scales.double()[..., None] * sub.reshape(out, -1, 4).double() / 63.0
        return ((nib.reshape(out, -1, 4, 64) - 8) * eff[..., None]).reshape(out, inn)
    group = 32 if kind == "q4g32h" else 64
    return ((nib.reshape(out, -1, group) - 8) * scales.double()[..., None]).reshape(out, inn)


def _host(t):
    return None if t is None else t.contiguous().cpu().numpy()


class _Weights:
    """The weights of a case in the order in which it uses them: bound on the device, or decoded."""

    def __init__(self, gen, ctx=None):
        self.gen, self.ctx, self.owned = gen, ctx, []

    def one(self, kind, bits, out, inn):
        p, s, sub = _pack(kind, bits, _normal(self.gen, out, inn))
        if self.ctx is None:
            return _decode(kind, bits, p, s, sub, out, inn)
        p, s, sub = _host(p), _host(s), _host(sub)
        t = self.ctx.bind(KINDS[kind], p, s.view("uint16") if kind == "q4g32h" else s, out, inn, bits=bits, sub=sub)
        self.owned.append(t)
        return t

    def stack(self, formats, out, inn):
        each = [self.one(k, b, out, inn) for k, b in formats]
        if self.ctx is None:
            return each
        del self.owned[-len(each):]                       # the stack owns its experts
        t = self.ctx.experts_from_tensors(each)
        self.owned.append(t)
        return t


# -------------------------------------------------------------------------------------- the programs
class _State:
    graph = None

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.graph = None
            for t in self.weights.owned:
                t.free()
            self.ctx.close()
        except Exception:
            pass


_STREAM = None


def _stream():
    """The stream that the program queues its work on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def _experts(case, seed):
    """The formats of a routed layer's experts, and of its shared experts."""
    if case["fmt"] != "mixed":
        return [(case["fmt"], 4)] * case["experts"], (case["fmt"] if case["fmt"] != "q4g64a" else "q4g64", 4)
    rng = random.Random(seed)
    return [rng.choice(MIXED) for _ in range(case["experts"])], rng.choice(MIXED)


def _layer_rows(case):
    return [case["hidden"], case["kv"], case["kv"]]


def _build(case, seed, ctx):
    """The inputs and weights of a case: what `prepare` binds and what `exact` decodes."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w, s = _Weights(gen, ctx), _State()
    s.case, s.weights, s.ctx = case, w, ctx
    call, m = case["call"], case.get("m", 1)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda")  # noqa: E731
    if call == "linear":
        s.rows = [int(r) for r in case["rows"].split(",")]
        s.x = rand(m, case["cols"])
        s.w = [w.one(case["kind"], case["bits"], r, case["cols"]) for r in s.rows]
        s.y = [torch.empty((m, r), device="cuda") for r in s.rows]
    elif call == "mlp":
        h, i = case["hidden"], case["inner"]
        s.x = rand(m, h)
        s.w = [w.one(case["kind"], case["bits"], o, k) for o, k in ((i, h), (i, h), (h, i))]
        s.h, s.y = torch.empty((m, i), device="cuda"), torch.empty((m, h), device="cuda")
    elif call == "step":
        h, i, n = case["hidden"], case["inner"], case["layers"]
        s.x = [[rand(m, h) for _ in range(3)] for _ in range(n)]                 # what q/k/v, o and the MLP block read
        a, f = (case["kind"], case["bits"]), (case["mlp_kind"], case["mlp_bits"])
        s.w = []
        for _ in range(n):
            qkv = [w.one(*a, r, h) for r in _layer_rows(case)]
            s.w.append((qkv, w.one(*a, h, h), [w.one(*f, o, k) for o, k in ((i, h), (i, h), (h, i))]))
        s.q, s.k, s.v = (torch.empty((n, m, r), device="cuda") for r in _layer_rows(case))
        s.o, s.y = torch.empty((n, m, h), device="cuda"), torch.empty((n, m, h), device="cuda")
    elif call == "moe":
        h, i, sh = case["hidden"], case["inner"], case["shared"]
        formats, shared = _experts(case, seed)
        s.x = rand(m, h)
        s.router = rand(case["experts"], h) / h ** 0.5                            # N(0, 1) logits
        s.w = [w.stack(formats, o, k) for o, k in ((i, h), (i, h), (h, i))]
        s.sh = [w.one(*shared, o, k) for o, k in ((sh, h), (sh, h), (h, sh))] if sh else None
        s.y = torch.empty((m, h), device="cuda")
    else:
        s.x = _normal(gen, int(case["rows"]), case["cols"])
        s.y = torch.empty_like(s.x)
    return s


def _issue(s):
    """The calls of one pass, queued on the context's stream."""
    case, ctx = s.case, s.ctx
    call = case["call"]
    act = ACTS[case["act"]] if "act" in case else None
    if call == "linear":
        if len(s.w) == 1:
            ctx.matmul(s.w[0], s.x, s.y[0], act=act)
        else:
            ctx.matmul_group(s.w, s.x, s.y, act=act)
    elif call == "mlp":
        ctx.mlp(*s.w, s.x, s.y, act=act, h_dev=s.h)
    elif call == "step":
        for n, (qkv, o, mlp) in enumerate(s.w):
            ctx.matmul_group(qkv, s.x[n][0], [s.q[n], s.k[n], s.v[n]], act=act)
            ctx.matmul(o, s.x[n][1], s.o[n], act=act)
            ctx.mlp(*mlp, s.x[n][2], s.y[n], act=act)
    elif call == "moe":
        ctx.moe_layer(s.router, *s.w, s.sh, s.x, case["top"], s.y)
    else:
        t = ctx.quantize(KINDS[case["kind"]], s.x, bits=case["bits"])
        ctx.dequant(t, 0, s.x.shape[0], s.y)
        t.free()


def prepare(case, seed):
    stream = _stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s = _build(case, seed, B.Context(0, stream.cuda_stream))
        if case["call"] == "step":
            _issue(s)                                                             # sizes the context's scratch
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                _issue(s)
            s.graph = graph
    torch.cuda.synchronize()
    return s


def run(s):
    if s.graph is not None:
        s.graph.replay()
        return {"q": s.q, "k": s.k, "v": s.v, "o": s.o, "y": s.y}
    _issue(s)
    return {"h": s.h, "y": s.y} if s.case["call"] == "mlp" else s.y


# ------------------------------------------------------------------------ what a pass cannot do without
def _products(case):
    """(kind, bits, out, in, columns) of every product of a pass."""
    call, m = case["call"], case.get("m", 1)
    if call == "linear":
        return [(case["kind"], case["bits"], int(r), case["cols"], m) for r in case["rows"].split(",")]
    if call in ("mlp", "step"):
        h, i = case["hidden"], case["inner"]
        f = (case["kind"], case["bits"]) if call == "mlp" else (case["mlp_kind"], case["mlp_bits"])
        block = [(*f, i, h, m), (*f, i, h, m), (*f, h, i, m)]
        if call == "mlp":
            return block
        a = (case["kind"], case["bits"])
        return ([(*a, r, h, m) for r in _layer_rows(case)] + [(*a, h, h, m)] + block) * case["layers"]
    return []


def work(case):
    call, m = case["call"], case.get("m", 1)
    if call == "pack":
        n = int(case["rows"]) * case["cols"]
        return {"bytes": 8.0 * n + 2 * _wbytes(case["kind"], case["bits"], int(case["rows"]), case["cols"]), "flops": 4.0 * n}
    if call == "moe":
        e, h, i, sh, k = (case[n] for n in ("experts", "hidden", "inner", "shared", "top"))
        touched = e * (1.0 - (1.0 - k / e) ** m)                                  # expected, for independent tokens
        # the mean over the formats that experts are drawn from
        formats = MIXED if case["fmt"] == "mixed" else [(case["fmt"], 4)]
        each = sum(_wbytes(f, b, 1, 3 * h * i) for f, b in formats) / len(formats)
        formats = [("q4g64", 4)] if case["fmt"] == "q4g64a" else formats
        common = sum(_wbytes(f, b, 1, 3 * h * sh) for f, b in formats) / len(formats)
        return {"bytes": touched * each + common + 4 * e * h + 8 * m * h, "flops": 6.0 * m * (k * h * i + h * sh) + 2.0 * m * e * h}
    products = _products(case)
    data = sum(_wbytes(k, b, o, i) for k, b, o, i, _ in products)
    if call == "linear":
        io = 4 * m * (case["cols"] + sum(p[2] for p in products))
    elif call == "mlp":
        io = 4 * m * (2 * case["hidden"] + case["inner"])
    else:
        io = 4 * m * case["layers"] * (5 * case["hidden"] + 2 * case["kv"])
    return {"bytes": data + io, "flops": sum(2.0 * o * i * n for _, _, o, i, n in products)}


def _cost(case):
    """Bytes and operations of a case in one figure, for the limit on drawn cases (wide codes cost more operations)."""
    w = work(case)
    return w["bytes"] / 2e12 + w["flops"] / 3e13 * max(1.0, case.get("bits", 8) / 8.0, case.get("mlp_bits", 8) / 8.0)


def tolerance(case):
    if case["call"] == "pack":
        return "exact"                                     # whole codes and scales: one right answer
    if case.get("act") == "w4a8":
        # integer dot products and an fp32 sum over the groups (3e-7 from 64 bits); in an MLP block a
        # last-bit change of h moves some of its int8 codes by one (1e-4)
        return {"rel": 1.2e-6} if case["call"] == "linear" else {"rel": 4e-4}
    return {"rel": 2.4e-6}                                 # 1.6e-7 to 5.6e-7 from 64 bits


# --------------------------------------------------------------------------------------- in 64 bits
def _over(t, v):
    """t / v as an fp32 division (a Python divisor becomes a product with 1 / v)."""
    return t / torch.full_like(t, v)


def _quantized(x, group):
    """fp32 rows as the int8 activations that the W4A8 products read, in 64 bits: code * scale."""
    g = x.float().reshape(x.shape[0], -1, group)
    s = _over(g.abs().amax(-1, keepdim=True).clamp_min(1e-8), 127.0)
    p = g * (1.0 / s)
    q = torch.trunc(p + torch.where(p >= 0, 0.5, -0.5)).clamp_(-128, 127)
    return (q.double() * s.double()).reshape(x.shape)


def _exact_product(case, kind, w, x):
    if case.get("act") == "w4a8":
        x = _quantized(x, 256 if kind == "g256sf" else 64)
    return x.double() @ w.t()


def _silu(g):
    return g / (1.0 + torch.exp(-g))


def _exact_mlp(case, kind, w, x):
    h = _silu(_exact_product(case, kind, w[0], x)) * _exact_product(case, kind, w[1], x)
    return h, _exact_product(case, kind, w[2], h)


def _exact_pack(case, w):
    """The packers' arithmetic: the scales and codes in fp32 as they are stored, the values in 64 bits."""
    kind, bits, (out, inn) = case["kind"], case["bits"], w.shape
    if kind != "q4g64":
        return None
    g = w.reshape(out, -1, 64)
    s = _over(g.abs().amax(-1), 7.0)
    s = torch.where(s < 1e-12, torch.ones_like(s), s)
    inv, err, q = 1.0 / s, torch.zeros_like(s), torch.empty_like(g)
    for p in range(64):                                    # error feedback runs along the group
        x = g[..., p] + err
        c = torch.round(x * inv).clamp_(-8, 7)
        err = x - c * s
        q[..., p] = c
    return (q.double() * s.double()[..., None]).reshape(out, inn)


def exact(case, seed):
    s = _build(case, seed, None)
    call = case["call"]
    if call == "linear":
        return [_exact_product(case, case["kind"], w, s.x) for w in s.w]
    if call == "mlp":
        h, y = _exact_mlp(case, case["kind"], s.w, s.x)
        return {"h": h, "y": y}
    if call == "step":
        got = {n: [] for n in "qkvoy"}
        for (qkv, o, mlp), x in zip(s.w, s.x):
            for n, w in zip("qkv", qkv):
                got[n].append(_exact_product(case, case["kind"], w, x[0]))
            got["o"].append(_exact_product(case, case["kind"], o, x[1]))
            got["y"].append(_exact_mlp(case, case["mlp_kind"], mlp, x[2])[1])
        return {n: torch.stack(v) for n, v in got.items()}
    if call == "moe":
        x = s.x.double()
        p = torch.softmax(x @ s.router.double().t(), -1)
        weight, chosen = p.topk(case["top"], -1)
        y = torch.zeros_like(x)
        for e in range(case["experts"]):
            t, k = (chosen == e).nonzero(as_tuple=True)
            if len(t):
                h = _silu(x[t] @ s.w[0][e].t()) * (x[t] @ s.w[1][e].t())
                y[t] += weight[t, k][:, None] * (h @ s.w[2][e].t())
        if s.sh:
            y += (_silu(x @ s.sh[0].t()) * (x @ s.sh[1].t())) @ s.sh[2].t()
        return y
    return _exact_pack(case, s.x)
