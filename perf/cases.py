"""The workloads this library is timed on: one model layer's worth of each path, from single-token decode to prefill.

`kind` names the path, `T` the tokens (rows) of the step, `layers` how many layers' weights one pass goes through (a
step of a model touches each layer's weights once, so they come from HBM and not from a cache), `graph` whether the
program captured those layers as one HIP graph (as a serving loop does with its short steps) or enqueues them.

- moe: router logits -> softmax top-K -> MXFP4 experts (w1 / w3 + SwiGLU, w2) -> combine, one uh_mx_moe_forward.
- dense: act_quant + block-scaled fp8 GEMM; scales "e8m0" (powers of two, 1x128 / 128x128) or "f32" (the fused entry
  point for up to 16 rows, as a decode loop calls it).
- shared: rmsnorm + act_quant, the shared expert's gate / up GEMV with SwiGLU and requantization, its down projection.
- grouped: the grouped "mgk,grk->mgr" projection of bf16 rows by fp8 weights.
"""
import functools
import math

import numpy as np
import torch

from unholy_amd import call
from unholy_amd.device import Graph, Stream

TOPK = 6
LIMIT = 10.0
EPS = 1e-6
ROUTER_SKEW = 0.5  # standard deviation of the experts' popularity (a bias on the logits)


def listed():
    return [
        # Single-user generation: one token, 6 of 256 experts; latency and launches.
        {"name": "moe_decode_1", "kind": "moe", "T": 1, "E": 256, "D": 4096, "I": 2048, "layers": 4, "graph": True},
        # A small decode batch, the benchmark's headline step.
        {"name": "moe_decode_8", "kind": "moe", "T": 8, "E": 256, "D": 4096, "I": 2048, "layers": 4, "graph": True},
        # Speculative verification of a batch, or a larger decode batch.
        {"name": "moe_verify_64", "kind": "moe", "T": 64, "E": 256, "D": 4096, "I": 2048, "layers": 1, "graph": False},
        # Decode rows and a short prompt in one step; a few rows per expert.
        {"name": "moe_mixed_203", "kind": "moe", "T": 203, "E": 256, "D": 4096, "I": 2048, "layers": 1, "graph": False},
        # A prompt (or prompt chunk) of ordinary length.
        {"name": "moe_chunk_1000", "kind": "moe", "T": 1000, "E": 256, "D": 4096, "I": 2048, "layers": 1,
         "graph": False},
        # The largest prefill chunk.
        {"name": "moe_prefill_4096", "kind": "moe", "T": 4096, "E": 256, "D": 4096, "I": 2048, "layers": 1,
         "graph": False},
        # One token through a projection with fp32 block scales.
        {"name": "dense_decode_1", "kind": "dense", "T": 1, "N": 4096, "K": 4096, "scales": "f32", "layers": 16,
         "graph": True},
        # A verify batch through a projection with power-of-two block scales.
        {"name": "dense_verify_64", "kind": "dense", "T": 64, "N": 4096, "K": 4096, "scales": "e8m0", "layers": 16,
         "graph": True},
        # A short prompt through the same.
        {"name": "dense_mixed_300", "kind": "dense", "T": 300, "N": 4096, "K": 4096, "scales": "e8m0", "layers": 8,
         "graph": False},
        # The largest prefill chunk through a projection.
        {"name": "dense_prefill_4096", "kind": "dense", "T": 4096, "N": 4096, "K": 4096, "scales": "f32", "layers": 1,
         "graph": False},
        # The shared expert of a small decode batch, behind its norm.
        {"name": "shared_decode_4", "kind": "shared", "T": 4, "D": 4096, "I": 2048, "layers": 8, "graph": True},
        # The grouped output projection of a decode batch.
        {"name": "grouped_decode_32", "kind": "grouped", "T": 32, "G": 8, "N": 1024, "K": 4096, "layers": 8,
         "graph": True},
    ]


def draw(rng):
    def tokens(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))

    kind = rng.choice(["moe"] * 5 + ["dense"] * 4 + ["shared"] + ["grouped"] * 2)
    if kind == "moe":
        e, d, i = rng.choice([(256, 4096, 2048)] * 3 + [(32, 4096, 2048), (64, 2048, 1024)])
        t = tokens(1, 4096)
        return {"kind": kind, "T": t, "E": e, "D": d, "I": i, "layers": 4 if t <= 16 else 1, "graph": t <= 16}
    if kind == "dense":
        n, k = rng.choice([(4096, 4096)] * 2 + [(8192, 1024), (32768, 1024), (4096, 2048), (2048, 4096), (4096, 8192)])
        t = tokens(1, 4096)
        layers = 1 if t > 1024 else 8 if t > 64 else 16
        return {"kind": kind, "T": t, "N": n, "K": k, "scales": rng.choice(["f32", "e8m0"]), "layers": layers,
                "graph": t <= 64}
    if kind == "shared":
        d, i = rng.choice([(4096, 2048), (2048, 1024)])
        return {"kind": kind, "T": tokens(1, 32), "D": d, "I": i, "layers": 8, "graph": True}
    t = tokens(1, 4096)
    return {"kind": kind, "T": t, "G": rng.choice([4, 8]), "N": 1024, "K": rng.choice([2048, 4096]),
            "layers": 1 if t > 1024 else 8, "graph": t <= 64}


# ---- inputs ----------------------------------------------------------------------------------------------------------
_stream = None


def stream():
    """The program's one stream for captured work."""
    global _stream
    if _stream is None:
        _stream = Stream()
    return _stream


def normal(gen, shape, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)


def codes(gen, shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, generator=gen, device="cuda")


def block_amax(w, rows, cols):
    """Largest magnitude of each rows x cols block of w [N, K]."""
    n, k = w.shape
    return w.abs().view(n // rows, rows, k // cols, cols).amax(dim=(1, 3)).clamp_min(1e-4)


def spread(s, rows, cols):
    return s.repeat_interleave(rows, 0).repeat_interleave(cols, 1)


def pow2_scale(amax, top):
    """e8m0 exponents of the smallest power of two at or above amax / top."""
    bits = (amax * (1.0 / top)).view(torch.int32)
    return ((bits >> 23) + ((bits & 0x7FFFFF) != 0).to(torch.int32)).to(torch.uint8)


def pow2(s):
    return torch.ldexp(torch.ones_like(s, dtype=torch.float32), s.to(torch.int32) - 127)


def quantized(x, rows, e8m0):
    """fp8 codes and scales of x [N, K] per rows x 128 block."""
    amax = block_amax(x.float(), rows, 128)
    s = pow2_scale(amax, 448.0) if e8m0 else amax * (1.0 / 448.0)
    f = pow2(s) if e8m0 else s
    return (x.float() / spread(f, rows, 128)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), s


def fp8_weight(gen, n, k, e8m0=True):
    """A projection's weights as a checkpoint holds them: fp8 codes and one scale per 128 x 128 block."""
    return quantized(torch.randn((n, k), generator=gen, device="cuda") * 0.02, 128, e8m0)


def expert_bytes(d, i):
    return 3 * (d * i // 2 + d * i // 32)


def expert_weights(gen, e, d, i):
    """E experts of MXFP4 weights, tile-major, one slot per expert (w1, w3, w2: codes, then scales), and the device
    table of their addresses."""
    cb, sb = d * i // 2, d * i // 32
    slots = codes(gen, (e, expert_bytes(d, i)))
    base = slots.data_ptr() + np.arange(e, dtype=np.int64) * slots.shape[1]
    table = []
    for m in range(3):
        at = m * (cb + sb)
        slots[:, at + cb:at + cb + sb] = torch.randint(119, 126, (e, sb), dtype=torch.uint8, generator=gen,
                                                       device="cuda")
        table += [base + at, base + at + cb]
    return slots, torch.from_numpy(np.concatenate(table)).cuda()


def inputs(c, seed):
    """One dict per layer: activations and weights."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    out = []
    for _ in range(c["layers"]):
        if c["kind"] == "moe":
            slots, table = expert_weights(gen, c["E"], c["D"], c["I"])
            skew = torch.randn((1, c["E"]), generator=gen, device="cuda") * ROUTER_SKEW
            out.append({"x": normal(gen, (c["T"], c["D"])), "slots": slots, "table": table,
                        "logits": torch.randn((c["T"], c["E"]), generator=gen, device="cuda") + skew})
        elif c["kind"] == "dense":
            w, sw = fp8_weight(gen, c["N"], c["K"], c["scales"] == "e8m0")
            out.append({"x": normal(gen, (c["T"], c["K"])), "w": w, "sw": sw})
        elif c["kind"] == "shared":
            d, i = c["D"], c["I"]
            out.append({"x": normal(gen, (c["T"], d)), "norm": normal(gen, (d,), 0.2) + 1.0,
                        "gate": fp8_weight(gen, i, d), "up": fp8_weight(gen, i, d), "down": fp8_weight(gen, d, i)})
        else:
            w, sw = fp8_weight(gen, c["G"] * c["N"], c["K"])
            out.append({"x": normal(gen, (c["T"], c["G"], c["K"])), "w": w, "sw": sw})
    return out


# ---- the calls -------------------------------------------------------------------------------------------------------
def moe_layer(c, y, st):
    t, e, d, i = c["T"], c["E"], c["D"], c["I"]
    call("uh_mx_moe_forward", y["x"].data_ptr(), y["logits"].data_ptr(), t, TOPK, e, d, i, y["table"].data_ptr(), LIMIT,
         y["ws"].data_ptr(), y["ws"].numel(), y["out"].data_ptr(), None, None, st)


def dense_layer(c, y, st):
    t, n, k = c["T"], c["N"], c["K"]
    x, w, sw, out = (y[f].data_ptr() for f in ("x", "w", "sw", "out"))
    if c["scales"] == "f32" and t <= 16 and t * k <= 120 * 1024:
        call("uh_gemm_fp8_f32s_x", x, k, w, sw, out, n, t, n, k, st)
        return
    q, s = y["q"].data_ptr(), y["s"].data_ptr()
    if c["scales"] == "f32":
        call("uh_act_quant_fp8_f32s", x, k, q, s, t, k, 128, st)
        call("uh_gemm_fp8_f32s", q, s, w, sw, out, n, t, n, k, st)
    else:
        call("uh_act_quant_fp8", x, k, q, s, t, k, 128, st)
        call("uh_gemm_w8a8_wmma", q, s, w, sw, out, n, t, n, k, st)


def shared_layer(c, y, st):
    t, d, i = c["T"], c["D"], c["I"]
    p = {f: y[f].data_ptr() for f in ("x", "norm", "normed", "q", "s", "g", "u", "hq", "hs", "counters", "out")}
    call("uh_rmsnorm_quant_slices", p["x"], d, p["norm"], p["normed"], d, p["q"], p["s"], t, d, EPS, None, st)
    (wg, sg), (wu, su), (wd, sd) = y["gate"], y["up"], y["down"]
    call("uh_gemv_w8a8_glu", p["q"], p["s"], wg.data_ptr(), sg.data_ptr(), p["g"], i, wu.data_ptr(), su.data_ptr(),
         p["u"], i, i, t, d, LIMIT, p["hq"], p["hs"], p["counters"], st)
    call("uh_gemv_w8a8", p["hq"], p["hs"], wd.data_ptr(), sd.data_ptr(), p["out"], d, t, d, i, st)


def grouped_layer(c, y, st):
    call("uh_gemm_grouped_fp8w_wmma", y["x"].data_ptr(), y["w"].data_ptr(), y["sw"].data_ptr(), y["out"].data_ptr(),
         c["T"], c["G"], c["N"], c["K"], st)


LAYER = {"moe": moe_layer, "dense": dense_layer, "shared": shared_layer, "grouped": grouped_layer}


def prepare(case, seed):
    c, t = case, case["T"]
    layers = inputs(c, seed)

    def new(*shape, dtype=torch.bfloat16):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    u8, f32 = torch.uint8, torch.float32
    if c["kind"] == "moe":  # one workspace serves every layer of a program
        ws = torch.zeros(call("uh_mx_moe_workspace_size", t, TOPK, c["E"], c["D"], c["I"]), dtype=u8, device="cuda")
        for y in layers:
            y["ws"], y["out"] = ws, new(t, c["D"])
    elif c["kind"] == "dense":
        q = new(t, c["K"], dtype=u8)
        s = new(t, c["K"] // 128, dtype=f32 if c["scales"] == "f32" else u8)
        for y in layers:
            y["q"], y["s"], y["out"] = q, s, new(t, c["N"])
    elif c["kind"] == "shared":
        d, i = c["D"], c["I"]
        for y in layers:
            y.update(normed=new(t, d), q=new(t, d, dtype=u8), s=new(t, d // 128, dtype=u8), g=new(t, i), u=new(t, i),
                     hq=new(t, i, dtype=u8), hs=new(t, i // 128, dtype=u8), out=new(t, d),
                     counters=new(i // 128, dtype=torch.int32))
    else:
        for y in layers:
            y["out"] = new(t, c["G"], c["N"])
    state = {"case": c, "layers": layers, "graph": None}
    if c["graph"]:
        torch.cuda.synchronize()

        def step():
            for y in layers:
                LAYER[c["kind"]](c, y, stream().handle)

        step()
        stream().synchronize()
        state["graph"] = Graph(stream(), step)
    return state


def run(state):
    c = state["case"]
    if state["graph"] is not None:
        state["graph"].launch()
    else:
        for y in state["layers"]:
            LAYER[c["kind"]](c, y, None)
    if c["kind"] == "shared":
        return [(y["normed"], y["out"]) for y in state["layers"]]
    return [y["out"] for y in state["layers"]]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
@functools.lru_cache(None)
def experts_hit(t, e):
    """Distinct experts that t tokens pick, on average."""
    rng = np.random.default_rng(0)
    hit = []
    for _ in range(8 if t < 512 else 2):
        logits = rng.standard_normal((t, e)) + rng.standard_normal((1, e)) * ROUTER_SKEW
        hit.append(len(np.unique(np.argpartition(-logits, TOPK - 1, axis=1)[:, :TOPK])))
    return sum(hit) / len(hit)


def work(case):
    c, t, n = case, case["T"], case["layers"]
    if c["kind"] == "moe":
        e, d, i = c["E"], c["D"], c["I"]
        return {"bytes": n * (experts_hit(t, e) * expert_bytes(d, i) + t * (4 * d + 4 * e)),
                "flops": n * 6.0 * t * TOPK * d * i}
    if c["kind"] == "dense":
        sb = 4 if c["scales"] == "f32" else 1
        return {"bytes": n * (c["N"] * c["K"] * (1 + sb / 16384) + 2 * t * (c["N"] + c["K"])),
                "flops": n * 2.0 * t * c["N"] * c["K"]}
    if c["kind"] == "shared":
        d, i = c["D"], c["I"]
        return {"bytes": n * (3 * d * i * (1 + 1 / 16384) + 2 * d + 6 * t * d), "flops": n * 6.0 * t * d * i}
    g = c["G"]
    return {"bytes": n * (g * c["N"] * c["K"] * (1 + 1 / 16384) + 2 * t * g * (c["N"] + c["K"])),
            "flops": n * 2.0 * t * g * c["N"] * c["K"]}


def tolerance(case):
    """bf16 outputs of sums in 32 bits, from operands quantized alike: another order of summation rounds some outputs to
    the next bf16 value. Where an fp8 requantization stands between two products (moe, shared), an intermediate value
    that rounds the other way moves one fp8 code, and with it a whole output row a little."""
    if case["kind"] in ("moe", "shared"):
        return {"rel": 4e-3, "max": 0.1}
    return {"rel": 2e-3, "max": 0.02}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------
E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def scale64(s):
    return (pow2(s) if s.dtype == torch.uint8 else s).double()


def fp8_values(q, s, rows):
    return q.double() * spread(scale64(s), rows, 128)


def mx_values(w, s, n, k):
    """[N, K] of one tile-major MXFP4 matrix: 64-input slabs of 16-output tiles, low nibble first, a scale per 32."""
    w = w.view(k // 64, n // 16, 16, 32).permute(1, 2, 0, 3).reshape(n, k // 2).long()
    s = s.view(k // 64, n // 16, 16, 2).permute(1, 2, 0, 3).reshape(n, k // 32)
    lut = torch.tensor(E2M1, dtype=torch.float64, device=w.device)
    return torch.stack((lut[w & 15], lut[w >> 4]), -1).view(n, k) * scale64(s).repeat_interleave(32, 1)


def silu_mul(g, u):
    g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
    return g / (1.0 + torch.exp(-g)) * u


def requantized(x):
    """Values after rounding to bf16 and to fp8 with a power-of-two scale per 128, as the path defines its operands."""
    q, s = quantized(x.to(torch.bfloat16), 1, True)
    return fp8_values(q, s, 1)


def moe_exact(c, y):
    t, e, d, i = c["T"], c["E"], c["D"], c["I"]
    top = torch.topk(y["logits"].double(), TOPK, dim=1)
    weight = torch.softmax(top.values, dim=1)
    x = requantized(y["x"])
    out = torch.zeros((t, d), dtype=torch.float64, device="cuda")
    cb, sb = d * i // 2, d * i // 32
    for j in torch.unique(top.indices).tolist():
        rows, pick = torch.nonzero(top.indices == j, as_tuple=True)
        m = [mx_values(y["slots"][j, a:a + cb], y["slots"][j, a + cb:a + cb + sb], *shape)
             for a, shape in ((0, (i, d)), (cb + sb, (i, d)), (2 * (cb + sb), (d, i)))]
        g, u = ((x[rows] @ w.t().contiguous()).to(torch.bfloat16).double() for w in m[:2])
        h = requantized(silu_mul(g, u) * weight[rows, pick][:, None])
        out.index_add_(0, rows, h @ m[2].t().contiguous())
    return out


def shared_exact(c, y):
    x, w = y["x"].double(), y["norm"].double()
    normed = w * (x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS)).to(torch.float32).double()
    a = requantized(normed)
    g, u = ((a @ fp8_values(*y[f], 128).t().contiguous()).to(torch.bfloat16).double() for f in ("gate", "up"))
    return normed, requantized(silu_mul(g, u)) @ fp8_values(*y["down"], 128).t().contiguous()


def exact(case, seed):
    c, out = case, []
    for y in inputs(c, seed):
        if c["kind"] == "moe":
            out.append(moe_exact(c, y))
        elif c["kind"] == "dense":
            q, s = quantized(y["x"], 1, c["scales"] == "e8m0")
            out.append(fp8_values(q, s, 1) @ fp8_values(y["w"], y["sw"], 128).t().contiguous())
        elif c["kind"] == "shared":
            out.append(shared_exact(c, y))
        else:
            w = fp8_values(y["w"], y["sw"], 128).view(c["G"], c["N"], c["K"])
            out.append(torch.stack([y["x"][:, g].double() @ w[g].t().contiguous() for g in range(c["G"])], 1))
    return out
