"""The work that users of dsk_moe have it do, as cases that can be timed and compared.

A case is one call of a public entry point: a MoE layer (``MoELayer``,
``moe_layer``) at decode, batched decode, a short prompt or a long one, a step of
a layer stack (``MoELayer.forward_residual``), or the requantisation of expert
weights (``fp4_dequant``, ``q3_quantize``).  Two geometries are in use: "full"
(hidden 4096, 256 experts, top-8, intermediate 2048, sigmoid gate, scale 2.5: the
benchmark's) and "ref" (hidden 5120, 384 experts, top-6, intermediate 2304,
sqrt-softplus gate, scale 1.5: DeepSeek-V4.1-Flash's own).

Expert weights are drawn as codes and scales with the distribution that N(0, 0.02)
weights quantise to; ``exact`` decodes the same bytes with plain torch and computes
the layer in float64.
"""

from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "deepseeker-v4.1_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import dsk_moe  # noqa: E402

GEOMETRY = {
    "full": dict(H=4096, E=256, k=8, I=2048, Is=2048, score="sigmoid", scale=2.5),
    "ref": dict(H=5120, E=384, k=6, I=2304, Is=2304, score="sqrtsoftplus", scale=1.5),
}
LIMIT = 10.0
EPS = 1e-6
DEV = "cuda"


def _layer(name, geo, quant, tokens, zipf=False, dtype="bf16", call="layer"):
    return {"name": name, "kind": call, "geo": geo, "quant": quant, "tokens": tokens, "zipf": zipf, "dtype": dtype}


def listed():
    return [
        # one token of decode: the headline of the benchmark, all latency
        _layer("decode_fp4_1", "full", "fp4", 1),
        # a full decode batch
        _layer("batch_fp4_64", "full", "fp4", 64),
        # a short prompt: every expert is touched, few rows each
        _layer("chunk_fp4_200", "full", "fp4", 200),
        # a long prompt with a skewed router, as the benchmark's prefill
        _layer("prompt_fp4_4096", "full", "fp4", 4096, zipf=True),
        # 3-bit experts: a decode batch and a medium prompt
        _layer("batch_q3_16", "full", "q3", 16),
        _layer("prompt_q3_700", "full", "q3", 700, zipf=True),
        # the model's own geometry through the drop-in function: decode, a batch, a prompt
        _layer("ref_decode_fp4_1", "ref", "fp4", 1, call="drop_in"),
        _layer("ref_batch_fp4_24", "ref", "fp4", 24, call="drop_in"),
        _layer("ref_prompt_fp4_2000", "ref", "fp4", 2000, call="drop_in"),
        # a float32 stream (a caller that keeps its activations in float32)
        _layer("batch_f32_20", "full", "fp4", 20, dtype="f32"),
        # a two-token verify step inside a stack: residual add, norm and layer
        _layer("stack_step_q3_2", "full", "q3", 2, call="residual"),
        # offline requantisation of 8 experts' rows, FP4 to 3-bit
        {"name": "requant_8", "kind": "requant", "experts": 8, "rows": 2048, "cols": 4096},
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["full_fp4"] * 4 + ["ref_fp4"] * 3 + ["q3"] * 3 + ["f32", "residual", "requant"])
    if kind == "full_fp4":
        c = _layer("", "full", "fp4", log_int(1, 4096), zipf=rng.random() < 0.5)
    elif kind == "ref_fp4":
        c = _layer("", "ref", "fp4", log_int(1, 2000), call="drop_in")
    elif kind == "q3":
        # the 3-bit prompts stop where they would cost more than the longest listed prompt
        c = (_layer("", "full", "q3", log_int(1, 700), zipf=rng.random() < 0.5) if rng.random() < 0.6
             else _layer("", "ref", "q3", log_int(1, 64), call="drop_in"))
    elif kind == "f32":
        c = _layer("", rng.choice(["full", "ref"]), "fp4", log_int(1, 64), dtype="f32")
    elif kind == "residual":
        c = _layer("", rng.choice(["full", "ref"]), rng.choice(["fp4", "q3"]), log_int(1, 32), call="residual")
    else:
        # an odd number of rows, or the down role's shape
        rows, cols = rng.choice([(rng.randrange(1, 2300), 4096), (5120, 2304), (rng.randrange(1, 5000), 2048)])
        c = {"kind": "requant", "experts": rng.randint(1, 6), "rows": rows, "cols": cols}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
# E2M1 magnitudes by code; code 8 (negative zero) is never written by a quantiser.
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _normal_quantiles(n):
    u = (torch.arange(n, dtype=torch.float64) + 0.5) / n
    return math.sqrt(2.0) * torch.erfinv(2.0 * u - 1.0)


@functools.lru_cache(maxsize=None)
def _code_table(quant):
    """65536 random 16-bit words -> four codes, whose distribution is that of N(0, 0.02) weights."""
    z = _normal_quantiles(16)
    if quant == "fp4":
        # amax of 32 normals over 6 rounds up to 2^-7 or 2^-6: 0.02 is 2.56 or 1.28 steps
        mag = (z.abs() * 1.9)[:, None] - torch.tensor(_E2M1, dtype=torch.float64)[None, :]
        code = mag.abs().argmin(1)
        code = torch.where((z < 0) & (code > 0), code + 8, code)
        bits = 4
    else:
        code = torch.clamp(torch.round(3.5 + z * 1.46), 0, 7).long()   # 4.8 sigma over 7 steps
        bits = 3
    r = torch.arange(65536)
    word = sum(code[(r >> (4 * i)) & 15] << (bits * i) for i in range(4))
    return word.to(torch.int32).to(DEV)


def _words(g, shape, quant, chunk=1 << 26):
    """Random words of four codes: int32 tensor of `shape`."""
    n = math.prod(shape)
    out = torch.empty(n, dtype=torch.int32 if quant == "q3" else torch.int16, device=DEV)
    table = _code_table(quant)
    for a in range(0, n, chunk):
        b = min(n, a + chunk)
        r = torch.randint(0, 65536, (b - a,), generator=g, device=DEV, dtype=torch.int32)
        out[a:b] = table[r.long()].to(out.dtype)
    return out.view(shape)


def _fp4_role(g, E, N, K):
    codes = _words(g, (E, N, K // 4), "fp4").view(torch.uint8).view(E, N, K // 2)
    scales = torch.randint(120, 122, (E, N, K // 32), generator=g, device=DEV, dtype=torch.uint8)
    return codes, scales


def _q3_role(g, E, N, K):
    """Row-major 3-byte packs as a checkpoint holds them, with fp16 scale and bias per 64."""
    packs = torch.empty((E, N, K // 8, 3), dtype=torch.uint8, device=DEV)
    for e in range(0, E, 32):
        v = _words(g, (min(32, E - e), N, K // 8, 2), "q3")
        v = v[..., 0] | (v[..., 1] << 12)
        for i in range(3):
            packs[e:e + 32, :, :, i] = (v >> (8 * i)).to(torch.uint8)
    step = torch.rand((E, N, K // 64), generator=g, device=DEV) * 0.003 + 0.0122
    return packs.view(E, N, 3 * K // 8), step.half(), (-3.5 * step).half()


def _inputs(case, seed):
    """Everything a layer call takes, on the GPU: codes and scales as a checkpoint holds them."""
    c, T = GEOMETRY[case["geo"]], case["tokens"]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    H, E, I, Is = c["H"], c["E"], c["I"], c["Is"]
    role = _fp4_role if case["quant"] == "fp4" else _q3_role
    d = {"gate_w": torch.randn((E, H), generator=g, device=DEV) / math.sqrt(H)}
    if case["zipf"]:
        d["gate_b"] = torch.from_numpy(_zipf(E)).float().to(DEV)
    else:
        d["gate_b"] = torch.rand((E,), generator=g, device=DEV) * 0.2 - 0.1
    d["roles"] = {"w1": role(g, E, I, H), "w3": role(g, E, I, H), "w2": role(g, E, H, I)}
    d["shared"] = [(torch.randn(s, generator=g, device=DEV) * 0.02).bfloat16() for s in ((Is, H), (Is, H), (H, Is))]
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    d["x"] = torch.randn((T, H), generator=g, device=DEV).to(dt)
    if case["kind"] == "residual":
        d["d"] = torch.randn((T, H), generator=g, device=DEV).to(dt)
        d["gamma"] = torch.rand((H,), generator=g, device=DEV) + 0.5
    return d


def _zipf(E, s=1.1):
    p = np.arange(1, E + 1, dtype=np.float64) ** -s
    return np.log(p / p.sum())


def _requant_inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    return _fp4_role(g, case["experts"], case["rows"], case["cols"])


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    if case["kind"] == "requant":
        codes, scales = _requant_inputs(case, seed)
        return {"kind": "requant", "codes": codes, "scales": scales}
    c = GEOMETRY[case["geo"]]
    d = _inputs(case, seed)
    if case["quant"] == "q3":       # what the checkpoint loader does with row-major packs
        roles = {r: (dsk_moe.q3_repack(p), s, b) for r, (p, s, b) in d["roles"].items()}
    else:
        roles = d["roles"]
    bank = dsk_moe.ResidentBank(case["quant"], roles)
    shared = dsk_moe.SharedExpert(*d["shared"], limit=LIMIT)
    st = {"kind": case["kind"], "c": c, "x": d["x"], "bank": bank, "shared": shared,
          "gate_w": d["gate_w"], "gate_b": d["gate_b"]}
    if case["kind"] != "drop_in":
        st["layer"] = dsk_moe.MoELayer(d["gate_w"], d["gate_b"], bank, shared, c["k"], score_func=c["score"],
                                       route_scale=c["scale"], limit=LIMIT)
    if case["kind"] == "residual":
        st.update(d=d["d"], gamma=d["gamma"], bufs=[torch.empty_like(d["x"]) for _ in range(3)])
    return st


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["layer"](state["x"])
    if kind == "drop_in":
        c = state["c"]
        return dsk_moe.moe_layer(state["x"], state["gate_w"], state["gate_b"], state["bank"], state["shared"],
                                 top_k=c["k"], limit=LIMIT, score_func=c["score"], route_scale=c["scale"])
    if kind == "residual":
        h_out, x_out, out = state["bufs"]
        state["layer"].forward_residual(state["x"], state["d"], h_out, x_out, out, gamma=state["gamma"], eps=EPS)
        return h_out, x_out, out
    w = dsk_moe.fp4_dequant(state["codes"], state["scales"])
    return (w,) + tuple(dsk_moe.q3_quantize(w))


# ------------------------------------------------------------------ what a pass cannot do without
def _role_bytes(n, k, quant):
    return n * k // 2 + n * k // 32 if quant == "fp4" else n * k * 3 // 8 + n * k // 64 * 4


@functools.lru_cache(maxsize=None)
def _active(geo, tokens, zipf):
    """How many experts a batch touches: the router simulated on N(0, 1) logits."""
    c = GEOMETRY[geo]
    r = np.random.default_rng(1)
    z = r.standard_normal((tokens, c["E"]))
    s = 1.0 / (1.0 + np.exp(-z)) if c["score"] == "sigmoid" else np.sqrt(np.log1p(np.exp(z)))
    key = s + (_zipf(c["E"]) if zipf else r.uniform(-0.1, 0.1, c["E"]))
    return len(np.unique(np.argpartition(-key, c["k"] - 1, axis=1)[:, :c["k"]]))


def work(case):
    if case["kind"] == "requant":
        n = case["experts"] * case["rows"] * case["cols"]
        # FP4 in, the float32 weights and the 3-bit form out
        return {"bytes": n // 2 + n // 32 + 4 * n + n * 3 // 8 + n // 16, "flops": 0}
    c, T = GEOMETRY[case["geo"]], case["tokens"]
    H, I, Is, E, k = c["H"], c["I"], c["Is"], c["E"], c["k"]
    el = 4 if case["dtype"] == "f32" else 2
    expert = 2 * _role_bytes(I, H, case["quant"]) + _role_bytes(H, I, case["quant"])
    rows = 5 if case["kind"] == "residual" else 2
    b = _active(case["geo"], T, case["zipf"]) * expert + 3 * Is * H * 2 + E * H * 4 + rows * T * H * el
    return {"bytes": b, "flops": 2 * T * (k * 3 * H * I + 3 * H * Is + H * E)}


def tolerance(case):
    if case["kind"] == "requant":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 2e-5}      # 4e-6 measured: float32 activations as bf16 hi / lo pairs
    return {"rel": 1e-2}          # 2e-3 to 3.3e-3 measured: bf16 outputs, bf16 or FP8-plane intermediates


# ------------------------------------------------------------------ the same in 64 bits
def _decode_fp4(codes, scales):
    lut = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=DEV)
    v = torch.stack((lut[(codes & 15).long()], lut[(codes >> 4).long()]), -1).flatten(-2)
    s = torch.exp2(scales.double() - 127.0)
    return (v.unflatten(-1, (-1, 32)) * s[..., None]).flatten(-2)


def _decode_q3(packs, scales, biases):
    p = packs.unflatten(-1, (-1, 3)).int()
    v = p[..., 0] | (p[..., 1] << 8) | (p[..., 2] << 16)
    q = torch.stack([(v >> (3 * i)) & 7 for i in range(8)], -1).flatten(-2).double()
    return (q.unflatten(-1, (-1, 64)) * scales.double()[..., None] + biases.double()[..., None]).flatten(-2)


def _swiglu(x, w1, w3):
    g = torch.clamp(x @ w1.T, max=LIMIT)
    u = torch.clamp(x @ w3.T, -LIMIT, LIMIT)
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    if case["kind"] == "requant":
        w = _decode_fp4(*_requant_inputs(case, seed))
        grp = w.unflatten(-1, (-1, 64))
        lo, hi = grp.amin(-1), grp.amax(-1)
        return w, None, (hi - lo) / 7.0, lo
    c = GEOMETRY[case["geo"]]
    d = _inputs(case, seed)
    x = d["x"].double()
    if case["kind"] == "residual":
        h = (x + d["d"].double()).to(d["x"].dtype)      # the stream and the layer's input have its type
        x = h.double()
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * d["gamma"].double()
        normed = x
        x = x.to(d["x"].dtype).double()
    z = x @ d["gate_w"].double().T
    s = torch.sigmoid(z) if c["score"] == "sigmoid" else torch.sqrt(torch.nn.functional.softplus(z, threshold=50.0))
    idx = torch.topk(s + d["gate_b"].double(), c["k"], dim=1).indices
    w = s.gather(1, idx)
    w = w / (w.sum(1, keepdim=True) + 1e-20) * c["scale"]
    decode = _decode_fp4 if case["quant"] == "fp4" else _decode_q3
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        rows, slot = torch.nonzero(idx == e, as_tuple=True)
        w1, w3, w2 = (decode(*(t[e] for t in d["roles"][r])) for r in ("w1", "w3", "w2"))
        out.index_add_(0, rows, (_swiglu(x[rows], w1, w3) * w[rows, slot, None]) @ w2.T)
    s1, s3, s2 = (t.double() for t in d["shared"])
    out += _swiglu(x, s1, s3) @ s2.T
    return (h, normed, out) if case["kind"] == "residual" else out
