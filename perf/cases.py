"""The work whose speed counts for this framework: the MoE step of the q36
layer (2048 wide, 256 experts of 512, top-8) and the two calls in front of
it, through the package's public entry points.

Four kinds of work:

  moe     one layer forward on router logits that the caller holds
  stack   a decode step of several layers captured in a HIP graph, as a
          serving loop runs it: norm, router and MoE of each layer
  chain   a prefill chunk of one layer: norm + quantise, router, MoE on the
          quantised activations
  router  the router matvec alone;  norm  residual + RMSNorm + quantise alone

and four weight layouts: every matrix MXFP4 ("plain", and "shared" with a
shared expert), the release file's MXFP4 experts with a Q8_0 shared expert
("release"), and its layers whose routed down projection is a k-quant
("kquant": held as int8 with f16 scales whatever the source type, so the
cheapest source, Q8_0, stands for Q5_K and Q6_K).
"""
import functools
import math

import numpy as np
import torch

from q36_amd import moe

D, E, FF, K = 2048, 256, 512, 8
EPS = 1e-6
# E8M0 exponents of the weights: E2M1 codes have a root mean square of 2.8,
# so the weights get about 0.02, as trained ones of this width have
EXP_LO, EXP_HI = -9, -5
MAT = D * FF // 2 + D * FF // 32      # bytes of one MXFP4 matrix
Q8MAT = D * FF + D * FF // 16         # and of one held as int8 + f16


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _moe(name, T, layout, x="f32", out="f32", routing="normal"):
    c = {"kind": "moe", "T": T, "layout": layout, "x": x, "out": out, "routing": routing}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one token of one layer, launched by itself: the smallest call, as a
        # program makes it that does not capture its decode loop
        _moe("decode1", 1, "shared"),
        # one sequence's decode step over 16 layers: what a chat costs per token
        {"name": "decode1_stack", "kind": "stack", "T": 1, "layers": 16, "layout": "shared"},
        # a few sequences decoded together, an odd number of them
        {"name": "decode7_stack", "kind": "stack", "T": 7, "layers": 8, "layout": "shared"},
        # a small batch of decoding sequences in half precision
        _moe("batch24", 24, "plain", x="bf16", out="bf16"),
        # a ragged batch whose tokens favour a few experts
        _moe("ragged61", 61, "shared", out="bf16", routing="zipf"),
        # the same size of batch in the release file's layout
        _moe("release40", 40, "release"),
        # the router of a batch between decode and prefill
        {"name": "router203", "kind": "router", "T": 203, "x": "f32"},
        # a prompt chunk of about a thousand tokens through one layer
        {"name": "chain1000", "kind": "chain", "T": 1000, "layout": "shared"},
        # a full prompt chunk
        _moe("prefill4096", 4096, "plain", out="bf16"),
        # a chunk of 4000 prompt tokens with six decoding sequences, release layout
        _moe("mixed4006_release", 4006, "release", out="bf16"),
        # a ragged chunk in a layer whose down projection is a k-quant
        _moe("kquant1531", 1531, "kquant", x="bf16", out="f32"),
        # the producer of the MoE input for a full chunk
        {"name": "norm4096", "kind": "norm", "T": 4096},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe", "stack", "chain", "router", "norm"])
    if kind == "moe":
        layout = rng.choice(["plain", "shared", "release", "kquant"])
        T = _spread(rng, 1, 2000 if layout == "kquant" else 4000)
        return _moe(None, T, layout, x=rng.choice(["f32", "bf16"]), out=rng.choice(["f32", "bf16"]),
                    routing=rng.choice(["normal", "zipf"]))
    if kind == "stack":
        return {"kind": kind, "T": rng.randint(1, 16), "layers": rng.randint(2, 8),
                "layout": rng.choice(["plain", "shared"])}
    if kind == "chain":
        return {"kind": kind, "T": _spread(rng, 17, 4000), "layout": rng.choice(["plain", "shared"])}
    if kind == "router":
        return {"kind": kind, "T": _spread(rng, 1, 4096), "x": rng.choice(["f32", "bf16"])}
    return {"kind": kind, "T": _spread(rng, 1, 4096)}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


@functools.lru_cache(maxsize=None)
def _zipf_p():
    p = 1.0 / np.arange(1, E + 1) ** 1.1
    return p / p.sum()


def _logits(g, T, routing):
    """N(0, 1), or logits whose top-k are drawn without replacement with
    Zipf(1.1) popularity (log p plus Gumbel noise)."""
    if routing == "normal":
        return _normal(g, T, E)
    p = torch.from_numpy(_zipf_p()).to("cuda", torch.float32)
    order = torch.randperm(E, generator=g, device="cuda")
    u = torch.rand(T, E, generator=g, device="cuda").clamp_(1e-7, 1 - 1e-6)
    return (p.log()[order] - (-u.log()).log()).contiguous()


def _mx_blocks(g, *lead):
    """Random GGUF block_mxfp4 bytes [*lead, 17]."""
    b = torch.randint(0, 256, (*lead, 17), generator=g, device="cuda", dtype=torch.uint8)
    span = EXP_HI - EXP_LO + 1
    b[..., 0] = 127 + EXP_LO + (b[..., 0].to(torch.int32) * span >> 8).to(torch.uint8)
    return b


def _q8_blocks(g, rows, k):
    """Random GGUF Q8_0 blocks [rows, k/32, 34]: f16 scale, 32 int8."""
    b = torch.randint(0, 256, (rows, k // 32, 34), generator=g, device="cuda", dtype=torch.uint8)
    d = torch.rand(rows, k // 32, 1, generator=g, device="cuda") * 4e-4 + 1e-4
    b[..., :2] = d.to(torch.float16).view(torch.uint8)
    return b


def _uploaded(case, seed):
    """GGUF blocks of a release or kquant layer, on the device."""
    g = _gen(seed, 7)
    w = {"gate": _mx_blocks(g, E, FF, D // 32), "up": _mx_blocks(g, E, FF, D // 32)}
    if case["layout"] == "kquant":
        w["down"] = _q8_blocks(g, E * D, FF).view(E, D, -1)
    else:
        w["down"] = _mx_blocks(g, E, D, FF // 32)
    w["sh_gate"], w["sh_up"], w["sh_down"] = (_q8_blocks(g, m, k).view(m, -1) for m, k in ((FF, D), (FF, D), (D, FF)))
    return w


def _weights(case, seed):
    if case["layout"] in ("plain", "shared"):
        w = moe.MoEWeights.alloc(E, D, FF, FF if case["layout"] == "shared" else 0)
        return w.fill_synthetic(int(seed), EXP_LO, EXP_HI)
    b = {k: v.cpu().numpy() for k, v in _uploaded(case, seed).items()}
    return moe.MoEWeights.upload(**b, down_type=moe.GGML_Q8_0 if case["layout"] == "kquant" else moe.GGML_MXFP4,
                                 sh_type=moe.GGML_Q8_0)


def _layer_seed(seed, layer):
    return int(seed) * 64 + layer


def _router_rows(g, rows=E + 1):
    return _normal(g, rows, D) / math.sqrt(D)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    T, kind = case["T"], case["kind"]
    g = _gen(seed, 1)
    if kind == "moe":
        x = _normal(g, T, D)
        s = {"x": x if case["x"] == "f32" else x.to(torch.bfloat16), "logits": _logits(g, T, case["routing"])}
        s["shg"] = _normal(g, T) if case["layout"] != "plain" else None
        return s
    if kind == "router":
        x = _normal(g, T, D)
        return {"x": x if case["x"] == "f32" else x.to(torch.bfloat16), "w": _router_rows(g)}
    if kind == "norm":
        return {"h0": _normal(g, T, D), "a": _normal(g, T, D) * 0.5, "g": 1 + 0.1 * _normal(g, D)}
    n = case["layers"] if kind == "stack" else 1
    rows = E + 1 if case["layout"] == "shared" else E
    return {"layers": [{"h": _normal(g, T, D), "g": 1 + 0.1 * _normal(g, D), "w": _router_rows(g, rows)}
                       for _ in range(n)]}


def _stack_pass(s):
    outs = []
    for p, w in zip(s["layers"], s["weights"]):
        y, _, _ = moe.add_rmsnorm_quant(p["h"], None, p["g"], eps=EPS, want_q=False)
        logits, shg = moe.router_logits(p["w"], y, E)
        outs.append((logits, s["layer"].forward(w, y, logits, shg, out_dtype=torch.float32)))
    return outs


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind, T = case["kind"], case["T"]
    if kind == "moe":
        s["weights"] = _weights(case, seed)
        s["layer"] = moe.MoELayer(T)
    elif kind == "norm":
        s["h"] = torch.empty_like(s["h0"])
    elif kind in ("stack", "chain"):
        s["weights"] = [_weights(case, _layer_seed(seed, i)) for i in range(len(s["layers"]))]
        s["layer"] = moe.MoELayer(T)
    if kind == "stack":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        s["layer"].set_stream(side)
        with torch.cuda.stream(side):
            _stack_pass(s)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            s["outs"] = _stack_pass(s)
        torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "moe":
        return s["layer"].forward(s["weights"], s["x"], s["logits"], s["shg"],
                                  out_dtype=torch.float32 if case["out"] == "f32" else torch.bfloat16)
    if kind == "router":
        return moe.router_logits(s["w"], s["x"], E)
    if kind == "norm":
        # the residual stream as the caller's previous layer leaves it
        s["h"].copy_(s["h0"])
        y, xq, xs = moe.add_rmsnorm_quant(s["h"], s["a"], s["g"], eps=EPS)
        return {"h": s["h"], "y": y, "xq": xq, "xs": xs}
    if kind == "stack":
        s["graph"].replay()
        return s["outs"]
    p = s["layers"][0]
    y, xq, xs = moe.add_rmsnorm_quant(p["h"], None, p["g"], eps=EPS)
    logits, shg = moe.router_logits(p["w"], y, E)
    return {"xq": xq, "xs": xs, "logits": logits,
            "out": s["layer"].forward_q8(s["weights"][0], xq, xs, logits, shg, out_dtype=torch.float32)}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _distinct(T, routing="normal"):
    """Expected number of experts that T tokens hit."""
    if routing == "normal":
        return E * (1 - (1 - K / E) ** T)
    q, left = np.zeros(E), float(K)
    p = _zipf_p()
    q = np.minimum(1.0, p * left)
    for _ in range(20):                       # the popular ones are hit once a token at most
        free = q < 1
        q[free] = np.minimum(1.0, p[free] * (K - (E - free.sum())) / p[free].sum())
    return float((1 - (1 - q) ** T).sum())


def _moe_work(T, layout, x_bytes, out_bytes, routing="normal"):
    down = Q8MAT if layout == "kquant" else MAT
    by = _distinct(T, routing) * (2 * MAT + down) + T * (D * (x_bytes + out_bytes) + E * 4)
    rows = T * K
    if layout != "plain":
        by += 3 * (MAT if layout == "shared" else Q8MAT) + T * 4
        rows += T
    return by, rows * 6 * D * FF


def _router_work(T, x_bytes, rows=E + 1):
    return rows * D * 4 + T * (D * x_bytes + rows * 4), 2 * T * rows * D


def work(case):
    T, kind = case["T"], case["kind"]
    if kind == "moe":
        b, f = _moe_work(T, case["layout"], 4 if case["x"] == "f32" else 2, 4 if case["out"] == "f32" else 2,
                         case["routing"])
    elif kind == "router":
        b, f = _router_work(T, 4 if case["x"] == "f32" else 2)
    elif kind == "norm":
        b, f = T * D * (4 * 4 + 1 + 1 / 32) + D * 4, 6 * T * D
    else:
        rows = E + 1 if case["layout"] == "shared" else E
        n = case["layers"] if kind == "stack" else 1
        # h and the norm's weight in, the router's rows, the experts, logits
        # and the layer's sum out; a chain also gives the quantised input
        mb, mf = _moe_work(T, case["layout"], 0, 4)
        b = n * (T * D * 4 + D * 4 + rows * D * 4 + T * rows * 4 + mb + (T * D * 33 / 32 if kind == "chain" else 0))
        f = n * (6 * T * D + 2 * T * rows * D + mf)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # four times what the results are off 64 bits: fp32 sums 3e-7 (router),
    # bf16 outputs 1.9e-3, and up to 8e-4 in f32 outputs (h codes on rounding
    # midpoints and the 16-bit staging of the weighted rows)
    kind = case["kind"]
    if kind == "router":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "norm":
        # codes flip where the norm's last bit decides a tie
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}
    if kind == "moe" and case["out"] == "bf16":
        return {"rel": 8e-3, "max": 5e-2}
    return {"rel": 3.5e-3, "max": 5e-2, "differ": 1e-4}


# --------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# --------------------------------------------------------------------------
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _mix64(z):
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _signed(0x94D049BB133111EB)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _synthetic(seed, salt, M, k):
    """The matrix [M, k] that fill_synthetic writes as its salt-th: bytes from
    a counter hash, in the documented device layout (tiles of 16 rows x 128)."""
    nib, n = M * k // 2, M * k // 2 + M * k // 32
    i = torch.arange(0, n, 16, device="cuda", dtype=torch.int64)
    a = _mix64(_signed(int(seed) * 0x100000001B3 + salt) ^ (i * _signed(0x9E3779B97F4A7C15)))
    b = _mix64(a ^ _signed(0x632BE59BD9B4E019))
    raw = torch.stack([a, b], 1).view(-1).view(torch.uint8)
    codes = raw[:nib].view(M // 16, k // 128, 4, 16, 16)            # row tile, K tile, K block, row, byte
    lut = torch.tensor(_E2M1, device="cuda", dtype=torch.float64)
    val = torch.stack([lut[(codes & 15).long()], lut[(codes >> 4).long()]], -1)
    val = val.view(M // 16, k // 128, 4, 16, 32).permute(0, 3, 1, 2, 4)
    exp = EXP_LO + (raw[nib:].to(torch.int64) * (EXP_HI - EXP_LO + 1) >> 8)
    exp = exp.view(M // 16, 4, 16, k // 128).permute(0, 2, 3, 1).unsqueeze(-1)
    return (val * torch.exp2(exp.double())).reshape(M, k)


def _dec_mx(b, M, k):
    b = b.view(M, k // 32, 17)
    lut = torch.tensor(_E2M1, device="cuda", dtype=torch.float64)
    v = torch.cat([lut[(b[..., 1:] & 15).long()], lut[(b[..., 1:] >> 4).long()]], -1)
    return (v * torch.exp2(b[..., :1].double() - 127)).view(M, k)


def _dec_q8(b, M, k):
    b = b.view(M, k // 32, 34)
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (b[..., 2:].contiguous().view(torch.int8).double() * d).view(M, k)


def _e4m3_pow2(v):
    """Per-32 e4m3 values with power-of-two scales: (codes, E8M0 bytes, values in 64 bits)."""
    f = v.float().view(*v.shape[:-1], -1, 32)
    amax = f.abs().amax(-1, keepdim=True)
    m, e = torch.frexp(amax / 448)
    e2 = torch.where(amax > 0, (e - (m == 0.5).int()).clamp(-127, 127), torch.full_like(e, -127))
    q = (f.double() * torch.exp2(-e2.double())).float().to(torch.float8_e4m3fn)
    return q.view(torch.uint8).view(v.shape), (e2 + 127).to(torch.uint8).squeeze(-1), \
        (q.double() * torch.exp2(e2.double())).view(v.shape)


def _int8_32(v):
    """Per-32 int8 codes times their fp32 scale, in 64 bits."""
    f = v.float().view(*v.shape[:-1], -1, 32)
    amax = f.abs().amax(-1, keepdim=True)
    inv = torch.where(amax > 0, 127 / amax, torch.zeros_like(amax))
    return ((f * inv).round().clamp(-127, 127).double() * (amax / 127).double()).view(v.shape)


def _exact_moe(layout, mats, x, logits, shg):
    """mats(which, expert) gives a matrix in 64 bits; expert E is the shared one."""
    T = x.shape[0]
    # the larger logit first, the lower index among equals
    idx = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :K]
    top = logits.gather(1, idx).double()
    wt = torch.softmax(top, 1)
    xq = _e4m3_pow2(x.float())[2]
    out = torch.zeros(T, D, dtype=torch.float64, device="cuda")

    def expert(e, xin, q8_down):
        gate, up = xin @ mats("gate", e).T, xin @ mats("up", e).T
        h = gate * torch.sigmoid(gate) * up
        return (_int8_32(h) if q8_down else _e4m3_pow2(h)[2]) @ mats("down", e).T

    for e in torch.unique(idx).tolist():
        t, s = (idx == e).nonzero(as_tuple=True)
        out[t] += wt[t, s, None] * expert(e, xq[t], layout == "kquant")
    if shg is not None:
        q8 = layout in ("release", "kquant")
        out += torch.sigmoid(shg.double())[:, None] * expert(E, _int8_32(x.float()) if q8 else xq, q8)
    return out


def _mats(case, seed):
    if case["layout"] in ("plain", "shared"):
        def get(which, e):
            k = ("gate", "up", "down").index(which)
            salt = 1 + 3 * E + k if e == E else 1 + k * E + e
            return _synthetic(seed, salt, *((D, FF) if which == "down" else (FF, D)))
        return get
    w = _uploaded(case, seed)

    def get(which, e):
        M, k = (D, FF) if which == "down" else (FF, D)
        if e == E:
            return _dec_q8(w["sh_" + which], M, k)
        return (_dec_q8 if which == "down" and case["layout"] == "kquant" else _dec_mx)(w[which][e], M, k)
    return get


def _exact_router(w, x):
    """fp32 operands up to 16 tokens, fp16 ones above."""
    if x.shape[0] > 16:
        w, x = w.to(torch.float16), x.float().to(torch.float16)
    r = x.double() @ w.double().T
    return r[:, :E], r[:, E] if w.shape[0] > E else None


def _exact_norm(h, g):
    h = h.double()
    return h * torch.rsqrt(h.square().mean(1, keepdim=True) + EPS) * g.double()


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "moe":
        return _exact_moe(case["layout"], _mats(case, seed), s["x"], s["logits"], s["shg"])
    if kind == "router":
        return _exact_router(s["w"], s["x"])
    if kind == "norm":
        h = s["h0"] + s["a"]
        y = _exact_norm(h, s["g"])
        xq, xs, _ = _e4m3_pow2(y)
        return {"h": h.double(), "y": y, "xq": xq, "xs": xs}
    outs = []
    for i, p in enumerate(s["layers"]):
        y = _exact_norm(p["h"], p["g"])
        logits, shg = _exact_router(p["w"], y.float())
        out = _exact_moe(case["layout"], _mats(case, _layer_seed(seed, i)), y, logits, shg)
        outs.append((logits, out))
    if kind == "stack":
        return outs
    xq, xs, _ = _e4m3_pow2(y)
    return {"xq": xq, "xs": xs, "logits": outs[0][0], "out": outs[0][1]}
