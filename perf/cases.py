"""What this library is timed on: the projections of a transformer as a serving program calls them.

A case is one pass: the activations are quantized (or normalised / gated and quantized) and projected through
`knivesysl_xe_amd.ops`, or a weight is repacked as a model is loaded. Decode passes walk several layers with weights of
their own, so that the weights come from memory as they do in a model, not from the last-level cache; where `graph` is
set the pass is the replay of a HIP graph, as a serving loop launches its decode step, else the calls are made one by
one.

Fields of a projection case: `rows` output rows of each weight that shares the activation, `K` its columns, `T` tokens,
`seg` the lengths of packed prompts ("" = one), and `mode`:
  token   int4 codes, FP16 scale per `group` (64 / 128), one activation scale per token
  block   int4 codes with zero points, `group` 32 / 64, one activation scale per (token, K32 block)
  k16     the same with group 16 (GEMV only)
  w8      int8 codes, FP16 scale per K32, activation scales per K32 block
  w4a4    int4 codes with zero points, group 64, s4 activations per (token, K64)
"""
import math

import torch

from knivesysl_xe_amd import ops
from knivesysl_xe_amd._lib import SCALE_FP16, SCALE_FP16_ZP4

HIDDEN, INTER, VOCAB = 5120, 17408, 248320
EPS = 1e-6


def _proj(mode, rows, K, T, group, call="gemm", x="f32", out="f32", residual=False, seg="", layers=1, copies=1,
          graph=False):
    return {"kind": "proj", "mode": mode, "rows": rows, "K": K, "T": T, "group": group, "call": call, "x": x,
            "out": out, "residual": residual, "seg": seg, "layers": layers, "copies": copies, "graph": graph}


def _mlp(T, mode, hidden=HIDDEN, inter=INTER, layers=1, graph=False):
    return {"kind": "mlp", "mode": mode, "hidden": hidden, "inter": inter, "T": T, "layers": layers, "graph": graph}


def _repack(M, K, tier):
    return {"kind": "repack", "M": M, "K": K, "tier": tier}


def listed():
    c = [
        # the smallest call: one token through one square projection, called from Python
        dict(_proj("token", "4096", 4096, 1, 128, "gemv", x="bf16", copies=24), name="gemv_small"),
        # single-stream decode: the MLP blocks of two layers, norm to residual
        dict(_mlp(1, "block", layers=2, graph=True), name="mlp_decode"),
        # a speculative wave or a batch of eight: gate and up of four layers
        dict(_proj("token", "17408,17408", HIDDEN, 8, 128, x="bf16", out="bf16", layers=4, graph=True),
             name="gate_up_wave8"),
        # a batch of 27 sequences: gate and up of two layers
        dict(_proj("block", "17408,17408", HIDDEN, 27, 32, layers=2), name="gate_up_batch27"),
        # a prompt of 49 tokens: down projection and residual of two layers
        dict(_proj("token", "5120", INTER, 49, 64, x="bf16", residual=True, layers=2), name="down_prompt49"),
        # one prefill chunk of 512 tokens through an MLP block
        dict(_mlp(512, "block"), name="mlp_prefill512"),
        # six prompts packed into one prefill, gate and up
        dict(_proj("token", "17408,17408", HIDDEN, 3965, 128, x="bf16", out="bf16", seg="17,64,300,512,1024,2048"),
             name="gate_up_packed"),
        # short prompts of unequal length packed into one prefill, attention output
        dict(_proj("block", "5120", HIDDEN, 512, 32, residual=True, seg="17,64,300,41,90"), name="out_packed_short"),
        # the W4A4 prefill of a chunk: down projection and residual
        dict(_proj("w4a4", "5120", INTER, 512, 64, residual=True), name="down_w4a4"),
        # the head over a wave of eight
        dict(_proj("w8", "%d" % VOCAB, HIDDEN, 8, 32), name="head_wave8"),
        # decode with the finest weight groups: down projection and residual of three layers
        dict(_proj("k16", "5120", INTER, 1, 16, "gemv", residual=True, layers=3, graph=True), name="down_k16"),
        # model load: one weight from its stored form
        _repack(INTER, HIDDEN, "w4k32"),
    ]
    c[-1]["name"] = "load_repack"
    return c


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    return max(m, _log(rng, lo, hi) // m * m)


def draw(rng):
    """Another case: the kind first, then its sizes over their whole range, most of them odd."""
    kind = rng.choice(["decode", "decode", "batch", "batch", "prefill", "prefill", "packed", "w4a4", "w8", "k16", "mlp",
                       "repack"])
    K = _mult(rng, 1024, INTER, 128)
    N = _mult(rng, 512, INTER, 16)
    tok = rng.random() < 0.5
    mode, group = ("token", rng.choice([64, 128])) if tok else ("block", rng.choice([32, 64]))
    x, out = rng.choice(["f32", "bf16"]), rng.choice(["f32", "bf16"])
    two = rng.random() < 0.4
    rows = "%d,%d" % (N, _mult(rng, 256, INTER, 16)) if two else str(N)
    residual = not two and rng.random() < 0.5
    if kind == "decode":
        if rng.random() < 0.5:
            call, T = ("fanout" if two else "gemv"), rng.choice([1, 1, 1, 2, 3, 4])
        else:
            call, T = "gemm", rng.randint(1, 16)
        return _proj(mode, rows, K, T, group, call, x, out, residual and call != "fanout", layers=_layers(rows, K, 0.5),
                     graph=rng.random() < 0.7)
    if kind == "batch":
        return _proj(mode, rows, K, rng.randint(17, 64), group, "gemm", x, out, residual, layers=_layers(rows, K, 0.5))
    if kind == "prefill":
        return _proj(mode, rows, K, _tokens(rng, 65, 4096, rows, K), group, "gemm", x, out, residual)
    if kind == "packed":
        lens = [_log(rng, 8, 600) for _ in range(rng.randint(2, 7))]
        return _proj(mode, rows, K, sum(lens), group, "gemm", x, out, residual, ",".join(map(str, lens)))
    if kind == "w4a4":
        return _proj("w4a4", str(N), K, _tokens(rng, 8, 2048, str(N), K), 64, "gemm", x, out, residual)
    if kind == "w8":
        if rng.random() < 0.5:
            rows = str(_mult(rng, 32000, VOCAB, 16))
            return _proj("w8", rows, _mult(rng, 1024, HIDDEN, 128), rng.randint(1, 16), 32, "gemm", x, out)
        return _proj("w8", str(N), K, _tokens(rng, 17, 1024, str(N), K), 32, "gemm", x, out, residual)
    if kind == "k16":
        return _proj("k16", str(N), K, _log(rng, 1, 16), 16, "gemv", x, out, residual, layers=_layers(str(N), K, 0.6),
                     graph=rng.random() < 0.7)
    if kind == "mlp":
        T = rng.choice([1, rng.randint(2, 16), rng.randint(17, 64), _log(rng, 65, 1024)])
        return _mlp(T, mode, _mult(rng, 1024, HIDDEN, 128), _mult(rng, 2048, INTER, 128),
                    layers=2 if T <= 64 else 1, graph=T <= 16)
    return _repack(N, K, rng.choice(["w4k32", "w4k64", "w4k16", "w8"]))


def _layers(rows, K, per_value):
    """Layers of a decode pass: about 200 MB of weights, at most 8 layers."""
    return max(1, min(8, int(200e6 / (sum(map(int, rows.split(","))) * K * per_value))))


def _tokens(rng, lo, hi, rows, K):
    """Tokens over [lo, hi], no more work than the largest listed case's half."""
    T = _log(rng, lo, hi)
    most = 0.35e12 / (sum(map(int, rows.split(","))) * K)
    return max(lo, min(T, int(most)))


# ---- inputs: from the seed alone, in a fixed order ---------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _natural_weight(g, M, K, mode, group):
    """Codes [M][K] int8 and scale bits [M][K/group] int16; zero points ride in the low nibble of a scale."""
    lo, hi = (-127, 128) if mode == "w8" else (-8, 8)
    codes = torch.randint(lo, hi, (M, K), generator=g, device="cuda", dtype=torch.int8)
    size = 0.0004 if mode == "w8" else 0.004
    s = (size * (0.5 + torch.rand(M, K // group, generator=g, device="cuda"))).to(torch.float16).view(torch.int16)
    if mode in ("block", "k16", "w4a4"):
        zp = torch.randint(0, 16, (M, K // group), generator=g, device="cuda", dtype=torch.int16)
        s = (s & -16) | zp
    return codes, s


def _x(g, T, K, dtype):
    """Activations: normal, with a few channels ten times larger, as hidden states have them."""
    x = torch.randn(T, K, generator=g, device="cuda")
    big = torch.randint(0, K, (K // 256,), generator=g, device="cuda")
    x[:, big] *= 10.0
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _proj_natural(case, seed, layer):
    g = _gen(seed * 1009 + layer)
    K, T = case["K"], case["T"]
    x = _x(g, T, K, case["x"])
    Ms = [int(r) for r in case["rows"].split(",")]
    res = torch.randn(T, Ms[0], generator=g, device="cuda") if case["residual"] else None
    ws = (_natural_weight(g, M, K, case["mode"], case["group"]) for M in Ms)
    return x, res, ws


def _mlp_groups(mode):
    return (32, 64) if mode == "block" else (128, 64)


def _mlp_natural(case, seed, layer):
    g = _gen(seed * 1009 + layer)
    H, I = case["hidden"], case["inter"]
    x = _x(g, case["T"], H, "f32")
    norm = (0.05 * torch.randn(H, generator=g, device="cuda")).to(torch.bfloat16)
    g1, g2 = _mlp_groups(case["mode"])
    ws = (_natural_weight(g, M, K, case["mode"], gr) for M, K, gr in ((I, H, g1), (I, H, g1), (H, I, g2)))
    return x, norm, ws


def _pack(codes, scales, mode, group):
    if mode == "w8":
        return ops.W4Weight.from_codes_s8(codes, scales)
    return ops.W4Weight.from_codes(codes, scales, group, SCALE_FP16 if mode == "token" else SCALE_FP16_ZP4)


def _clone(w):
    return ops.W4Weight(w.M, w.K, w.group, w.scale_enc, w.codes.clone(), w.scales.clone())


# ---- one layer ---------------------------------------------------------------------------------------------------

def _dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _offsets(seg):
    if not seg:
        return None
    off = [0]
    for n in seg.split(","):
        off.append(off[-1] + int(n))
    return off


def _run_proj(case, lay):
    ws, x, res, act = lay["ws"][lay["turn"] % len(lay["ws"])], lay["x"], lay["res"], lay["act"]
    lay["turn"] += 1
    dt = _dtype(case["out"])
    if case["mode"] == "w4a4":
        return [ops.gemm_w4a4(ws[0], ops.quantize_act_s4(x, out=act), dt, residual=res)]
    a = ops.quantize_act(x, 0 if case["mode"] == "token" else 32, out=act)
    if case["call"] == "gemv":
        return [ops.gemv(ws[0], a, dt, residual=res)]
    if case["call"] == "fanout":
        return ops.gemv_fanout(ws, a, dt)
    off = _offsets(case["seg"])
    if len(ws) == 1:
        return [ops.gemm(ws[0], a, dt, residual=res, offsets=off)]
    return ops.gemm_fanout(ws, a, dt, offsets=off)


def _run_small(lay):
    ops.quantize_act(lay["x"], 0, out=lay["act"])
    lay["turn"] += 1
    return [lay["calls"][lay["turn"] % len(lay["calls"])]()]


def _run_mlp(case, lay):
    (gate, up, down), x = lay["ws"], lay["x"]
    block = 32 if case["mode"] == "block" else 0
    _, a = ops.rmsnorm_quant(x, lay["norm"], EPS, block, keep_normed=False)
    if case["T"] == 1:
        yg, yu = ops.gemv_fanout([gate, up], a)
        _, h = ops.silu_mul_quant(yg, yu, block, keep_hidden=False)
        return [ops.gemv(down, h, residual=x)]
    yg, yu = ops.gemm_fanout([gate, up], a)
    _, h = ops.silu_mul_quant(yg, yu, block, keep_hidden=False)
    return [ops.gemm(down, h, residual=x)]


def _layer(case, seed, i):
    if case["kind"] == "mlp":
        x, norm, ws = _mlp_natural(case, seed, i)
        g1, g2 = _mlp_groups(case["mode"])
        return {"x": x, "norm": norm, "ws": [_pack(c, s, case["mode"], gr) for (c, s), gr in zip(ws, (g1, g1, g2))]}
    x, res, nat = _proj_natural(case, seed, i)
    ws = [_pack(c, s, case["mode"], case["group"]) for c, s in nat]
    T, K = case["T"], case["K"]
    act = (ops.QuantActS4.empty(T, K) if case["mode"] == "w4a4"
           else ops.QuantAct.empty(T, K, 0 if case["mode"] == "token" else 32))
    # `copies`: the same weight at other addresses, in turn, as the other layers of a model would come
    sets = [ws] + [[_clone(w) for w in ws] for _ in range(case["copies"] - 1)]
    lay = {"x": x, "res": res, "ws": sets, "act": act, "turn": 0}
    if case["copies"] > 1:   # a serving loop keeps its checked calls
        lay["calls"] = [ops.PreparedGemv(w[0], act, _dtype(case["out"]), residual=res) for w in sets]
    return lay


def prepare(case, seed):
    if case["kind"] == "repack":
        payload, bs = _stored(case, seed)
        return {"case": case, "payload": payload, "bs": bs, "graph": None}
    st = {"case": case, "layers": [_layer(case, seed, i) for i in range(case["layers"])], "graph": None}
    if case["graph"]:
        _pass(st)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            st["out"] = _pass(st)
        st["graph"] = g
    return st


def _pass(st):
    case = st["case"]
    if case["kind"] == "mlp":
        return [_run_mlp(case, lay) for lay in st["layers"]]
    if case["copies"] > 1:
        return [_run_small(lay) for lay in st["layers"]]
    return [_run_proj(case, lay) for lay in st["layers"]]


def run(st):
    case = st["case"]
    if case["kind"] == "repack":
        M, K, tier = case["M"], case["K"], case["tier"]
        if tier == "w8":
            w = ops.W4Weight.repack_e2m3_s8(st["payload"], st["bs"], K // 128, M, K)
        else:
            w = ops.W4Weight.repack_e2m3(st["payload"], st["bs"], K // 128, M, K,
                                         {"w4k32": 0, "w4k16": 1, "w4k64": 2}[tier])
        return [w.codes, w.scales]
    if st["graph"] is not None:
        st["graph"].replay()
        return st["out"]
    return _pass(st)


def _stored(case, seed):
    """E2M3 payload of roughly normal values (96-bit little-endian streams of 16 six-bit codes) and block scales."""
    g = _gen(seed)
    M, K = case["M"], case["K"]
    v = 2.0 * torch.randn(M * K // 4, 4, generator=g, device="cuda")
    a = v.abs().clamp(max=7.5)
    e = torch.floor(torch.log2(a.clamp(min=1.0))).clamp(0, 2)
    mag = torch.where(a < 1.0, torch.round(a * 8), (e + 1) * 8 + torch.round((a / torch.exp2(e) - 1) * 8))
    c = mag.clamp(0, 31).to(torch.int32) | torch.where(v < 0, 32, 0).to(torch.int32)
    word = c[:, 0] | (c[:, 1] << 6) | (c[:, 2] << 12) | (c[:, 3] << 18)
    payload = torch.stack([word & 255, (word >> 8) & 255, (word >> 16) & 255], 1).to(torch.uint8).reshape(-1)
    bs = 0.002 + 0.004 * torch.rand((M + 127) // 128, K // 128, generator=g, device="cuda")
    return payload.contiguous(), bs.contiguous()


# ---- work, tolerance, exact results ------------------------------------------------------------------------------

def _weight_bytes(M, K, mode, group):
    return M * K * (1.0 if mode == "w8" else 0.5) + 2.0 * M * K / group


def work(case):
    if case["kind"] == "repack":
        M, K, tier = case["M"], case["K"], case["tier"]
        group = {"w4k32": 32, "w4k16": 16, "w4k64": 64, "w8": 32}[tier]
        out = _weight_bytes(M, K, "w8" if tier == "w8" else "block", group)
        return {"bytes": M * K * 0.75 + 4.0 * M * K / 16384 + out, "flops": 0}
    T, L = case["T"], case["layers"]
    if case["kind"] == "mlp":
        H, I = case["hidden"], case["inter"]
        g1, g2 = _mlp_groups(case["mode"])
        b = 2 * _weight_bytes(I, H, case["mode"], g1) + _weight_bytes(H, I, case["mode"], g2)
        return {"bytes": L * (b + 4.0 * T * H * 2 + 2 * H), "flops": L * 6.0 * T * H * I}
    K, Ms = case["K"], [int(r) for r in case["rows"].split(",")]
    b = sum(_weight_bytes(M, K, case["mode"], case["group"]) for M in Ms)
    b += T * K * (2 if case["x"] == "bf16" else 4) + T * sum(Ms) * (2 if case["out"] == "bf16" else 4)
    b += T * Ms[0] * 4 if case["residual"] else 0
    return {"bytes": L * float(b), "flops": L * 2.0 * T * sum(Ms) * K}


def tolerance(case):
    if case["kind"] == "repack":
        return "exact"
    if case["kind"] == "mlp":
        # the gated activations are quantized again: a value that rounds another way there moves its
        # token's outputs by a part of one code
        return {"rel": 1e-3, "max": 5e-2}
    if case["out"] == "bf16":
        return {"rel": 4e-3, "max": 2e-2}
    # 32-bit sums of at most K/16 terms
    return {"rel": 1e-5, "max": 1e-3}


def _exact_weight(codes, scales, mode, group, lo, hi):
    """Rows [lo, hi) in 64 bits."""
    bits = scales[lo:hi]
    z = 0.0
    if mode in ("block", "k16", "w4a4"):
        n = (bits & 15).to(torch.float64)
        z = torch.where(n >= 8, n - 16, n).repeat_interleave(group, 1)
        bits = bits & -16
    s = bits.contiguous().view(torch.float16).to(torch.float64).repeat_interleave(group, 1)
    return (codes[lo:hi].to(torch.float64) - z) * s


def _exact_act(x, block, top):
    """Codes times scales: per row (block 0) or per block of a row. The format defines scales and codes by FP32
    divisions (absmax / top, value / scale), so they are taken so; the rest is in 64 bits."""
    v = x.to(torch.float32)
    T, K = v.shape
    v = v.view(T, -1, block or K)
    m = v.abs().amax(2, keepdim=True)
    s = m / torch.full_like(m, top)    # (a division by a plain number is a product with its inverse)
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (torch.clamp(torch.round(v / s), -top, top).to(torch.float64) * s.to(torch.float64)).view(T, K)


def _exact_project(a, codes, scales, mode, group):
    M, K = codes.shape
    step = max(16, (1 << 27) // K)
    return torch.cat([a @ _exact_weight(codes, scales, mode, group, lo, min(M, lo + step)).t()
                      for lo in range(0, M, step)], 1)


def exact(case, seed):
    if case["kind"] == "repack":
        return None
    out = []
    for i in range(case["layers"]):
        mode = case["mode"]
        block = {"token": 0, "w4a4": 64}.get(mode, 32)
        if case["kind"] == "mlp":
            x, norm, ws = _mlp_natural(case, seed, i)
            g1, g2 = _mlp_groups(mode)
            v = x.to(torch.float64)
            n = v * torch.rsqrt((v * v).mean(1, keepdim=True) + EPS) * (1.0 + norm.to(torch.float64))
            a = _exact_act(n, block, 127.0)
            gate = _exact_project(a, *next(ws), mode, g1)
            up = _exact_project(a, *next(ws), mode, g1)
            h = _exact_act(gate / (1.0 + torch.exp(-gate)) * up, block, 127.0)
            out.append([_exact_project(h, *next(ws), mode, g2) + v])
            continue
        x, res, ws = _proj_natural(case, seed, i)
        a = _exact_act(x, block, 7.0 if mode == "w4a4" else 127.0)
        ys = [_exact_project(a, c, s, mode, case["group"]) for c, s in ws]
        if res is not None:
            ys[0] = ys[0] + res.to(torch.float64)
        out.append(ys)
    return out
