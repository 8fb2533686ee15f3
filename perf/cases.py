"""The framework's measured work: what a program that serves, loads or quantizes
a Qwen3-shaped model has it do, through the public entry points of
gophonic_amd.gphq.

One case is a dict of plain values; `kind` names the path:

  gemv        one token's projection (the single-vector GEMV)
  gemv_batch  a stream of independent projections in one launch
  gemv_vec    one projection for several decode lanes (multi-vector GEMV)
  i8          per-row int8 activations times int8 weights, exact int32
  mm          batched projection on FP16 tiles (Q8, Q8B, Q8B_F32, Q4, GPTQ int4)
  block32     block-32 int8 activations times block-32 int8 weights
  decode      whole decode steps over a K/V cache: hidden states and logits
  prefill     a whole batched pass over a prompt: hidden state and K/V rows
  project     one layer's projection of a batched pass
  gptq        the GPTQ producer's H = X^T X and its inverse factor

Weights are Gaussian codes with scales that keep every product's output near
unit size, activations are Gaussian with a few large channels.
"""
import numpy as np
import torch

from gophonic_amd import gphq

FMT = dict(q8=gphq.FMT_Q8, q8b=gphq.FMT_Q8B, q8b_f32=gphq.FMT_Q8B_F32, q4=gphq.FMT_Q4, gptq4=gphq.FMT_GPTQ4_G128)

# Qwen3 widths (Qwen3-0.6B, the Qwen3-ASR-1.7B decoder, Qwen3-8B); 128-wide heads, 8 KV heads.
GEOM = {
    "0.6b": dict(hidden=1024, heads=16, inter=3072),
    "1.7b": dict(hidden=2048, heads=16, inter=6144),
    "8b": dict(hidden=4096, heads=32, inter=12288),
}
HD, KV_HEADS, VOCAB, MAX_POS, EPS, THETA = 128, 8, 151936, 40960, 1e-6, 1e6
KVD = KV_HEADS * HD
PROMPT_VOCAB = 16384  # a batched pass reads embedding rows, not the head: a shorter table for it


def listed():
    return [
        # The smallest call: one token through one Qwen3-8B o_proj, in the decode format.
        dict(name="gemv_o_proj", kind="gemv", fmt="q8b", k=4096, n=4096),
        # The headline stream: 32 projections with fp32 block scales in one launch.
        dict(name="gemv_stream32", kind="gemv_batch", fmt="q8b_f32", count=32, k=4096, n=4096),
        # Eight decode lanes sharing one 4-bit gate/up projection.
        dict(name="lanes8_q4_gate_up", kind="gemv_vec", fmt="q4", lanes=8, k=4096, n=24576),
        # The int8 GEMM on 512 activation rows, quantizer included.
        dict(name="i8_rows512", kind="i8", m=512, k=4096, n=12288),
        # A 77-token prompt through one Qwen3-8B QKV projection.
        dict(name="mm_q8b_rows77", kind="mm", fmt="q8b", m=77, k=4096, n=6144),
        # GPTQ int4 (group 128, zero points) at 256 rows.
        dict(name="mm_gptq4_rows256", kind="mm", fmt="gptq4", m=256, k=4096, n=12288),
        # The block-scaled int8 product at 128 rows, quantizer included.
        dict(name="block32_rows128", kind="block32", m=128, k=4096, n=12288),
        # One decode step of a whole Qwen3-0.6B at a 1024-token context: latency.
        dict(name="decode_06b_lane1", kind="decode", geom="0.6b", layers=28, fmt="q8b", lanes=1, ctx=1024),
        # A step of 16 lanes at a 4096-token context, two of Qwen3-8B's layers and its head.
        dict(name="decode_8b_lanes16", kind="decode", geom="8b", layers=2, fmt="q8b", lanes=16, ctx=4096),
        # A 4096-token prompt through two of Qwen3-8B's layers (FP16 tiles).
        dict(name="prefill_8b_4096", kind="prefill", geom="8b", layers=2, fmt="q8b", route="fp16", keep=0, tokens=4096),
        # One gate/up projection of a 4096-row pass on the int8 route.
        dict(name="project_i8_gate_up", kind="project", geom="8b", fmt="q8", route="int8", proj=2, rows=4096),
        # The GPTQ factor of one Qwen3-8B projection input over a full calibration set.
        dict(name="gptq_factor_4096", kind="gptq", k=4096, rows=4096),
    ]


def draw(rng):
    def log(lo, hi, step=1):
        return max(1, round(lo * (hi / lo) ** rng.random() / step)) * step

    kind = rng.choice(["gemv", "gemv_batch", "gemv_vec", "i8", "mm", "block32", "decode", "prefill", "project", "gptq"])
    if kind == "gemv":
        return dict(kind=kind, fmt=rng.choice(["q8", "q8b", "q8b_f32", "q4"]), k=log(1024, 12288, 32), n=log(512, 25000))
    if kind == "gemv_batch":
        return dict(kind=kind, fmt=rng.choice(["q8", "q8b", "q8b_f32", "q4"]), count=rng.randint(2, 32),
                    k=log(512, 4096, 32), n=log(512, 4096))
    if kind == "gemv_vec":
        return dict(kind=kind, fmt=rng.choice(["q8", "q8b", "q8b_f32", "q4"]), lanes=rng.randint(2, 32),
                    k=log(512, 12288, 32), n=log(512, 25000))
    if kind == "i8":
        return dict(kind=kind, m=log(1, 1024), k=log(512, 8192), n=log(512, 12288))
    if kind == "mm":
        return dict(kind=kind, fmt=rng.choice(["q8", "q8b", "q8b_f32", "q4", "gptq4"]), m=log(1, 1024),
                    k=log(512, 12288, 128), n=log(512, 12288))
    if kind == "block32":
        return dict(kind=kind, m=log(1, 512), k=log(512, 8192, 32), n=log(512, 12288))
    geom = rng.choice(["0.6b", "1.7b", "8b"])
    fmt = rng.choice(["q8", "q8b", "q4"])
    if kind == "decode":
        return dict(kind=kind, geom=geom, layers=rng.randint(1, 3), fmt=fmt, lanes=log(1, 16), ctx=log(16, 4096))
    route = "int8" if fmt == "q8" and rng.random() < 0.7 else "fp16"
    if kind == "prefill":
        tokens = log(8, 3000)
        return dict(kind=kind, geom=geom, layers=rng.randint(1, 2), fmt=fmt, route=route,
                    keep=0 if rng.random() < 0.6 else log(8, 1000), tokens=tokens)
    if kind == "project":
        return dict(kind=kind, geom=geom, fmt=fmt, route=route, proj=rng.randint(0, 3), rows=log(2, 4096))
    return dict(kind=kind, k=log(256, 4096, 64), rows=log(256, 4096))


# ---- inputs -------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * seed + 17)


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _acts(g, rows, k):
    """Activations: N(0,1), one channel in 256 eight times as large."""
    x = _randn(g, rows, k)
    x[:, 5::256] *= 8
    return x


def _matrix(g, fmt, n, k, pad=0):
    """(codes, scales, zeros) of an n x k weight matrix with unit-size outputs; `pad` zero rows below."""
    if fmt in ("q4", "gptq4"):
        nib = (_randn(g, n, k) * 2.7 + 8).round_().clamp_(0, 15).to(torch.uint8)
        group = 32 if fmt == "q4" else 128
        s = ((0.6 + 0.8 * torch.rand((n, k // group), device="cuda", generator=g)) / (2.7 * k ** 0.5)).half()
        if fmt == "q4":
            b = nib.view(n, k // 32, 2, 16)
            return (b[:, :, 0] | (b[:, :, 1] << 4)).view(n, k // 2).contiguous(), s, None
        b = nib.view(n, k // 2, 2)
        codes = (b[:, :, 0] | (b[:, :, 1] << 4)).contiguous().view(torch.int32)
        return codes, s, torch.randint(6, 11, (n, k // group), dtype=torch.uint8, device="cuda", generator=g)
    codes = torch.zeros((n + pad, k), dtype=torch.int8, device="cuda")
    for r in range(0, n, 16384):
        e = min(n, r + 16384)
        codes[r:e] = (_randn(g, e - r, k) * 40).round_().clamp_(-127, 127).to(torch.int8)
    per = 1 if fmt == "q8" else k // 32
    s = (0.6 + 0.8 * torch.rand((n, per), device="cuda", generator=g)) / (40 * k ** 0.5)
    s = torch.cat([s, torch.zeros((pad, per), device="cuda")]) if pad else s
    return codes, s.half() if fmt == "q8b" else s, None


def _norm_weight(g, n):
    return 1 + 0.05 * _randn(g, n)


def _layers(g, c, layers):
    """Per layer {qkv, o, gu, down: matrix, q_norm, k_norm}, gate and up rows interleaved."""
    G = GEOM[c["geom"]]
    H, I, qd = G["hidden"], G["inter"], G["heads"] * HD
    shapes = dict(qkv=(qd + 2 * KVD, H), o=(H, qd), gu=(2 * I, H), down=(H, I))
    out = []
    for _ in range(layers):
        L = {name: _matrix(g, c["fmt"], n, k) for name, (n, k) in shapes.items()}
        L["q_norm"], L["k_norm"] = _norm_weight(g, HD), _norm_weight(g, HD)
        out.append(L)
    return out


def _model(g, c, layers, vocab):
    """The raw model: layers, BF16 embedding table, final norm, Q8B head (rows padded to 16)."""
    H = GEOM[c["geom"]]["hidden"]
    embed = torch.cat([_randn(g, min(16384, vocab - r), H).bfloat16() for r in range(0, vocab, 16384)])
    head_vocab = vocab if c["kind"] == "decode" else 256
    return dict(layers=_layers(g, c, layers), embed=embed, final_norm=_norm_weight(g, H), head_vocab=head_vocab,
                head=_matrix(g, "q8b", head_vocab, H, pad=-head_vocab % 16))


def _bind(c, model, vocab):
    """The loaded model: layer buffers, embedding table and head laid out once, as a loader leaves them."""
    G = GEOM[c["geom"]]
    cfg = gphq.lm_config(G["hidden"], len(model["layers"]), G["heads"], KV_HEADS, HD, G["inter"], vocab, MAX_POS,
                         FMT[c["fmt"]], EPS, THETA)
    desc, nbytes = gphq.lm_layer_layout(cfg)
    lm = gphq.Lm(cfg)
    for i, L in enumerate(model["layers"]):
        buf = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
        for name, at, sc in (("qkv", desc.qkv, desc.qkv_scale), ("o", desc.o, desc.o_scale),
                             ("gu", desc.gu, desc.gu_scale), ("down", desc.d, desc.d_scale)):
            for off, t in zip((at, sc), L[name]):
                b = t.reshape(-1).view(torch.uint8)
                buf[off:off + b.numel()] = b
        lm.bind_layer(i, buf, desc, L["q_norm"].cpu().numpy(), L["k_norm"].cpu().numpy())
    lm.bind_embed(model["embed"].view(torch.int16))
    rows, so, hb = gphq.lm_head_layout(cfg)
    head = torch.zeros(hb, dtype=torch.uint8, device="cuda")
    for off, t in zip((0, so), model["head"]):
        b = t.reshape(-1).view(torch.uint8)
        head[off:off + b.numel()] = b
    lm.bind_head(head, model["final_norm"].cpu().numpy())
    return lm


class _Rows:
    """Device memory of a prefix. A tensor made from it keeps this object, and so the prefix, alive."""

    def __init__(self, prefix, address, shape):
        self.prefix = prefix
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(address, False), version=2)


def _kv(prefix, layers):
    """Torch views of a prefix's K and V rows, [layers][capacity][KVD]."""
    k, v, cap = prefix.kv()
    return [torch.as_tensor(_Rows(prefix, a, (layers, cap, KVD)), device="cuda") for a in (k, v)]


def _cache_rows(g, layers, rows):
    return _randn(g, layers, rows, KVD), _randn(g, layers, rows, KVD)


def _io(c, g):
    """A projection's inputs and outputs: (x, y) as `project` takes them."""
    G = GEOM[c["geom"]]
    H, I, qd = G["hidden"], G["inter"], G["heads"] * HD
    k, n = [(H, qd + 2 * KVD), (qd, H), (H, I), (I, H)][c["proj"]]
    x = _acts(g, c["rows"], k)
    y = _randn(g, c["rows"], n) if c["proj"] in (1, 3) else torch.zeros((c["rows"], n), device="cuda")
    return x, y


def _ids(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    s = dict(case=c)
    if kind == "gemv":
        s["w"] = _matrix(g, c["fmt"], c["n"], c["k"])
        s["x"], s["y"] = _acts(g, 1, c["k"])[0], torch.empty(c["n"], device="cuda")
    elif kind == "gemv_batch":
        s["w"] = [_matrix(g, c["fmt"], c["n"], c["k"]) for _ in range(c["count"])]
        s["x"], s["y"] = _acts(g, c["count"], c["k"]), torch.empty((c["count"], c["n"]), device="cuda")
        s["args"] = [w[0] for w in s["w"]], [w[1] for w in s["w"]], list(s["x"]), list(s["y"])
    elif kind == "gemv_vec":
        s["w"] = _matrix(g, c["fmt"], c["n"], c["k"])
        s["x"], s["y"] = _acts(g, c["lanes"], c["k"]), torch.empty((c["lanes"], c["n"]), device="cuda")
        s["work"] = torch.empty(gphq.gemv_vec_workspace_bytes(c["lanes"], c["k"]), dtype=torch.uint8, device="cuda")
    elif kind == "i8":
        codes, scales, _ = _matrix(g, "q8", c["n"], c["k"])
        s["w"] = gphq.WeightsI8(c["k"], c["n"])
        s["w"].pack(codes.cpu().numpy().reshape(-1), scales.cpu().numpy().reshape(-1))
        s["ws"] = gphq.WorkspaceI8(c["k"], c["m"])
        s["x"], s["y"] = _acts(g, c["m"], c["k"]), torch.empty((c["m"], c["n"]), device="cuda")
    elif kind == "mm":
        s["w"] = _matrix(g, c["fmt"], c["n"], c["k"])
        s["x"], s["y"] = _acts(g, c["m"], c["k"]), torch.empty((c["m"], c["n"]), device="cuda")
        s["work"] = torch.empty(gphq.mm_split_workspace_bytes(c["m"], c["k"], c["n"]), dtype=torch.uint8, device="cuda")
    elif kind == "block32":
        s["w"] = _matrix(g, "q8b_f32", c["n"], c["k"])
        s["x"], s["y"] = _acts(g, c["m"], c["k"]), torch.empty((c["m"], c["n"]), device="cuda")
        s["q"] = torch.empty((c["m"], c["k"]), dtype=torch.int8, device="cuda")
        s["d"] = torch.empty((c["m"], c["k"] // 32), device="cuda")
    elif kind == "decode":
        s["lm"] = _bind(c, _model(g, c, c["layers"], VOCAB), VOCAB)
        s["ws"] = gphq.DecodeBatch(s["lm"], c["lanes"])
        s["kvs"] = [gphq.Prefix(s["lm"], c["ctx"] + 64) for _ in range(c["lanes"])]
        s["rows"] = []
        for p in s["kvs"]:
            for buf, rows in zip(_kv(p, c["layers"]), _cache_rows(g, c["layers"], c["ctx"])):
                buf[:, : c["ctx"]] = rows
                s["rows"].append(buf[:, c["ctx"]])
        s["pos"], s["ids"] = [c["ctx"]] * c["lanes"], _ids(seed, c["lanes"], VOCAB)
        s["hidden"] = torch.empty((c["lanes"], GEOM[c["geom"]]["hidden"]), device="cuda")
        s["logits"] = torch.empty((c["lanes"], VOCAB), device="cuda")
    elif kind == "prefill":
        s["lm"] = _bind(c, _model(g, c, c["layers"], PROMPT_VOCAB), PROMPT_VOCAB)
        s["ws"] = gphq.Prefill(s["lm"], c["tokens"])
        if c["route"] == "int8":
            s["ws"].set_arith(gphq.PASS_INT8)
        s["kv"] = gphq.Prefix(s["lm"], c["keep"] + c["tokens"])
        s["rows"] = []
        for buf, rows in zip(_kv(s["kv"], c["layers"]), _cache_rows(g, c["layers"], c["keep"])):
            buf[:, : c["keep"]] = rows
            s["rows"].append(buf[:, c["keep"]:])
        s["ids"] = _ids(seed, c["tokens"], PROMPT_VOCAB)
        s["hidden"] = torch.empty(GEOM[c["geom"]]["hidden"], device="cuda")
    elif kind == "project":
        s["lm"] = _bind(c, _model(g, c, 1, 256), 256)
        s["ws"] = gphq.Prefill(s["lm"], c["rows"])
        if c["route"] == "int8":
            s["ws"].set_arith(gphq.PASS_INT8)
        s["x"], s["y"] = _io(c, g)
        # proj 1 and 3 add into a residual: each pass starts from the same one.
        s["residual"] = s["y"].clone() if c["proj"] in (1, 3) else None
    else:
        s["x"] = _calibration(c, g)
        s["u"] = torch.empty((c["k"], c["k"]), device="cuda")
        s["dead"] = torch.empty(c["k"], dtype=torch.uint8, device="cuda")
    return s


def _calibration(c, g):
    """Calibration rows: channel scales over a decade, a shared low-rank part, a few dead channels."""
    x = _randn(g, c["rows"], c["k"]) * torch.exp(0.5 * _randn(g, c["k"]))
    x += 0.3 * (_randn(g, c["rows"], 16) @ _randn(g, 16, c["k"]))
    x[:, 11::509] = 0
    return x


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "gemv":
        gphq.gemv(FMT[c["fmt"]], s["w"][0], s["w"][1], s["x"], s["y"], c["k"], c["n"])
        return s["y"]
    if kind == "gemv_batch":
        gphq.gemv_batch(FMT[c["fmt"]], *s["args"], c["k"], c["n"])
        return s["y"]
    if kind == "gemv_vec":
        gphq.gemv_vec(FMT[c["fmt"]], s["w"][0], s["w"][1], s["x"], s["y"], c["lanes"], c["k"], c["n"], s["work"])
        return s["y"]
    if kind == "i8":
        s["ws"].pack(s["x"], c["m"], c["k"])
        gphq.mul_panels_i8(s["y"], c["n"], s["ws"], s["w"], 0, s["w"].panels())
        return s["y"]
    if kind == "mm":
        gphq.mm(FMT[c["fmt"]], s["w"][0], s["w"][1], s["x"], s["y"], c["m"], c["k"], c["n"], s["work"], zeros=s["w"][2])
        return s["y"]
    if kind == "block32":
        gphq.q8b_quantize(s["x"], c["m"], c["k"], s["q"], s["d"])
        gphq.q8b_gemm(s["q"], s["d"], s["w"][0], s["w"][1], s["y"], c["m"], c["k"], c["n"])
        return s["y"], s["q"], s["d"]
    if kind == "decode":
        s["ws"].into(s["kvs"], s["pos"], s["ids"], s["hidden"], s["logits"])
        return s["hidden"], s["logits"], s["rows"]
    if kind == "prefill":
        s["ws"].extend(s["kv"], c["keep"], s["ids"], s["hidden"])
        return s["hidden"], s["rows"]
    if kind == "project":
        if s["residual"] is not None:
            s["y"].copy_(s["residual"])
        s["ws"].project(0, c["proj"], s["x"], c["rows"], s["y"])
        return s["y"]
    gphq.gptq_factor(s["x"], c["rows"], c["k"], s["u"], s["dead"])
    return s["u"], s["dead"]


# ---- sizes and tolerances -------------------------------------------------------


def _bits(fmt, n, k):
    """Stored bytes of an n x k matrix: codes, scales, zero points."""
    return {"q8": n * k + 4 * n, "q8b": n * k + n * k // 16, "q8b_f32": n * k + n * k // 8,
            "q4": n * k // 2 + n * k // 16, "gptq4": n * k // 2 + 3 * n * k // 128}[fmt]


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "gemv_batch", "gemv_vec", "i8", "mm", "block32"):
        m, count = c.get("m", c.get("lanes", 1)), c.get("count", 1)
        fmt = {"i8": "q8", "block32": "q8b_f32"}.get(kind, c.get("fmt"))
        k, n = c["k"], c["n"]
        return dict(bytes=count * (_bits(fmt, n, k) + 4 * m * (k + n)), flops=2 * count * m * n * k)
    if kind == "gptq":
        k, r = c["k"], c["rows"]
        # H is symmetric (half the products); Cholesky and the inverse factor are k^3/3 multiply-adds each.
        return dict(bytes=4 * r * k + 4 * k * k, flops=r * k * k + 2 * k ** 3 / 3 + 2 * k ** 3 / 3)
    G = GEOM[c["geom"]]
    H, I, qd = G["hidden"], G["inter"], G["heads"] * HD
    shapes = [(qd + 2 * KVD, H), (H, qd), (2 * I, H), (H, I)]
    if kind == "project":
        n, k = shapes[c["proj"]]
        out = I if c["proj"] == 2 else n * (2 if c["proj"] in (1, 3) else 1)
        return dict(bytes=_bits(c["fmt"], n, k) + 4 * c["rows"] * (k + out), flops=2 * c["rows"] * n * k)
    rows = c["lanes"] if kind == "decode" else c["tokens"]
    past = c["ctx"] if kind == "decode" else c["keep"]
    weights = c["layers"] * sum(_bits(c["fmt"], n, k) for n, k in shapes)
    flops = 2 * rows * c["layers"] * sum(n * k for n, k in shapes)
    if kind == "decode":
        kv = rows * c["layers"] * 2 * KVD * 4 * (past + 1)
        flops += 2 * rows * VOCAB * H + 4 * rows * c["layers"] * qd * (past + 1)
        return dict(bytes=weights + _bits("q8b", VOCAB, H) + kv + rows * (6 * H + 4 * VOCAB), flops=flops)
    kv = c["layers"] * 2 * KVD * 4 * (past + rows)
    flops += 4 * c["layers"] * qd * (rows * past + rows * (rows + 1) // 2)
    return dict(bytes=weights + kv + rows * 2 * H, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind in ("i8", "block32"):
        return "exact"  # int32 sums and a fixed order of the fp32 scaling
    if kind in ("gemv", "gemv_batch", "gemv_vec"):
        return dict(rel=1e-5, max=1e-4)
    if kind == "decode":
        return dict(rel=2e-5, max=5e-4)
    if kind == "gptq":
        return dict(rel=6e-4, max=3e-2)  # the damped inverse amplifies float32 sums' rounding
    if kind == "project" and case["route"] == "int8":
        return dict(rel=2e-4, max=2e-2)  # a sum in another order moves a code at a rounding boundary
    if kind == "prefill":
        return dict(rel=8e-3, max=2e-1) if case["route"] == "int8" else dict(rel=2e-3, max=1e-1)
    return dict(rel=1e-3, max=2e-2)


# ---- the same results in 64 bits ------------------------------------------------


def _dequant(fmt, w, n, k):
    codes, scales, zeros = w
    if fmt == "q4":
        b = codes.view(n, k // 32, 16)
        v = torch.cat([b & 15, b >> 4], dim=2).double() - 8
        return (v * scales.double().view(n, -1, 1)).view(n, k)
    if fmt == "gptq4":
        b = codes.view(torch.uint8).view(n, k // 2, 1)
        v = torch.cat([b & 15, b >> 4], dim=2).view(n, k // 128, 128).double() - zeros.double().view(n, -1, 1)
        return (v * scales.double().view(n, -1, 1)).view(n, k)
    return (codes.double().view(n, scales.shape[1], -1) * scales.double().view(n, -1, 1)).view(n, k)


def _quantize(x):
    """Rows of x as (codes, step): step = max/127, codes round-half-even of x * (127/max), in float32."""
    m = x.abs().amax(dim=-1, keepdim=True)
    ok = (m > 0) & torch.isfinite(m)
    safe = torch.where(ok, m, torch.ones_like(m))
    q = (x * (127 / safe)).round().clamp(-128, 127)
    return torch.where(ok, q, torch.zeros_like(q)), torch.where(ok, safe / 127, torch.zeros_like(m))


def _signs(width):
    """The model rotation's signs (splitmix64 from the golden ratio xor the width), its block and scale."""
    mask, state, out = (1 << 64) - 1, 0x9E3779B97F4A7C15 ^ width, []
    for _ in range(width):
        state = (state + 0x9E3779B97F4A7C15) & mask
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        out.append(-1.0 if (z ^ (z >> 31)) & 1 else 1.0)
    block = 1
    while block < 4096 and width % (2 * block) == 0:
        block *= 2
    return torch.tensor(out, dtype=torch.float64, device="cuda"), block


def _hadamard(v, block):
    shape, h = v.shape, 1
    while h < block:
        v = v.reshape(-1, 2, h)
        v = torch.stack([v[:, 0] + v[:, 1], v[:, 0] - v[:, 1]], dim=1)
        h *= 2
    return v.reshape(shape)


def _rotate(v, rot):
    signs, block = rot
    return _hadamard(v * signs, block) / block ** 0.5


def _unrotate(v, rot):
    signs, block = rot
    return _hadamard(v, block) * signs / block ** 0.5


def _rms(v):
    return v / (v.square().mean(dim=-1, keepdim=True) + EPS).sqrt()


def _product(x, w, route):
    if route == "int8":
        q, step = _quantize(x.float())
        x = q.double() * step.double()
    return x @ w.T


def _projection(c, w, proj, x, rot):
    """One projection of a pass on float64 rows: norm, product, SwiGLU or rotation as the pass has it."""
    if proj in (0, 2):
        x = _rms(x)
    if proj == 3 and c["fmt"] != "q8b":
        x = _rotate(x, rot)
    out = _product(x, w, c.get("route", "fp16"))
    if proj == 2:
        gate, up = out[:, 0::2], out[:, 1::2]
        out = gate * torch.sigmoid(gate) * up
    return out


def _rope(x, pos):
    inv = 1.0 / THETA ** (torch.arange(64, dtype=torch.float64, device="cuda") / 64)
    ang = pos.double()[:, None] * inv
    cos, sin = ang.cos().float().double()[:, None], ang.sin().float().double()[:, None]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attend(q, k, v, past):
    """q [rows][heads][128] at positions past.., over k, v [past + rows][8][128]."""
    rows, heads = q.shape[:2]
    mask = torch.arange(past + rows, device="cuda")[None] > past + torch.arange(rows, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        kh = h // (heads // KV_HEADS)
        s = (q[:, h] @ k[:, kh].T / HD ** 0.5).masked_fill(mask, -torch.inf)
        out[:, h] = s.softmax(dim=1) @ v[:, kh]
    return out.reshape(rows, -1)


def _forward(c, model, ids, caches, past):
    """Every layer in float64: one sequence (a pass) or one row per cache (decode lanes).
    Returns (residual, [K rows, V rows per cache])."""
    G = GEOM[c["geom"]]
    heads, qd = G["heads"], G["heads"] * HD
    hrot, irot = _signs(G["hidden"]), _signs(G["inter"])
    h = _rotate(model["embed"][torch.from_numpy(np.asarray(ids)).cuda()].double(), hrot)
    rows = h.shape[0] // len(caches)
    new = [[[], []] for _ in caches]
    for i, L in enumerate(model["layers"]):
        dense = lambda name, n, k: _dequant(c["fmt"], L[name], n, k)  # noqa: E731
        qkv = _projection(c, dense("qkv", qd + 2 * KVD, G["hidden"]), 0, h, None)
        ctx = []
        for j, (kc, vc) in enumerate(caches):
            pos = past + torch.arange(rows, device="cuda")
            one = qkv[j * rows:(j + 1) * rows]
            q = _rope(_rms(one[:, :qd].view(rows, heads, HD)) * L["q_norm"].double(), pos)
            k = _rope(_rms(one[:, qd:qd + KVD].view(rows, KV_HEADS, HD)) * L["k_norm"].double(), pos)
            v = one[:, qd + KVD:]
            new[j][0].append(k.reshape(rows, KVD))
            new[j][1].append(v)
            keys = torch.cat([kc[i].double().view(-1, KV_HEADS, HD), k])
            values = torch.cat([vc[i].double(), v]).view(-1, KV_HEADS, HD)
            ctx.append(_attend(q, keys, values, past))
        h = h + _projection(c, dense("o", G["hidden"], qd), 1, torch.cat(ctx), None)
        act = _projection(c, dense("gu", 2 * G["inter"], G["hidden"]), 2, h, None)
        h = h + _projection(c, dense("down", G["hidden"], G["inter"]), 3, act, irot)
    return h, [torch.stack(t) for pair in new for t in pair]


def _inverse_factor(c, x):
    """U upper triangular with H^-1 = U^T U, H the damped Gram matrix of x, and the dead channels."""
    x = x.double()
    h = x.T @ x
    d = h.diagonal()
    dead = d == 0
    d[dead] = 1
    d += 0.01 * d.mean()
    inv = torch.cholesky_inverse(torch.linalg.cholesky(h.cpu()))
    return torch.linalg.cholesky(inv, upper=True), dead.to(torch.uint8)


def exact(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind in ("gemv", "gemv_vec", "mm"):
        w = _dequant(c["fmt"], _matrix(g, c["fmt"], c["n"], c["k"]), c["n"], c["k"])
        y = _acts(g, c.get("m", c.get("lanes", 1)), c["k"]).double() @ w.T
        return y[0] if kind == "gemv" else y
    if kind == "gemv_batch":
        w = [_matrix(g, c["fmt"], c["n"], c["k"]) for _ in range(c["count"])]
        x = _acts(g, c["count"], c["k"]).double()
        return torch.stack([_dequant(c["fmt"], w[i], c["n"], c["k"]) @ x[i] for i in range(c["count"])])
    if kind == "i8":
        w = _dequant("q8", _matrix(g, "q8", c["n"], c["k"]), c["n"], c["k"])
        return _product(_acts(g, c["m"], c["k"]).double(), w, "int8")
    if kind == "block32":
        w = _dequant("q8b_f32", _matrix(g, "q8b_f32", c["n"], c["k"]), c["n"], c["k"])
        q, d = _quantize(_acts(g, c["m"], c["k"]).view(c["m"], -1, 32))
        return (q.double() * d.double()).view(c["m"], -1) @ w.T, None, d.double()[:, :, 0]
    if kind == "gptq":
        return _inverse_factor(c, _calibration(c, g))
    G = GEOM[c["geom"]]
    if kind == "project":
        H, I, qd = G["hidden"], G["inter"], G["heads"] * HD
        n, k = [(qd + 2 * KVD, H), (H, qd), (2 * I, H), (H, I)][c["proj"]]
        L = _model(g, c, 1, 256)["layers"][0]
        x, y = _io(c, g)
        w = _dequant(c["fmt"], L[["qkv", "o", "gu", "down"][c["proj"]]], n, k)
        out = _projection(c, w, c["proj"], x.double(), _signs(I))
        return y.double() + out if c["proj"] in (1, 3) else out
    vocab = VOCAB if kind == "decode" else PROMPT_VOCAB
    model = _model(g, c, c["layers"], vocab)
    lanes, rows = (c["lanes"], 1) if kind == "decode" else (1, c["tokens"])
    past = c["ctx"] if kind == "decode" else c["keep"]
    caches = [_cache_rows(g, c["layers"], past) for _ in range(lanes)]
    h, new = _forward(c, model, _ids(seed, lanes * rows, vocab), caches, past)
    hrot = _signs(G["hidden"])
    last = h if kind == "decode" else h[-1:]
    hidden = _rms(_unrotate(last, hrot)) * model["final_norm"].double()
    if kind == "prefill":
        return hidden[0], new
    x, (codes, scales, _) = _rotate(hidden, hrot), model["head"]
    logits = [x @ _dequant("q8b", (codes[r:r + 16384], scales[r:r + 16384], None), min(16384, len(codes) - r), G["hidden"]).T
              for r in range(0, len(codes), 16384)]
    return hidden, torch.cat(logits, dim=1)[:, :VOCAB], [t[:, 0] for t in new]
