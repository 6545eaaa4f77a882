"""The work that a program using this framework gives it: dynamically quantized linears, the
int8 matrix product, the fp32 ops around them (elementwise chains, LayerNorm, attention) and
whole encoder forwards, each through its public entry point.

A case is a dict of plain values; ``kind`` selects the path:

  linear          DynamicQuantizeLinear(x), then MatMulInteger with a weight packed once and
                  the dequant / bias / elementwise epilogue (ops.gpu_dynamic_quantize_linear
                  and ops.gpu_qlinear)
  dequant_gemm    ops.gpu_qlinear over an activation that is uint8 already
  matmul_integer  ops.gpu_matmul_integer of two plain tensors, int32 out
  chain           ops.gpu_fused_chain
  layer_norm      ops.gpu_layer_norm (with a residual or without)
  attention       ops.gpu_attention (heads of 64)
  attention_graph the exported self-attention subgraph in a GpuGraphExecutor, captured once
                  and replayed, for any head size
  encoder         the exported DistilBERT-shaped encoder (Int64 ids and padding mask, 6 layers,
                  hidden 768) in a GpuGraphExecutor: captured and replayed, or run eagerly
"""
import functools

import numpy as np
import torch

from iconnx_amd import graphs, ops
from iconnx_amd.executor import GpuGraphExecutor

LAYERS, HIDDEN, HEADS, FFN, VOCAB, EPS = 6, 768, 12, 3072, 30522, 1e-12


def listed():
    return [
        # a pooled batch through a classifier's first linear: 16 rows, nothing but latency
        dict(name="linear_pooled", kind="linear", M=16, K=768, N=768, weight="int8", epilogue="bias"),
        # the FFN-down projection of one short text
        dict(name="linear_short_text", kind="linear", M=100, K=3072, N=768, weight="int8", epilogue="bias"),
        # the FFN-up projection of a DistilBERT batch (32 x 128 tokens) and a chain after it
        dict(name="linear_ffn_up", kind="linear", M=4096, K=768, N=3072, weight="int8", epilogue="chain"),
        # a BERT-large batch (64 x 384 tokens), weights with a scale and zero point per column
        dict(name="linear_per_channel", kind="linear", M=24576, K=1024, N=4096, weight="per_channel",
             epilogue="bias"),
        # two plain tensors of sizes that fit no tile, uint8 by uint8 with zero points
        dict(name="matmul_integer_ragged", kind="matmul_integer", M=1530, K=1000, N=1500, a="uint8", b="uint8",
             zero_points=True),
        # the largest product: 16384 x 4096 by 4096 x 4096, dequantized
        dict(name="gemm_large", kind="dequant_gemm", M=16384, K=4096, N=4096),
        # the elementwise chain alone over 65536 rows
        dict(name="chain", kind="chain", rows=65536, cols=768, residual=False),
        # the residual LayerNorm of a small-model batch (32 x 384 tokens, hidden 384)
        dict(name="layer_norm_residual", kind="layer_norm", rows=12288, cols=384, residual=True),
        # BERT-large's self-attention over 384 tokens
        dict(name="attention_long", kind="attention", B=64, S=384, H=16),
        # the exported self-attention of a small model: 12 heads of 32, 32 x 128 tokens
        dict(name="attention_heads_of_32", kind="attention_graph", B=32, S=128, H=12, D=32),
        # a whole encoder forward over a batch, recorded once and replayed for every batch
        dict(name="encoder_batch", kind="encoder", B=32, S=128, replay=True),
        # one short text through the whole encoder, run eagerly (its length changes per call)
        dict(name="encoder_one_text", kind="encoder", B=1, S=37, replay=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi + 1))))))


def _feature_size(rng, lo, hi):
    """A feature dimension: mostly multiples of 64, some of 8 or 16, some odd."""
    n, step = _log_int(rng, lo, hi), rng.choice([128, 128, 64, 64, 16, 8, 1])
    return max(lo, min(hi, n // step * step if n >= step else n))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "dequant_gemm", "matmul_integer", "matmul_integer", "chain",
                       "layer_norm", "attention", "attention_graph", "encoder"])
    if kind in ("linear", "dequant_gemm", "matmul_integer"):
        K, N = _feature_size(rng, 64, 4096), _feature_size(rng, 64, 4096)
        M = _log_int(rng, 1, min(24576, (1 << 36) // (K * N), (96 << 20) // N))
        case = dict(kind=kind, M=M, K=K, N=N)
        if kind == "linear":
            case.update(weight=rng.choice(["int8", "int8", "per_channel", "uint8"]),
                        epilogue=rng.choice(["bias", "bias", "chain", "gelu"]))
        elif kind == "matmul_integer":
            case.update(a=rng.choice(["uint8", "int8"]), b=rng.choice(["int8", "uint8"]),
                        zero_points=rng.random() < 0.5)
        return case
    if kind in ("chain", "layer_norm"):
        cols = _feature_size(rng, 64, 4096)
        return dict(kind=kind, rows=_log_int(rng, 1, min(65536, (40 << 20) // cols)), cols=cols,
                    residual=rng.random() < 0.5)
    if kind == "attention":
        S, H = _log_int(rng, 16, 1024), rng.choice([1, 8, 12, 16])
        return dict(kind=kind, B=_log_int(rng, 1, max(1, min(64, (1 << 27) // (S * S * H)))), S=S, H=H)
    if kind == "attention_graph":
        S, H, D = _log_int(rng, 16, 512), rng.choice([4, 8, 12, 16]), rng.choice([32, 32, 40, 80, 96, 128])
        return dict(kind=kind, B=_log_int(rng, 1, max(1, min(64, (1 << 31) // (S * S * H * D)))), S=S, H=H, D=D)
    S = _log_int(rng, 8, 256)
    return dict(kind=kind, B=_log_int(rng, 1, max(1, 4096 // S)), S=S, replay=rng.random() < 0.5)


# ---- inputs and weights -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _normal(g, shape, mean=0.0, std=1.0):
    return torch.randn(shape, generator=g, device="cuda").mul_(std).add_(mean)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda").mul_(hi - lo).add_(lo)


def _ints(g, shape, name):
    dt = torch.int8 if name == "int8" else torch.uint8
    lo, hi = (-127, 128) if name == "int8" else (0, 256)
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32).to(dt)


def _const(v, dtype=torch.float32):
    return torch.tensor(v, dtype=dtype, device="cuda")


def _chain_constants(g, n):
    return [("Mul", _normal(g, (n,), 1.0, 0.1)), ("Add", _normal(g, (n,), 0.0, 0.1)),
            ("Div", _uniform(g, (n,), 1.5, 2.5)), ("Mul", _normal(g, (n,), 0.5, 0.1))]


def _linear_inputs(case, seed):
    g = _gen(seed)
    M, K, N = case["M"], case["K"], case["N"]
    per_channel = case["weight"] == "per_channel"
    d = dict(x=_normal(g, (M, K), 0.5 if per_channel else 0.0), bias=_normal(g, (N,), 0.0, 0.02))
    d["w"] = _ints(g, (K, N), "uint8" if case["weight"] == "uint8" else "int8")
    d["w_scale"], d["w_zp"] = _const(0.25 / K ** 0.5 / 20), None
    if per_channel:
        d["w_scale"] = _uniform(g, (N,), 0.005, 0.03)
        d["w_zp"] = torch.randint(-8, 9, (N,), generator=g, device="cuda", dtype=torch.int32).to(torch.int8)
    elif case["weight"] == "uint8":
        d["w_zp"] = _const(131, torch.uint8)
    d["chain"] = []
    if case["epilogue"] == "chain":
        d["chain"] = [(op, c, False) for op, c in _chain_constants(g, N)]
    elif case["epilogue"] == "gelu":
        d["chain"] = [("Save", None, False), ("Div", _const(1.4142135381698608), False), ("Erf", None, False),
                      ("Add", _const(1.0), False), ("MulSaved", None, False), ("Mul", _const(0.5), False)]
    return d


def _product_inputs(case, seed):
    g = _gen(seed)
    M, K, N = case["M"], case["K"], case["N"]
    if case["kind"] == "dequant_gemm":
        return dict(a=_ints(g, (M, K), "uint8"), b=_ints(g, (K, N), "int8"), a_zp=_const(128, torch.uint8),
                    b_zp=None, scales=(_const(0.0125), _const(0.01)))
    d = dict(a=_ints(g, (M, K), case["a"]), b=_ints(g, (K, N), case["b"]), a_zp=None, b_zp=None)
    if case["zero_points"]:
        d["a_zp"] = _const(121 if case["a"] == "uint8" else 3, d["a"].dtype)
        d["b_zp"] = _const(131 if case["b"] == "uint8" else -5, d["b"].dtype)
    return d


def _rows_inputs(case, seed):
    g = _gen(seed)
    rows, cols = case["rows"], case["cols"]
    d = dict(x=_normal(g, (rows, cols)), residual=_normal(g, (rows, cols)) if case["residual"] else None)
    if case["kind"] == "chain":
        d["ops"] = [(op, c, False) for op, c in _chain_constants(g, cols)]
        if case["residual"]:
            d["ops"].append(("Add", d["residual"], False))
    else:
        d["scale"], d["bias"] = _uniform(g, (cols,), 0.9, 1.1), _normal(g, (cols,), 0.0, 0.02)
    return d


def _head_size(case):
    return case.get("D", 64)


def _attention_inputs(case, seed):
    g = _gen(seed)
    shape = (case["B"], case["S"], case["H"] * _head_size(case))
    return [_normal(g, shape) for _ in range(3)]


class _Recorder:
    """Records a graph's add_* calls (one model, loaded once) for any number of executors."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if not name.startswith("add_"):
            raise AttributeError(name)
        return lambda *a: self.calls.append((name, a))

    def executor(self):
        ex = GpuGraphExecutor()
        for name, a in self.calls:
            getattr(ex, name)(*a)
        return ex


@functools.lru_cache(maxsize=1)
def _encoder_model():
    rec = _Recorder()
    out, _, params, emb = graphs.export_encoder_graph(rec, LAYERS, HEADS, HIDDEN, FFN, EPS, VOCAB)
    return rec, out, params, emb


def _encoder_inputs(case, seed):
    g = _gen(seed)
    B, S = case["B"], case["S"]
    ids = torch.randint(0, VOCAB, (B, S), generator=g, device="cuda")
    lens = torch.randint(max(1, S // 4), S + 1, (B, 1), generator=g, device="cuda")
    lens[0] = S
    return ids, (torch.arange(S, device="cuda")[None, :] < lens).to(torch.int64)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        d = _linear_inputs(case, seed)
        d["w"] = ops.PackedWeight(d["w"])
    elif kind == "dequant_gemm":
        d = _product_inputs(case, seed)
        d["b"] = ops.PackedWeight(d["b"])
    elif kind == "matmul_integer":
        d = _product_inputs(case, seed)
    elif kind in ("chain", "layer_norm"):
        d = _rows_inputs(case, seed)
    elif kind == "attention":
        d = dict(qkv=_attention_inputs(case, seed))
    elif kind == "attention_graph":
        q, k, v = _attention_inputs(case, seed)
        ex = GpuGraphExecutor()
        for n in ("q", "k", "v"):
            ex.add_input(n, [None, None, q.shape[-1]])
        out = graphs.add_self_attention(ex, "q", "k", "v", case["H"], case["D"], "attn")
        d = dict(ex=ex, out=out, inputs=dict(q=q, k=k, v=v))
        ex.capture(d["inputs"], [out])
    else:
        ids, mask = _encoder_inputs(case, seed)
        rec, out, _, _ = _encoder_model()
        d = dict(ex=rec.executor(), out=out, inputs=dict(input_ids=ids, attention_mask=mask))
        if case["replay"]:
            d["ex"].capture(d["inputs"], [out])
        else:  # weights uploaded and packed; the shapes of a call are not known before it
            d["ex"].add_output(out)
            d["ex"].compile()
    d["case"] = case
    return d


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        # a weight with a zero point reads the activation's row sums, which DQL leaves
        zp = state["w_zp"]
        q = ops.gpu_dynamic_quantize_linear(state["x"], case["K"] if zp is not None else None)
        y = ops.gpu_qlinear(q[0], state["w"], q[2], zp, a_rowsum=q[3] if zp is not None else None,
                            epilogue=[("Mul", (q[1], state["w_scale"]), False), ("Add", state["bias"], False)]
                            + state["chain"])
        return q[0], q[1], q[2], y
    if kind == "dequant_gemm":
        return ops.gpu_qlinear(state["a"], state["b"], state["a_zp"], epilogue=[("Mul", state["scales"], False)])
    if kind == "matmul_integer":
        return ops.gpu_matmul_integer(state["a"], state["b"], state["a_zp"], state["b_zp"])
    if kind == "chain":
        return ops.gpu_fused_chain(state["x"], state["ops"])
    if kind == "layer_norm":
        return ops.gpu_layer_norm(state["x"], state["scale"], state["bias"], EPS, state["residual"])
    if kind == "attention":
        return ops.gpu_attention(*state["qkv"], heads=case["H"], scale=8.0)
    ex, out = state["ex"], state["out"]
    if kind == "encoder" and not case["replay"]:
        return ex.run_device(state["inputs"], [out])[out]
    ex.replay()
    return ex.outputs([out])[out]


# ---- what a pass cannot do without --------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("linear", "dequant_gemm", "matmul_integer"):
        M, K, N = case["M"], case["K"], case["N"]
        # linear: x in, its quantization out; then the weight in and the result out
        a = 5 * M * K if kind == "linear" else M * K
        return dict(bytes=a + K * N + 4 * M * N, flops=2 * M * K * N)
    if kind in ("chain", "layer_norm"):
        n = case["rows"] * case["cols"]
        return dict(bytes=(12 if case["residual"] else 8) * n, flops=8 * n)
    B, S = case["B"], case["S"]
    if kind == "encoder":
        T, h = B * S, HIDDEN
        weights = LAYERS * (4 * h * h + 2 * h * FFN)
        return dict(bytes=weights + T * (16 + h + 4 * h), flops=2 * T * weights + LAYERS * 4 * B * S * S * h)
    hd = case["H"] * _head_size(case)
    return dict(bytes=16 * B * S * hd, flops=4 * B * S * S * hd)


def tolerance(case):
    kind = case["kind"]
    if kind == "matmul_integer":
        return "exact"
    # each about four times what the path shows against the same arithmetic in 64 bits
    if kind == "encoder":
        # a last-bit change ahead of one of the 36 quantizations moves some values by a whole
        # step of it, and every later layer sees those (2 to 3e-2)
        return dict(rel=0.1, max=0.6)
    if kind in ("attention", "attention_graph"):  # sums and exponentials in 32 bits: 5e-7, 4e-6
        return dict(rel=2e-6, max=2e-5)
    if kind == "linear":  # the epilogue's roundings, erf's formula with them: 1.2e-7, 4e-7
        return dict(rel=5e-7, max=2e-6)
    return dict(rel=4e-7, max=1.6e-6)  # a rounding per operation: 9e-8, 4e-7


# ---- the same results in 64 bits ----------------------------------------------------------
def _dql64(x):
    x = x.double()
    lo, hi = x.min().clamp(max=0.0), x.max().clamp(min=0.0)
    s = (hi - lo) / 255.0
    zp = torch.round(-lo / s).clamp(0, 255)
    return (torch.round(x / s) + zp).clamp(0, 255), s, zp


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / 2.0 ** 0.5))


def _attention64(q, k, v, H, mask=None):
    B, S, HD = q.shape
    q, k, v = (t.double().view(B, S, H, HD // H).transpose(1, 2) for t in (q, k, v))
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / (HD // H) ** 0.5
    if mask is not None:
        s = s.masked_fill(mask[:, None, None, :] == 0, torch.finfo(torch.float32).min)
    return torch.matmul(torch.softmax(s, -1), v.contiguous()).transpose(1, 2).reshape(B, S, HD)


def _norm64(x, scale, bias):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + EPS) * scale.double() + bias.double()


def _encoder64(case, seed):
    dev = lambda a: torch.from_numpy(np.array(a)).cuda().double()  # noqa: E731
    _, _, params, emb = _encoder_model()
    ids, mask = _encoder_inputs(case, seed)
    x = (torch.from_numpy(emb["word"]).cuda()[ids].double() - float(emb["zp"])) * float(emb["scale"])
    x = _norm64(x + dev(emb["pos"])[:case["S"]], dev(emb["ln"]["scale"]), dev(emb["ln"]["bias"]))

    def linear(q, p):
        xq, s, zp = q
        return torch.matmul(xq - zp, dev(p["w"])) * s * float(p["w_scale"]) + dev(p["bias"])

    for p in params:
        q = _dql64(x)
        ctx = _attention64(*(linear(q, p[n]) for n in ("q", "k", "v")), H=HEADS, mask=mask)
        x = _norm64(linear(_dql64(ctx), p["o"]) + x, dev(p["ln1"]["scale"]), dev(p["ln1"]["bias"]))
        h = _gelu64(linear(_dql64(x), p["ff1"]))
        x = _norm64(linear(_dql64(h), p["ff2"]) + x, dev(p["ln2"]["scale"]), dev(p["ln2"]["bias"]))
    return x


def _apply64(y, chain):
    for op, c, _ in chain:
        c = c.double()
        y = y * c if op == "Mul" else y + c if op == "Add" else y / c
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        d = _linear_inputs(case, seed)
        xq, s, zp = _dql64(d["x"])
        w = d["w"].double()
        if d["w_zp"] is not None:
            w = w - d["w_zp"].double()
        y = torch.matmul(xq - zp, w) * (s * d["w_scale"].double()) + d["bias"].double()
        y = _gelu64(y) if case["epilogue"] == "gelu" else _apply64(y, d["chain"])
        return xq.to(torch.uint8), s, zp.to(torch.uint8), y
    if kind in ("dequant_gemm", "matmul_integer"):
        d = _product_inputs(case, seed)
        a, b = d["a"].double(), d["b"].double()
        if d["a_zp"] is not None:
            a = a - d["a_zp"].double()
        if d["b_zp"] is not None:
            b = b - d["b_zp"].double()
        y = torch.matmul(a, b)
        if kind == "matmul_integer":
            return y.to(torch.int32)
        return y * (d["scales"][0].double() * d["scales"][1].double())
    if kind == "chain":
        d = _rows_inputs(case, seed)
        return _apply64(d["x"].double(), d["ops"])
    if kind == "layer_norm":
        d = _rows_inputs(case, seed)
        x = d["x"].double()
        return _norm64(x if d["residual"] is None else x + d["residual"].double(), d["scale"], d["bias"])
    if kind in ("attention", "attention_graph"):
        q, k, v = _attention_inputs(case, seed)
        if case["H"] * case["B"] * case["S"] ** 2 > 1 << 28:
            return None
        return _attention64(q, k, v, case["H"])
    return _encoder64(case, seed)
