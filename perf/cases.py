"""What the framework's users run, as timed cases.

A case is one call path through the public Python entry points: the quantized
products of `mivi_hip` (matvec, row products, dequantization), the device
sampler, and the hybrid model (`mivi_hip.Model`, `mivi_hip.PrefixCache`).
Shapes are those of the 1.2B hybrid model (dim 2048, FFN 8192, 32 query and 8
kv heads of 64, vocabulary 65536) and of the loader's default configuration
(dim 1024, FFN 4608), with ragged batches and lengths between them.

`exact` restates each path in 64 bits from the stored bytes of the weights and
caches; it uses the package only to produce those inputs.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mivi-v4_amd"))

import mivi_hip  # noqa: E402
from mivi_hip import GgmlType, KvPrecision  # noqa: E402
from mivi_hip.gguf import read_tensor_index  # noqa: E402
from mivi_hip.synthmodel import build_hybrid, q6k_matrices  # noqa: E402

TYPES = {"q4_k": GgmlType.Q4_K, "q6_k": GgmlType.Q6_K, "q8_0": GgmlType.Q8_0, "f16": GgmlType.F16,
         "bf16": GgmlType.BF16, "f32": GgmlType.F32}
KV = {"f32": KvPrecision.F32, "f16": KvPrecision.F16, "q8_0": KvPrecision.Q8_0}
FULL_ATTN = (2, 5, 8, 11, 13, 15)  # attention layers of the 16-layer model
SAMPLERS = {
    # GenerationConfig::default, plain categorical sampling, nucleus without a
    # top-k, and the penalised greedy choice
    "default": dict(),
    "categorical": dict(temperature=0.8, top_p=1.0, top_k=0, repetition_penalty=1.0),
    "nucleus": dict(temperature=0.7, top_p=0.95, top_k=0),
    "greedy": dict(temperature=0.0, repetition_penalty=1.1),
}


def listed():
    return [
        # one small projection of a decode step on the weights as the file holds
        # them (attn_k of the 1.2B model): all latency
        dict(name="matvec_q4k_small", kind="matvec", type="q4_k", rows=512, cols=2048, packed=False),
        # the tied output head of an unquantized model of the default
        # configuration, one token
        dict(name="matvec_bf16_head", kind="matvec", type="bf16", rows=65536, cols=1024, packed=False),
        # the 1.2B model's output head, packed once at load, one token
        dict(name="head_q6k_packed", kind="matvec", type="q6_k", rows=65536, cols=2048, packed=True),
        # a weight matrix decoded to f32 (an embedding or adapter merge), an
        # odd number of rows
        dict(name="dequant_q6k", kind="dequant", type="q6_k", rows=12289, cols=2048),
        # FFN gate / up of one 512-token prefill tile, weights converted at load
        dict(name="rows_q4k_tile", kind="rows", type="q4_k", batch=512, rows=8192, cols=2048, packed=True),
        # FFN down of a mixed-format file over a ragged prompt, weights as the
        # file holds them
        dict(name="rows_q6k_ragged", kind="rows", type="q6_k", batch=333, rows=2048, cols=8192, packed=False),
        # FFN gate of the default configuration over a short prompt
        dict(name="rows_q4k_dim1024", kind="rows", type="q4_k", batch=200, rows=4608, cols=1024, packed=False),
        # an output projection of a Q8_0 file over a short prompt
        dict(name="rows_q8_0", kind="rows", type="q8_0", batch=128, rows=2048, cols=2048, packed=False),
        # the next token of eight sequences, the default sampling settings
        dict(name="sample_8", kind="sample", rows=8, n=65536, sampler="default", recent=64),
        # a prompt through the 1.2B model in tiles of 512 (a ragged last one),
        # then the next token's logits
        dict(name="prefill_1b2", kind="prefill", dim=2048, hidden=8192, layers=16, heads=32, kv_heads=8, vocab=65536,
             weights="q4_k", kv="f16", tokens=2500, tile=512, max_ctx=4096),
        # a cached prompt restored, then a few tokens one at a time with their
        # logits (one user)
        dict(name="decode_1b2", kind="decode", dim=2048, hidden=8192, layers=16, heads=32, kv_heads=8, vocab=65536,
             weights="q4_k", kv="f16", batch=1, cached=4000, steps=8, max_ctx=4096),
        # the same for eight users on long Q8_0 caches, a batch a step
        dict(name="decode_batch8", kind="decode", dim=2048, hidden=8192, layers=16, heads=32, kv_heads=8, vocab=65536,
             weights="q4_k", kv="q8_0", batch=8, cached=8192, steps=4, max_ctx=8448),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "dequant", "rows", "rows", "rows", "sample", "prefill", "prefill", "decode"])
    if kind == "matvec":
        t = rng.choice(list(TYPES))
        cols = rng.choice([1024, 1536, 2048, 2048, 4096, 4608, 8192])
        if t in ("f16", "bf16", "f32") and rng.random() < 0.3:
            cols += rng.randrange(1, 64)
        rows = _log(rng, 64, (120 << 20) // (cols * (4 if t == "f32" else 2)))
        packed = (t == "q6_k" and cols in (2048, 4096, 8192) or t == "q4_k" and cols in (2048, 8192)) and rng.random() < 0.6
        return dict(kind=kind, type=t, rows=rows // 4 * 4 if packed else rows, cols=cols, packed=packed)
    if kind == "dequant":
        return dict(kind=kind, type=rng.choice(["q4_k", "q6_k", "q8_0", "f16", "bf16"]), rows=_log(rng, 1, 16000),
                    cols=rng.choice([1024, 2048, 4608]))
    if kind == "rows":
        t = rng.choice(["q4_k", "q4_k", "q6_k", "q6_k", "q8_0", "f16", "bf16"])
        cols = rng.choice([1024, 1536, 2048, 2048, 4096, 4608, 8192])
        rows = rng.choice([512, 1024, 2048, 4608, 6144, 8192, _log(rng, 100, 8192)])
        packed = t == "q4_k" and cols % 2048 == 0 and rows % 32 == 0 and rng.random() < 0.6
        return dict(kind=kind, type=t, batch=_log(rng, 2, 512), rows=rows, cols=cols, packed=packed)
    if kind == "sample":
        return dict(kind=kind, rows=rng.randint(1, 8), n=_log(rng, 4000, 65536), sampler=rng.choice(list(SAMPLERS)),
                    recent=rng.choice([0, 17, 64]))
    dim, hidden, heads = rng.choice([(2048, 8192, 32), (2048, 8192, 32), (1024, 4608, 16)])
    case = dict(kind=kind, dim=dim, hidden=hidden, layers=rng.randint(2, 6), heads=heads, kv_heads=8,
                vocab=rng.choice([8192, 10007, 32768]))
    if kind == "prefill":
        case["weights"] = rng.choice(["q4_k", "q4_k", "q4_k_m", "q8_0"])
        case["kv"] = rng.choice(["f16", "f16", "q8_0", "f32"])
        case["tokens"] = _log(rng, 20, 256 if case["weights"] == "q8_0" else 4000)
        case["tile"] = rng.choice([64, 256, 512, 512])
    else:
        case["weights"] = rng.choice(["q4_k", "q4_k", "q4_k_m"])
        case["kv"] = rng.choice(["f16", "q8_0", "f32"])
        case["batch"] = rng.choice([1, 1, 2, 3, 5, 8])
        case["cached"] = 16 * _log(rng, 4, 250)
        case["steps"] = rng.randint(1, 8)
    case["max_ctx"] = 4096
    return case


# ------------------------------------------------------------------ inputs

def _weights(t, seed, rows, cols):
    """rows x cols of N(0, 0.02) in the stored format (host bytes)."""
    if t == "f32":
        return mivi_hip.synth_normal(seed, rows * cols, 0.0, 0.02).view(np.uint8)
    if t in ("f16", "bf16"):
        g = torch.Generator(device="cuda").manual_seed(seed)
        w = torch.randn(rows * cols, generator=g, device="cuda", dtype=torch.float32) * 0.02
        return w.to(torch.float16 if t == "f16" else torch.bfloat16).view(torch.uint8)
    return mivi_hip.synth_random_weights(TYPES[t], seed, rows, cols, 0.02)


def _device(raw):
    return raw if isinstance(raw, torch.Tensor) else torch.from_numpy(raw).cuda()


def _activations(seed, *shape):
    """N(0, 1) activations, what follows an RMSNorm."""
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float32).cuda()


def _logits(seed, rows, n):
    """Head outputs: N(0, 1.5) with a few tokens that stand out."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, n, generator=g) * 1.5
    top = torch.randint(0, n, (rows, 12), generator=g)
    x.scatter_add_(1, top, torch.rand(rows, 12, generator=g) * 6.0)
    return x.cuda()


def _image(case, seed):
    layers = case["layers"]
    attn = FULL_ATTN if layers == 16 else tuple(i for i in range(layers) if i % 3 == 1)
    mixed = "q4_k_m" if case["weights"] == "q4_k_m" else None
    wt = GgmlType.Q8_0 if case["weights"] == "q8_0" else GgmlType.Q4_K
    img = build_hybrid(case["dim"], case["hidden"], layers, attn, case["heads"], case["kv_heads"], case["vocab"],
                       weight_type=wt, seed=1 + seed % 100003, mixed=mixed)
    return img, attn


def _prompt(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n, dtype=np.uint32)


def _kv_rows(case, n_attn, seed):
    """A cached prompt: K and V rows ([attention layer][token][kv_dim]) of
    N(0, 0.9), as the projections of normalised rows give them, in the cache's
    precision (host bytes), and the ShortConv state."""
    kvd = case["kv_heads"] * (case["dim"] // case["heads"])
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for _ in range(2):
        x = torch.randn(n_attn * case["cached"], kvd, generator=g, device="cuda") * 0.9
        if case["kv"] == "q8_0":
            b = x.view(x.shape[0], kvd // 32, 32)
            d = b.abs().amax(2, keepdim=True) / 127.0
            q = torch.round(b / d).to(torch.int8)
            raw = torch.cat([d.to(torch.float16).view(torch.uint8), q.view(torch.uint8)], dim=2)
        else:
            raw = x.to(torch.float16 if case["kv"] == "f16" else torch.float32).view(torch.uint8)
        out.append(raw.reshape(-1).cpu().numpy())
    conv = np.random.default_rng(seed).normal(0.0, 0.5, case["layers"] * case["dim"] * 3).astype(np.float32)
    return out[0], out[1], conv


def prepare(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        n, d, t = case["rows"], case["cols"], TYPES[case["type"]]
        w = _device(_weights(case["type"], seed, n, d))
        if case["packed"]:
            p = torch.empty_like(w)
            mivi_hip.pack_weights(t, w, p, n, d)
            w = p
        return dict(case=case, w=w, x=_activations(seed + 1, d), out=torch.empty(n, device="cuda"))
    if kind == "dequant":
        w = _device(_weights(case["type"], seed, case["rows"], case["cols"]))
        return dict(case=case, w=w, out=torch.empty(case["rows"] * case["cols"], device="cuda"))
    if kind == "rows":
        b, n, d, t = case["batch"], case["rows"], case["cols"], TYPES[case["type"]]
        w = _device(_weights(case["type"], seed, n, d))
        wg = None
        if case["packed"]:
            wg = torch.empty(mivi_hip.gemm_packed_size(t, n, d), dtype=torch.uint8, device="cuda")
            mivi_hip.pack_weights_gemm(t, w, wg, n, d)
        return dict(case=case, w=w, wg=wg, x=_activations(seed + 1, b, d), out=torch.empty(b, n, device="cuda"))
    if kind == "sample":
        rows, n = case["rows"], case["n"]
        rec = torch.randint(0, n, (rows, case["recent"]), generator=torch.Generator().manual_seed(seed + 2),
                            dtype=torch.int32).cuda()
        rng = torch.tensor([seed * 1000 + 17 * r + 1 for r in range(rows)], dtype=torch.int64, device="cuda")
        return dict(case=case, logits=_logits(seed, rows, n), recent=rec, rng=rng,
                    cfg=mivi_hip.SamplerConfig.make(**SAMPLERS[case["sampler"]]),
                    probs=torch.empty(rows, n, device="cuda"), rng_out=torch.empty_like(rng),
                    tokens=torch.empty(rows, dtype=torch.int32, device="cuda"))
    img, attn = _image(case, seed)
    if kind == "prefill":
        m = mivi_hip.Model(img, max_ctx=case["max_ctx"], kv_precision=KV[case["kv"]], max_batch=1)
        m.set_prefill_strategy(case["tile"])
        return dict(case=case, model=m, tokens=_prompt(seed, case["tokens"] + 1, case["vocab"]))
    # decode: the prompt's state is held by a prefix cache, one snapshot for
    # every sequence
    m = mivi_hip.Model(img, max_ctx=case["max_ctx"], kv_precision=KV[case["kv"]], max_batch=case["batch"])
    prefix = _prompt(seed, case["cached"], case["vocab"])
    k, v, conv = _kv_rows(case, len(attn), seed)
    m.import_state(case["cached"], k, v, conv)
    pc = mivi_hip.PrefixCache(chunk_size=case["cached"], max_memory_bytes=4 << 30)
    pc.insert_chunk(m, 0, prefix, 0, case["cached"])
    return dict(case=case, model=m, cache=pc, prefix=prefix,
                tokens=_prompt(seed + 3, case["steps"] * case["batch"], case["vocab"]).reshape(case["steps"], -1))


# -------------------------------------------------------------------- runs

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matvec":
        f = mivi_hip.quantized_matvec_packed if case["packed"] else mivi_hip.quantized_matvec
        f(state["out"], TYPES[case["type"]], state["w"], state["x"], case["rows"], case["cols"])
        return state["out"]
    if kind == "dequant":
        mivi_hip.dequantize_slice(TYPES[case["type"]], state["w"], state["out"])
        return state["out"]
    if kind == "rows":
        t, b, n, d = TYPES[case["type"]], case["batch"], case["rows"], case["cols"]
        if case["packed"]:
            mivi_hip.quantized_matmul_rows_gemm_packed(state["out"], t, state["w"], state["wg"], state["x"], b, n, d)
        else:
            mivi_hip.quantized_matmul_rows(state["out"], t, state["w"], state["x"], b, n, d)
        return state["out"]
    if kind == "sample":
        # the sampler works in place on the logits a head has just written
        state["probs"].copy_(state["logits"])
        state["rng_out"].copy_(state["rng"])
        mivi_hip.sample_rows(state["probs"], state["recent"], state["cfg"], state["rng_out"], state["tokens"])
        return dict(probs=state["probs"], tokens=state["tokens"], rng=state["rng_out"])
    m, tok = state["model"], state["tokens"]
    if kind == "prefill":
        m.reset_context()
        m.prefill(tok[:-1])
        return m.forward(int(tok[-1]), len(tok) - 1)
    pos, batch = case["cached"], case["batch"]
    for b in range(batch):
        state["cache"].restore_longest_prefix(m, state["prefix"], seq=b)
    logits = []
    for s in range(case["steps"]):
        if batch == 1:
            logits.append(m.forward(int(tok[s, 0]), pos + s))
        else:
            logits.append(m.forward_batch(tok[s], [pos + s] * batch))
    return logits


# ------------------------------------------------------- work and precision

def _row_bytes(t, cols):
    return {"q4_k": cols // 256 * 144, "q6_k": cols // 256 * 210, "q8_0": cols // 32 * 34, "f16": 2 * cols,
            "bf16": 2 * cols, "f32": 4 * cols}[t]


def _model_work(case):
    """(weight bytes, weights) of the layers' projections, of the head, and the
    attention layer count."""
    layers = case["layers"]
    attn = FULL_ATTN if layers == 16 else tuple(i for i in range(layers) if i % 3 == 1)
    D, H, KVD = case["dim"], case["hidden"], case["kv_heads"] * (case["dim"] // case["heads"])
    base = "q8_0" if case["weights"] == "q8_0" else "q4_k"
    q6 = q6k_matrices(layers, attn, "q4_k_m") if case["weights"] == "q4_k_m" else set()
    nbytes = n = 0
    for i in range(layers):
        p = "blk.%d." % i
        if i in attn:
            mats = [("attn_q", D, D), ("attn_k", KVD, D), ("attn_v", KVD, D), ("attn_output", D, D)]
        else:
            mats = [("shortconv.in_proj", 3 * D, D), ("shortconv.out_proj", D, D)]
        for name, r, c in mats + [("ffn_gate", H, D), ("ffn_up", H, D), ("ffn_down", D, H)]:
            nbytes += r * _row_bytes("q6_k" if p + name + ".weight" in q6 else base, c)
            n += r * c
    return nbytes, n, case["vocab"] * _row_bytes("q6_k", D), case["vocab"] * D, len(attn), KVD


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        n, d = case["rows"], case["cols"]
        return {"bytes": n * _row_bytes(case["type"], d) + 4 * d + 4 * n, "flops": 2 * n * d}
    if kind == "dequant":
        n = case["rows"] * case["cols"]
        return {"bytes": case["rows"] * _row_bytes(case["type"], case["cols"]) + 4 * n, "flops": n}
    if kind == "rows":
        b, n, d = case["batch"], case["rows"], case["cols"]
        return {"bytes": n * _row_bytes(case["type"], d) + 4 * b * (n + d), "flops": 2 * b * n * d}
    if kind == "sample":
        n = case["rows"] * case["n"]
        return {"bytes": 16 * n, "flops": 4 * n}  # the logits' copy, then read and written once
    wb, wn, hb, hn, n_attn, kvd = _model_work(case)
    row = {"f32": 4 * kvd, "f16": 2 * kvd, "q8_0": kvd // 32 * 34}[case["kv"]] * 2 * n_attn
    if kind == "prefill":
        t = case["tokens"]
        return {"bytes": 2 * wb + hb + 2 * t * row + 4 * case["vocab"],
                "flops": 2 * wn * (t + 1) + 2 * hn + 2 * n_attn * case["dim"] * t * t}
    b, s, c = case["batch"], case["steps"], case["cached"]
    return {"bytes": 2 * b * c * row + s * (wb + hb + b * c * row + 4 * b * case["vocab"]),
            "flops": s * b * (2 * (wn + hn) + 4 * n_attn * case["dim"] * c)}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind in ("matvec", "rows"):
        # f32 sums; the activations enter as integer digits or fp16 pairs of
        # about 22 bits
        return {"rel": 2.5e-6, "max": 1.5e-5}
    if kind == "sample":
        return {"rel": 2e-6, "max": 1e-5}
    # rounding differences of every layer (f32 activations) carried to the
    # logits; cached values round to 11 bits (fp16) or to steps of 1/127 of
    # their block's largest (Q8_0), and a value on the edge of a step may fall
    # to either side
    rel = {"f32": 6e-5, "f16": 1e-4, "q8_0": 4e-4}[case["kv"]]
    return {"rel": rel, "max": 5 * rel}


# ------------------------------------------------------------ 64-bit results

def _decode64(t, raw, rows, cols):
    """The stored weights as 64-bit values [rows, cols] on the GPU."""
    raw = _device(raw).reshape(rows, -1)
    if t in ("f16", "bf16", "f32"):
        return raw.reshape(-1).view({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[t]).reshape(
            rows, cols).double()
    if t == "q8_0":
        b = raw.reshape(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).double()
        return (d * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if t == "q6_k":
        b = raw.reshape(-1, 210)
        ql, qh = b[:, :128].reshape(-1, 2, 64).int(), b[:, 128:192].reshape(-1, 2, 32).int()
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(-1, 2, 4, 2, 1)
        d = b[:, 208:].contiguous().view(torch.float16).double().reshape(-1, 1, 1, 1, 1)
        lo, hi = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([(lo & 15) | ((qh & 3) << 4), (hi & 15) | ((qh >> 2 & 3) << 4),
                         (lo >> 4) | ((qh >> 4 & 3) << 4), (hi >> 4) | ((qh >> 6 & 3) << 4)], dim=2) - 32
        return (d * sc * q.double().reshape(-1, 2, 4, 2, 16)).reshape(rows, cols)
    b = raw.reshape(-1, 144)
    dm = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].int()
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | (lo >> 6 << 4)], dim=1).double()
    mn = torch.cat([mid & 63, (hi >> 4) | (mid >> 6 << 4)], dim=1).double()
    qs = b[:, 16:].reshape(-1, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], dim=2).double().reshape(-1, 8, 32)
    return ((dm[:, :1] * sc)[:, :, None] * q - (dm[:, 1:] * mn)[:, :, None]).reshape(rows, cols)


def _exact_sample(case, seed):
    cfg = dict(temperature=0.2, top_p=0.9, top_k=40, min_p=0.0, repetition_penalty=1.05)
    cfg.update(SAMPLERS[case["sampler"]])
    st = prepare(case, seed)
    x, rec = st["logits"].double(), st["recent"].long()
    if rec.shape[1] and cfg["repetition_penalty"] != 1.0:
        seen = torch.zeros_like(x, dtype=torch.bool).scatter_(1, rec, True)
        rep = float(np.float32(cfg["repetition_penalty"]))
        x = torch.where(seen, torch.where(x > 0, x / rep, x * rep), x)
    if cfg["temperature"] > 0:
        x = x / float(np.float32(cfg["temperature"]))
        if 0 < cfg["top_k"] < x.shape[1]:
            cut = x.topk(cfg["top_k"], dim=1).values[:, -1:]
            x = torch.where(x < cut, -math.inf, x)
        x = torch.softmax(x, dim=1)
    return dict(probs=x, tokens=None, rng=None)


class _Exact:
    """The hybrid model in 64 bits over one image."""

    def __init__(self, case, seed):
        self.case = case
        self.img, self.attn = _image(case, seed)
        self.index = read_tensor_index(self.img)
        self.hd = case["dim"] // case["heads"]
        half = self.hd // 2
        # RoPE frequencies and angles in the 32 bits the tables are defined in
        base = np.float32(1.0) / np.power(np.float32(1e6), np.arange(half, dtype=np.float32) * np.float32(2) / np.float32(self.hd))
        if case["max_ctx"] > 4096:  # YaRN
            wl = np.float32(2.0 * math.pi) / base
            ramp = np.clip((wl - np.float32(128)) / np.float32(4096 - 128), 0, 1).astype(np.float32)
            base = (np.float32(1) - ramp) * base + ramp * (base / np.float32(case["max_ctx"] / 4096.0))
        ang = np.arange(case["max_ctx"], dtype=np.float32)[:, None] * base.astype(np.float32)
        self.cos = torch.from_numpy(np.cos(ang.astype(np.float64))).cuda()
        self.sin = torch.from_numpy(np.sin(ang.astype(np.float64))).cuda()

    def mat(self, name):
        t, dims, off, n = self.index[name]
        kind = {12: "q4_k", 14: "q6_k", 8: "q8_0", 0: "f32"}[t]
        rows = int(np.prod(dims[1:])) if len(dims) > 1 else 1
        return _decode64(kind, self.img[off:off + n].copy(), rows, dims[0])

    def rope(self, x, pos):
        c, s = self.cos[pos][:, None], self.sin[pos][:, None]
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], dim=-1).reshape(x.shape)

    def stored(self, x):
        """x as the cache holds it."""
        kv = self.case["kv"]
        if kv != "q8_0":
            return x.to(torch.float16 if kv == "f16" else torch.float32).double()
        b = x.reshape(-1, 32)
        d = b.abs().amax(1, keepdim=True) / 127.0
        q = torch.where(d > 0, torch.round(b / d), torch.zeros_like(b))
        return (q * d.to(torch.float16).double()).reshape(x.shape)

    def forward(self, tokens, pos0, kv, conv):
        """Tokens at pos0.. after the cached rows kv ((K, V) per attention layer)
        and the ShortConv state; the residual rows after the last layer."""
        case = self.case
        T, D, nh, nkv, hd = len(tokens), case["dim"], case["heads"], case["kv_heads"], self.hd
        emb = self.mat("token_embd.weight")
        x = emb[torch.from_numpy(tokens.astype(np.int64)).cuda()].clone()
        del emb
        pos = torch.arange(pos0, pos0 + T, device="cuda")

        def norm(v):
            return v / torch.sqrt(v.square().mean(1, keepdim=True) + 1e-5)

        a = 0
        for i in range(case["layers"]):
            p = "blk.%d." % i
            h = norm(x)
            if i in self.attn:
                q = self.rope((h @ self.mat(p + "attn_q.weight").T).view(T, nh, hd), pos)
                k = self.rope((h @ self.mat(p + "attn_k.weight").T).view(T, nkv, hd), pos)
                k, v = self.stored(k), self.stored((h @ self.mat(p + "attn_v.weight").T).view(T, nkv, hd))
                K, V = torch.cat([kv[a][0], k]), torch.cat([kv[a][1], v])
                out = torch.empty(T, nh, hd, dtype=torch.float64, device="cuda")
                later = torch.arange(K.shape[0], device="cuda")[None] > pos[:, None]
                for n in range(nh):
                    g = n // (nh // nkv)
                    sc = (q[:, n] @ K[:, g].T.contiguous()) / math.sqrt(hd)
                    out[:, n] = torch.softmax(sc.masked_fill_(later, -math.inf), dim=1) @ V[:, g]
                x = x + out.reshape(T, D) @ self.mat(p + "attn_output.weight").T
                a += 1
            else:
                B, C, X = (h @ self.mat(p + "shortconv.in_proj.weight").T).split(D, dim=1)
                s = torch.cat([conv[i][:, 1:].T, B * X])  # the two rows before the tokens
                w = self.mat(p + "shortconv.conv.weight")
                y = C * (s[:-2] * w[:, 0] + s[1:-1] * w[:, 1] + s[2:] * w[:, 2])
                x = x + y @ self.mat(p + "shortconv.out_proj.weight").T
            h = norm(x)
            g = h @ self.mat(p + "ffn_gate.weight").T
            x = x + (g * torch.sigmoid(g) * (h @ self.mat(p + "ffn_up.weight").T)) @ self.mat(p + "ffn_down.weight").T
        return norm(x)

    def logits(self, x):
        return x @ self.mat("token_embd.weight").T


def _exact_model(case, seed):
    e = _Exact(case, seed)
    n_attn, nkv, hd = len(e.attn), case["kv_heads"], e.hd
    if case["kind"] == "prefill":
        none = [(torch.empty(0, nkv, hd, dtype=torch.float64, device="cuda"),) * 2] * n_attn
        conv = torch.zeros(case["layers"], case["dim"], 3, dtype=torch.float64, device="cuda")
        x = e.forward(_prompt(seed, case["tokens"] + 1, case["vocab"]), 0, none, conv)
        return e.logits(x[-1:])[0]
    k, v, conv = _kv_rows(case, n_attn, seed)
    kind = case["kv"]
    kv = [_decode64(kind, r, n_attn * case["cached"], nkv * hd).view(n_attn, case["cached"], nkv, hd) for r in (k, v)]
    conv = torch.from_numpy(conv).cuda().double().view(case["layers"], case["dim"], 3)
    tok = _prompt(seed + 3, case["steps"] * case["batch"], case["vocab"]).reshape(case["steps"], -1)
    rows = [e.logits(e.forward(tok[:, b], case["cached"], [(kv[0][a], kv[1][a]) for a in range(n_attn)], conv))
            for b in range(case["batch"])]
    if case["batch"] == 1:
        return [rows[0][s] for s in range(case["steps"])]
    return [torch.stack([r[s] for r in rows]) for s in range(case["steps"])]


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind in ("prefill", "decode"):
        return _exact_model(case, seed)
    w = _decode64(case["type"], _weights(case["type"], seed, case["rows"], case["cols"]), case["rows"], case["cols"])
    if kind == "dequant":
        return w.reshape(-1)
    if kind == "matvec":
        return w @ _activations(seed + 1, case["cols"]).double()
    return _activations(seed + 1, case["batch"], case["cols"]).double() @ w.T
