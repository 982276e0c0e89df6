"""The work this framework is used for, as cases that can be timed and checked.

Decoder (the decision path): whole requests through `Engine.evaluate` (a cold
state with its question branches, and one branch on a resident state), blocks
of a few layers at the larger models' widths (long prefill, per-layer-input
layers with 512-wide heads, many branches on a resident state), the gated MLP
and the label readout through `DeviceWeight`.  Encoder: whole requests through
`LayaEngine.evaluate`, the q/k/v projection with its attention, and the gated
MLP through `DeviceWeight` / `attention_bi`.

Sizes are those of the benchmark configurations (`BASELINE_CONFIGS`,
`GEMMA4_CONFIGS`, `laya.C4`) and of the ranges around them.  `exact` restates
each path in plain torch float64 on the dequantized weights.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import grande_amd as g
from grande_amd import laya as ly
from grande_amd.engine import attention_bi

DEV = "cuda"
DTYPES = {"q4": g.Q4, "q8": g.Q8, "f16": g.F16}
WEIGHT_SEED = 0x5EED


def _model(base: dict, **over) -> dict:
    m = dict(base)
    m.update(over)
    return m


# What each decoder engine is built for: model shape, storage type, token
# capacity, most answer rows, and the readout a request asks for.
DECODERS = {
    # the 270M model whole: label logits + log-sum-exp per question
    "270m": dict(model=g.BASELINE_CONFIGS["c2"]["model"], dtype="q4", capacity=2448, max_rows=64, want="labels"),
    # six layers at the 1B width, Q8_0 weights (five sliding, one global)
    "1b": dict(model=_model(g.BASELINE_CONFIGS["c3"]["model"], layers=6), dtype="q8", capacity=2448, max_rows=64,
               want="hidden"),
    # three layers at the 4B width (sliding, global, sliding)
    "4b": dict(model=_model(g.BASELINE_CONFIGS["c5"]["model"], layers=3, sliding=[True, False, True]), dtype="q4",
               capacity=16384, max_rows=256, want="hidden"),
    # five layers at the E2B width: 512-wide global heads, per-layer inputs,
    # the last two sharing an earlier layer's K/V (more layers amplify the
    # f16 rounding through these models' sharp softmax: 4e-2 after seven)
    "e2b": dict(model=_model(g.GEMMA4_CONFIGS["e2b"]["model"], layers=5, shared_kv_layers=2,
                             sliding=[True, False, True, True, False]),
                dtype="q4", capacity=2752, max_rows=64, want="hidden", gemma4=True),
}
ENC_CAPACITY, ENC_ROWS = 192 * 256, 1024
ENC_MAX_LEN = 512
LABELS = g.LABEL_IDS


# ------------------------------------------------------------------ cases

def listed() -> list[dict]:
    return [
        # a new 2,000-token state with 12 questions of 32 tokens: the headline request
        dict(name="decide_cold_270m", kind="request", model="270m", resident=False, state=2000, branches=12, tokens=32),
        # one more question on the state that is already resident: the smallest call, latency alone
        dict(name="branch_warm_270m", kind="request", model="270m", resident=True, state=2000, branches=1, tokens=32),
        # a full batch of questions on a resident state, Q8_0 weights
        dict(name="branches_warm_1b_q8", kind="request", model="1b", resident=True, state=2000, branches=12, tokens=32),
        # the longest request: an 8,000-token state with 208 questions
        dict(name="prefill_4b_16k", kind="request", model="4b", resident=False, state=8000, branches=208, tokens=40),
        # the per-layer-input family, a 2,663-token request of ragged questions
        dict(name="prefill_e2b", kind="request", model="e2b", resident=False, state=2000, branches=12, tokens=55),
        # one gated MLP on f16 weights (an unquantized export), a state's worth of rows
        dict(name="mlp_f16_1b", kind="mlp", dtype="f16", rows=2384, d=1152, ff=6912),
        # the readout of one request's answer rows
        dict(name="readout_12_rows", kind="readout", dtype="q4", rows=12, d=640, vocab=25_000),
        # the readout of a large batch at the 4B width
        dict(name="readout_208_rows_4b", kind="readout", dtype="q4", rows=208, d=2560, vocab=25_000),
        # one request of the encoder path: three questions with three options each
        dict(name="encoder_request", kind="encoder", seqs=3, length=181, options=3),
        # the encoder's batch: 64 requests of three 256-token questions
        dict(name="encoder_batch_192", kind="encoder", seqs=192, length=256, options=1),
        # one local attention layer of the encoder on a middling ragged batch
        dict(name="encoder_attention", kind="enc_attention", seqs=48, length=509, window=64, dtype="q8"),
        # one encoder MLP on the full batch
        dict(name="encoder_mlp_batch", kind="enc_mlp", dtype="q8", rows=49_152, d=768, ff=1152),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["270m", "270m", "1b", "4b", "e2b", "mlp", "readout", "readout", "encoder", "encoder",
                       "enc_attention", "enc_mlp"])
    if kind in DECODERS:
        cap = {"270m": 2384, "1b": 2384, "4b": 16320, "e2b": 2663}[kind]
        most = {"270m": 24, "1b": 24, "4b": 208, "e2b": 24}[kind]
        tokens, branches = rng.randint(9, 56), _log_int(rng, 1, most)
        branches = max(1, min(branches, (cap - 64) // tokens))
        state = _log_int(rng, 60, min(8000, cap - branches * tokens))
        return dict(kind="request", model=kind, resident=bool(rng.random() < 0.5), state=state, branches=branches,
                    tokens=tokens)
    if kind == "mlp":
        d, ff = rng.choice([(640, 2048), (1152, 6912)])
        return dict(kind="mlp", dtype=rng.choice(["f16", "q8", "q4"]), rows=_log_int(rng, 24, 2384), d=d, ff=ff)
    if kind == "readout":
        return dict(kind="readout", dtype=rng.choice(["q4", "q4", "q8", "f16"]), rows=_log_int(rng, 1, 208),
                    d=rng.choice([640, 1152, 1536, 2560]), vocab=rng.randint(20_000, 25_000))
    if kind == "encoder":
        length = rng.randint(40, 256)
        return dict(kind="encoder", seqs=_log_int(rng, 3, min(192, ENC_CAPACITY // length)), length=length,
                    options=rng.randint(1, 4))
    if kind == "enc_attention":
        length = rng.randint(48, 512)
        return dict(kind="enc_attention", seqs=_log_int(rng, 3, ENC_CAPACITY // 2 // length), length=length,
                    window=rng.choice([0, 64, 64]), dtype=rng.choice(["q8", "q8", "q4"]))
    return dict(kind="enc_mlp", dtype=rng.choice(["q8", "q8", "q4", "f16"]), rows=_log_int(rng, 500, 49_152), d=768,
                ff=1152)


# ------------------------------------------------- weights a program keeps

_kept: dict = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _decoder_weights(name: str) -> g.Weights:
    def make():
        spec = DECODERS[name]
        cfg = (g.gemma4_config_json if spec.get("gemma4") else g.config_json)(**spec["model"])
        return g.Weights.synth(cfg, WEIGHT_SEED, DTYPES[spec["dtype"]], DTYPES[spec["dtype"]])
    return _keep(("decoder weights", name), make)


def _new_decoder(name: str) -> g.Engine:
    spec = DECODERS[name]
    return g.Engine.new(_decoder_weights(name), spec["capacity"], spec["max_rows"])


def _encoder_weights() -> g.Weights:
    def make():
        cfg = ly.laya_config_json(**ly.MMBERT_BASE, head_layers=2, act_costs={"ask": 1.0, "escalate": 2.0},
                                  max_len=ENC_MAX_LEN)
        return ly.synth_weights(cfg, WEIGHT_SEED, g.Q8, g.Q8)
    return _keep("encoder weights", make)


def _linear(dtype: str, rows: int, cols: int, which: int):
    """A linear weight (N(0, 1/cols), quantized as the checkpoints are) as
    the host tensor and its device copy."""
    def make():
        gen = torch.Generator().manual_seed(WEIGHT_SEED + 7919 * which + rows * 31 + cols)
        v = torch.randn(rows, cols, generator=gen).mul_(cols ** -0.5).numpy()
        if dtype == "f16":
            t = g.QTensor("w", g.F16, (rows, cols), v.astype(np.float16).view(np.uint8).ravel().copy(),
                          np.zeros(0, np.uint8))
        else:
            t = g.QTensor("w", DTYPES[dtype], (rows, cols), *g.quantize(DTYPES[dtype], v))
        return t, g.DeviceWeight(t)
    return _keep(("linear", dtype, rows, cols, which), make)


# ---------------------------------------------------------------- prepare

def _lengths(case) -> list[int]:
    """Ragged sequence lengths: the longest as given, the others from half
    of it up (a batch of exactly 256-token questions stays even)."""
    n, top = case["seqs"], case["length"]
    if top == 256:
        return [top] * n
    r = np.random.default_rng(top * 1009 + n)
    return [top] + r.integers(max(8, top // 2), top + 1, n - 1).tolist()


def _request(case, seed):
    rng = np.random.default_rng(seed)
    vocab = DECODERS[case["model"]]["model"]["vocab"]
    prefix = rng.integers(0, vocab, case["state"]).astype(np.uint32)
    branches = []
    for b in range(case["branches"]):
        n = case["tokens"] + (1 if case["model"] == "e2b" and b < 3 and case["branches"] >= 12 else 0)
        branches.append(g.BranchTokens(rng.integers(0, vocab, n).astype(np.uint32), [n - 1]))
    return prefix, branches


def _questions(case, seed) -> list[ly.Sequence]:
    rng = np.random.default_rng(seed)
    seqs = []
    for i, n in enumerate(_lengths(case)):
        ids = rng.integers(5, ly.MMBERT_BASE["vocab"], n)
        ids[0], ids[-1] = 1, 2
        marks = np.sort(rng.choice(np.arange(1, n - 1), size=case["options"], replace=False))
        ids[marks] = 4
        seqs.append(ly.Sequence(ids.astype(np.uint32), marks.astype(np.uint32), i % 3))
    return seqs


def _randn(seed, *shape):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    return torch.randn(*shape, generator=gen, device=DEV)


def _span_meta(case) -> np.ndarray:
    rows, at = [], 0
    for s, n in enumerate(_lengths(case)):
        rows += [(i, s, at, at + n) for i in range(n)]
        at += n
    return np.array(rows, np.int32)


def _rope_table(theta: float, rows: int) -> torch.Tensor:
    f = theta ** (-torch.arange(0, 64, 2, dtype=torch.float64) / 64)
    ang = torch.arange(rows, dtype=torch.float64)[:, None] * f
    return torch.stack([ang.cos(), ang.sin()], -1)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "request":
        name = case["model"]
        prefix, branches = _request(case, seed)
        st.update(prefix=prefix, branches=branches)
        st["want"] = g.Want.LABELS_LSE if DECODERS[name]["want"] == "labels" else g.Want.HIDDEN
        st["labels"] = LABELS if DECODERS[name]["want"] == "labels" else None
        if case["resident"]:
            # the state decoded by an earlier request, in an engine of its own
            st["engine"] = _new_decoder(name)
            st["engine"].evaluate(prefix, [g.BranchTokens(prefix[:1], [0])], st["want"], st["labels"])
        else:
            st["engine"] = _keep(("engine", name), lambda: _new_decoder(name))
        return st
    if kind == "encoder":
        st["engine"] = _keep("encoder", lambda: ly.LayaEngine.new(_encoder_weights(), ENC_CAPACITY, ENC_ROWS))
        st["seqs"] = _questions(case, seed)
        return st
    if kind == "readout":
        st["embed"] = _linear(case["dtype"], case["vocab"], case["d"], 0)[1]
        st["rows"] = _randn(seed, case["rows"], case["d"])
        st["labels"] = torch.tensor(LABELS, dtype=torch.int32, device=DEV)
        st["out"] = torch.empty(case["rows"], len(LABELS) + 1, device=DEV)
        return st
    d = case["d"] if "d" in case else ly.MMBERT_BASE["d"]
    if kind in ("mlp", "enc_mlp"):
        st["x"] = _randn(seed, case["rows"], d).half()
        st["gate"] = _linear(case["dtype"], case["ff"], d, 1)[1]
        st["up"] = _linear(case["dtype"], case["ff"], d, 2)[1]
        st["down"] = _linear(case["dtype"], d, case["ff"], 3)[1]
        st["act"] = torch.empty(case["rows"], case["ff"], dtype=torch.float16, device=DEV)
        st["y"] = torch.empty(case["rows"], d, device=DEV)
        return st
    meta = _span_meta(case)
    t = len(meta)
    tpad = (t + 63) // 64 * 64
    st["x"] = _randn(seed, t, d).half()
    st["w"] = _linear(case["dtype"], 3 * d, d, 4)[1]
    st["meta"] = torch.from_numpy(meta).to(DEV)
    st["rope"] = _rope_table(10000.0, ENC_MAX_LEN).float().to(DEV)
    st["heads"] = [torch.zeros(d // 64 * tpad * 64, dtype=torch.float16, device=DEV) for _ in range(3)]
    st["t"], st["tpad"], st["d"] = t, tpad, d
    st["out"] = torch.empty(t, d, dtype=torch.float16, device=DEV)
    return st


# -------------------------------------------------------------------- run

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "request":
        if not case["resident"]:
            st["engine"].evict_resident()  # another state was served in between
        out = st["engine"].evaluate(st["prefix"], st["branches"], st["want"], st["labels"])
        return np.stack([r for b in out for r in b.rows])
    if kind == "encoder":
        out = st["engine"].evaluate(st["seqs"])
        return {"logits": np.concatenate([o.logits for o in out]), "act": np.array([o.act_probability for o in out])}
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "readout":
        st["embed"].label_readout(st["rows"].data_ptr(), case["rows"], st["labels"].data_ptr(), len(LABELS), 0.0,
                                  st["out"].data_ptr(), stream)
        return st["out"]
    if kind in ("mlp", "enc_mlp"):
        m, d, ff = case["rows"], case["d"], case["ff"]
        gated = st["gate"].gemm_geglu_erf if kind == "enc_mlp" else st["gate"].gemm_geglu
        gated(st["up"], st["x"].data_ptr(), d, m, st["act"].data_ptr(), ff, stream)
        st["down"].gemm(st["act"].data_ptr(), ff, m, st["y"].data_ptr(), d, stream)
        return {"act": st["act"], "y": st["y"]}
    q, k, vt = (h.data_ptr() for h in st["heads"])
    st["w"].qkv_heads(st["x"].data_ptr(), st["d"], st["t"], None, st["rope"].data_ptr(), st["meta"].data_ptr(), 0.125,
                      st["tpad"], q, k, vt, stream)
    attention_bi(q, k, vt, st["meta"].data_ptr(), st["d"] // 64, st["t"], st["tpad"], case["window"],
                 st["out"].data_ptr(), stream)
    return st["out"]


# ------------------------------------------------------------------- work

_BYTES = {"q4": 18 / 32, "q8": 34 / 32, "f16": 2.0}  # per stored weight


def _pairs(case, window: int) -> int:
    """Query-key pairs the block-causal mask admits in one layer, for the
    tokens the request decodes."""
    P, n, bt = case["state"], case["branches"], case["tokens"]
    pre = sum(min(q + 1, window) if window else q + 1 for q in range(P)) if not case["resident"] else 0
    own = sum((min(P, max(0, window - j - 1)) + min(j + 1, window)) if window else P + j + 1 for j in range(bt))
    return pre + n * own


def work(case) -> dict:
    kind = case["kind"]
    if kind == "request":
        spec = DECODERS[case["model"]]
        m, b = spec["model"], _BYTES[spec["dtype"]]
        new = case["branches"] * case["tokens"] + (0 if case["resident"] else case["state"])
        wanted, L = case["branches"], m["layers"]
        own = L - m.get("shared_kv_layers", 0)
        types = m.get("sliding") or [(i + 1) % 6 != 0 for i in range(L)]
        flops = bytes_ = 0.0
        for i in range(L):
            hd = m["head_dim"] if types[i] else m.get("global_head_dim", m["head_dim"])
            window = m["window"] if types[i] else 0
            ff = m["ff"] * (2 if i >= own and m.get("double_wide_mlp") else 1)
            q, kv = m["heads"] * hd, 2 * m["kv_heads"] * hd * (i < own)
            # every row up to the last layer with K/V of its own; there the
            # keys and values alone, and from there on the answer rows
            rows = new if i + 1 < own else wanted
            flops += 2.0 * m["d"] * ((q + q + 3 * ff) * rows + kv * new)
            pairs = _pairs(case, window) if i + 1 < own else wanted * (case["state"] if not window else window)
            flops += 4.0 * m["heads"] * hd * pairs
            p = m.get("per_layer_dim", 0)
            flops += 2.0 * m["d"] * p * 3 * rows
            bytes_ += b * m["d"] * (q + kv + q + 3 * ff + 3 * p)
            keys = (min(window, case["state"]) if window else case["state"]) if case["resident"] else 0
            bytes_ += 2.0 * (keys * 2 * m["kv_heads"] * hd + new * kv)
        bytes_ += new * m["d"] * b
        if spec["want"] == "labels":
            flops += 2.0 * wanted * m["vocab"] * m["d"]
            bytes_ += b * m["vocab"] * m["d"] + 4.0 * wanted * (len(LABELS) + 1)
        else:
            bytes_ += 4.0 * wanted * m["d"]
        return {"bytes": bytes_, "flops": flops}
    if kind == "readout":
        n, d, v = case["rows"], case["d"], case["vocab"]
        return {"bytes": v * d * _BYTES[case["dtype"]] + 4.0 * n * (d + len(LABELS) + 1), "flops": 2.0 * n * d * v}
    if kind in ("mlp", "enc_mlp"):
        n, d, ff = case["rows"], case["d"], case["ff"]
        return {"bytes": 3 * d * ff * _BYTES[case["dtype"]] + n * (2.0 * d + 2 * ff + 4 * d), "flops": 6.0 * n * d * ff}
    m = ly.MMBERT_BASE
    d, ff = m["d"], m["ff"]
    lens = _lengths(case)
    t = sum(lens)

    def pairs(n, w):
        return n * n if not w else sum(min(n, i + w + 1) - max(0, i - w) for i in range(n))

    if kind == "enc_attention":
        return {"bytes": 3 * d * d * _BYTES[case["dtype"]] + t * (2.0 * d + 3 * 2 * d + 2 * d),
                "flops": 6.0 * t * d * d + 4.0 * d * sum(pairs(n, case["window"]) for n in lens)}
    window = m["local_attention"] // 2
    everything, local = sum(pairs(n, 0) for n in lens), sum(pairs(n, window) for n in lens)
    rows = len(lens) * (1 + case["options"])
    n_global = sum(1 for i in range(m["layers"]) if i % m["global_every"] == 0)
    lin = m["layers"] * (4 * d * d + 3 * d * ff)
    flops = 2.0 * t * lin + 4.0 * d * (n_global * everything + (m["layers"] - n_global) * local)
    # the decision head: one whole layer, then keys and values of every row
    # and the rest of the second layer on the rows that are scored
    flops += 2.0 * t * (12 * d * d + 2 * d * d) + 2.0 * rows * 10 * d * d + 4.0 * d * everything
    flops += 2.0 * rows * d * d
    bytes_ = _BYTES["q8"] * (lin + 24 * d * d) + 4.0 * d * d + t * d * _BYTES["q8"] + 4.0 * rows
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times the distance to float64 measured over the listed and
    a dozen drawn cases (f16 operands; the readout is f32 throughout)."""
    kind = case["kind"]
    if kind == "request":
        return {"rel": {"270m": 2.5e-4, "1b": 5e-4, "4b": 2.5e-4, "e2b": 1.5e-2}[case["model"]]}
    return {"rel": {"encoder": 2e-2, "readout": 2e-6, "enc_attention": 2.5e-3, "mlp": 1.7e-3, "enc_mlp": 1.7e-3}[kind]}


# ------------------------------------------------------------------ exact

def _dequant(t: g.QTensor) -> torch.Tensor:
    """A stored tensor's values in float64, on the GPU."""
    rows = t.shape[0]
    data = torch.from_numpy(t.data).to(DEV)
    if t.dtype == g.F16:
        return data.view(torch.float16).double().view(t.shape)
    scale = torch.from_numpy(t.scales).to(DEV).view(torch.float16).double()[:, None]
    if t.dtype == g.Q8:
        return (data.view(torch.int8).view(-1, 32).double() * scale).view(t.shape)
    data = data.view(-1, 16)
    q = torch.cat([data & 15, data >> 4], 1).double() - 8.0
    return (q * scale).view(rows, -1)


def _tensors(weights) -> dict:
    return _keep(("host", id(weights)), lambda: {t.name: t for t in weights.tensors()})


def _rms(x, w, eps=1e-6):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _gelu_tanh(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope(x, pos, theta, dims):
    """Pairs (i, i + hd/2) of [t, heads, hd] rotated for i < dims/2."""
    half = x.shape[-1] // 2
    i = torch.arange(half, device=x.device, dtype=torch.float64)
    ang = pos[:, None] * theta ** (-i / half)
    ang = torch.where(i < dims // 2, ang, torch.zeros_like(ang))[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _decoder_exact(case, seed):
    name = case["model"]
    spec = DECODERS[name]
    m = spec["model"]
    W = _tensors(_decoder_weights(name))

    def w(n):
        return _dequant(W[n]) if len(W[n].shape) > 1 else torch.from_numpy(W[n].to_f32()).double().to(DEV)

    prefix, branches = _request(case, seed)
    P = len(prefix)
    ids = np.concatenate([prefix] + [b.tokens for b in branches]).astype(np.int64)
    pos = np.concatenate([np.arange(P)] + [P + np.arange(len(b.tokens)) for b in branches])
    seq = np.concatenate([np.zeros(P, int)] + [np.full(len(b.tokens), i + 1) for i, b in enumerate(branches)])
    ends = P + np.cumsum([len(b.tokens) for b in branches]) - 1
    ids, seq = torch.from_numpy(ids).to(DEV), torch.from_numpy(seq).to(DEV)
    ipos = torch.from_numpy(pos).to(DEV)
    pos = ipos.double()
    d, L, H, KV = m["d"], m["layers"], m["heads"], m["kv_heads"]
    gemma4, p = bool(spec.get("gemma4")), m.get("per_layer_dim", 0)
    own = L - m.get("shared_kv_layers", 0)
    types = m.get("sliding") or [(i + 1) % 6 != 0 for i in range(L)]
    x = w("embed")[ids] * math.sqrt(d)
    if p:
        pl = (x @ w("pl_model_proj").T).view(-1, L, p) / math.sqrt(d)
        pl = (_rms(pl, w("pl_proj_norm")) + w("per_layer_table")[ids].view(-1, L, p) * math.sqrt(p)) / math.sqrt(2.0)
    cache: dict = {}
    for i in range(L):
        n = f"blk.{i}."
        hd = m["head_dim"] if types[i] else m.get("global_head_dim", m["head_dim"])
        theta = 1e4 if types[i] else 1e6
        dims = hd if types[i] or not gemma4 else int(hd * m["partial_rotary_global"])
        y = (_rms(x, w(n + "attn_norm")) @ w(n + "qkv").T).view(len(ids), -1, hd)
        q = _rope(_rms(y[:, :H], w(n + "q_norm")), pos, theta, dims) * (1.0 if gemma4 else hd ** -0.5)
        if i < own:
            k = _rope(_rms(y[:, H:H + KV], w(n + "k_norm")), pos, theta, dims)
            v = y[:, H + KV:]
            cache[types[i]] = (k, _rms(v, None) if gemma4 else v)
        k, v = cache[types[i]]
        att = torch.empty(len(ids), H, hd, dtype=torch.float64, device=DEV)
        for lo in range(0, len(ids), 2048):
            s = slice(lo, min(lo + 2048, len(ids)))
            back = ipos[s, None] - ipos[None]
            see = (back >= 0) & ((seq[None] == 0) | (seq[s, None] == seq[None]))
            if types[i]:
                see &= back < m["window"]
            for h in range(H):
                sc = (q[s, h] @ k[:, h * KV // H].T).masked_fill_(~see, -math.inf)
                att[s, h] = torch.softmax(sc, -1) @ v[:, h * KV // H]
        x = x + _rms(att.flatten(1) @ w(n + "o").T, w(n + "post_attn_norm"))
        h = _rms(x, w(n + "ffn_norm"))
        h = _gelu_tanh(h @ w(n + "gate").T) * (h @ w(n + "up").T)
        x = x + _rms(h @ w(n + "down").T, w(n + "post_ffn_norm"))
        if p:
            h = _gelu_tanh(x @ w(n + "pl_gate").T) * pl[:, i]
            x = (x + _rms(h @ w(n + "pl_proj").T, w(n + "pl_norm"))) * w(n + "out_scale")
    rows = _rms(x[torch.from_numpy(ends).to(DEV)], w("final_norm"))
    if spec["want"] == "labels":
        z = rows @ w("embed").T
        rows = torch.cat([z[:, LABELS], torch.logsumexp(z, -1, keepdim=True)], 1)
    return rows.cpu().numpy()


def _ln(x, w, b=None, eps=1e-5):
    y = torch.nn.functional.layer_norm(x, x.shape[-1:], w, b, eps)
    return y


def _gelu_erf(x):
    return torch.nn.functional.gelu(x)


def _rope_heads(x, table, pos):
    """[t, heads, 64] rotated: pairs (c, c + 32) by the table's (cos, sin)."""
    cs = table[pos]
    c, s = cs[:, None, :, 0], cs[:, None, :, 1]
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _spans_attention(q, k, v, lens, window):
    """softmax(q k^T) v within each sequence, |i - j| <= window when set."""
    out, at = [], 0
    for n in lens:
        s = slice(at, at + n)
        sc = torch.matmul(q[s].transpose(0, 1).contiguous(), k[s].permute(1, 2, 0).contiguous())
        if window:
            i = torch.arange(n, device=DEV)
            sc.masked_fill_((i[:, None] - i[None]).abs() > window, -math.inf)
        out.append(torch.matmul(torch.softmax(sc, -1), v[s].transpose(0, 1).contiguous()).transpose(0, 1).flatten(1))
        at += n
    return torch.cat(out)


def _encoder_exact(case, seed):
    m = ly.MMBERT_BASE
    W = _tensors(_encoder_weights())

    def w(n):
        return _dequant(W[n]) if len(W[n].shape) > 1 else torch.from_numpy(W[n].to_f32()).double().to(DEV)

    seqs = _questions(case, seed)
    lens = [len(s.ids) for s in seqs]
    ids = torch.from_numpy(np.concatenate([s.ids for s in seqs]).astype(np.int64)).to(DEV)
    pos = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(DEV)
    d, heads = m["d"], m["heads"]
    tables = {s: _rope_table(t, ENC_MAX_LEN).to(DEV) for s, t in ((True, 10000.0), (False, 160000.0))}
    x = _ln(w("embed")[ids], w("embed_norm"))
    for i in range(m["layers"]):
        n, sliding = f"enc.{i}.", i % m["global_every"] != 0
        h = _ln(x, w(n + "attn_norm")) if i else x
        q, k, v = (h @ w(n + "qkv").T).view(-1, 3, heads, 64).unbind(1)
        q, k = _rope_heads(q, tables[sliding], pos) * 0.125, _rope_heads(k, tables[sliding], pos)
        x = x + _spans_attention(q, k, v, lens, m["local_attention"] // 2 if sliding else 0) @ w(n + "o").T
        h = _ln(x, w(n + "mlp_norm"))
        x = x + (_gelu_erf(h @ w(n + "wi_val").T) * (h @ w(n + "wi_gate").T)) @ w(n + "wo").T
    kinds = torch.from_numpy(np.repeat([s.qtype for s in seqs], lens)).to(DEV)
    x = _ln(x, w("final_norm")) + w("type_emb")[kinds]
    for i in range(2):
        n = f"head.{i}."
        h = _ln(x, w(n + "norm1_w"), w(n + "norm1_b"))
        q, k, v = (h @ w(n + "in_proj").T + w(n + "in_proj_b")).view(-1, 3, heads, 64).unbind(1)
        x = x + _spans_attention(q, k, v, lens, 0) @ w(n + "out_proj").T + w(n + "out_proj_b")
        h = torch.relu(_ln(x, w(n + "norm2_w"), w(n + "norm2_b")) @ w(n + "l1").T + w(n + "l1_b"))
        x = x + h @ w(n + "l2").T + w(n + "l2_b")
    starts = np.cumsum([0] + lens[:-1])
    marks = np.concatenate([a + s.markers.astype(np.int64) for a, s in zip(starts, seqs)])
    z = _ln(x[torch.from_numpy(marks).to(DEV)], w("scorer.norm_w"), w("scorer.norm_b"))
    z = _gelu_erf(z @ w("scorer.l1").T + w("scorer.l1_b"))
    logits = (z @ w("scorer.l2").T + w("scorer.l2_b")).view(len(seqs), -1)
    # the act head: the [CLS] row and the confidence of the untempered softmax
    k = max(2, logits.shape[1])
    padded = torch.full((len(seqs), k), -1e4, dtype=torch.float64, device=DEV)
    padded[:, :logits.shape[1]] = logits
    p = torch.softmax(padded, -1)
    entropy = -(p * p.clamp_min(1e-9).log()).sum(-1) / math.log(k)
    top = p.sort(-1, descending=True).values
    feats = torch.stack([top[:, 0], top[:, 0] - top[:, 1], entropy, torch.full_like(entropy, k / 255.0)], 1)
    h = torch.cat([x[torch.from_numpy(starts).to(DEV)], feats], 1)
    h = _gelu_erf(h @ w("act.l1").T + w("act.l1_b"))
    act = torch.softmax(h @ w("act.l2").T + w("act.l2_b"), -1)[:, 0]
    return {"logits": logits.flatten().cpu().numpy(), "act": act.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "request":
        return _decoder_exact(case, seed)
    if kind == "encoder":
        return _encoder_exact(case, seed)
    if kind == "readout":
        z = _randn(seed, case["rows"], case["d"]).double() @ _dequant(_linear(case["dtype"], case["vocab"], case["d"],
                                                                              0)[0]).T
        return torch.cat([z[:, LABELS], torch.logsumexp(z, -1, keepdim=True)], 1)
    if kind in ("mlp", "enc_mlp"):
        d, ff = case["d"], case["ff"]
        wg, wu, wd = (_dequant(_linear(case["dtype"], *s)[0]) for s in ((ff, d, 1), (ff, d, 2), (d, ff, 3)))
        x = _randn(seed, case["rows"], d).half().double()
        act = (_gelu_erf if kind == "enc_mlp" else _gelu_tanh)(x @ wg.T) * (x @ wu.T)
        return {"act": act, "y": act @ wd.T}
    lens = _lengths(case)
    d = ly.MMBERT_BASE["d"]
    pos = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(DEV)
    table = _rope_table(10000.0, ENC_MAX_LEN).to(DEV)
    y = (_randn(seed, sum(lens), d).half().double() @ _dequant(_linear(case["dtype"], 3 * d, d, 4)[0]).T)
    q, k, v = y.view(-1, 3, d // 64, 64).unbind(1)
    q, k = _rope_heads(q, table, pos) * 0.125, _rope_heads(k, table, pos)
    return _spans_attention(q, k, v, lens, case["window"])
