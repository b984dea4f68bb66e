"""What this framework is timed on: the work a program that serves or evaluates a quantized model
gives it, through the Python view of the C-ABI (edgeforge_amd.hip, edgeforge_amd.model).

Kinds of work (a case's "kind"):
  qkv       the attention block's input projections: RMSNorm + q/k/v products in one call
            (matvec_jobs_rmsnorm), mixed Q4_0 / Q8_0 as the TinyLlama policy stores them.
  mlp       the feed-forward block: RMSNorm + gate/up + SwiGLU, then the down projection
            (matvec_swiglu, matvec), for one sequence, a few, a batch, or a prompt's rows.
  decode    one decode step of the engine at a given position (forward), with its logits.
  prefill   a prompt through the engine (prefill), with the logits of its last position.
  score     teacher-forced scoring of a text window (score): NLL and logits of every position, as
            the quality harness does for each chunk.
  sample    the sampler over a batch's logits, with the history's repetition penalty.
  quantize  packing a float matrix into Q4_0 (with the scale search) or Q8_0 blocks.

Shapes are TinyLlama-1.1B's (D 2048, F 5632, 32 heads over 4 KV heads of 64, 32000 ids), the
repository's own workload, with sizes around them in the drawn cases.  Weights are N(0, 0.02)
rounded to Q4_0 / Q8_0 blocks, norms 1 + 0.1 N(0, 1), activations N(0, 1), logits N(0, 3) as in
bench.py.  Engines of the long cases have 4 layers instead of 22: every layer does the same work.
"""
import ctypes
import math

import numpy as np
import torch

from edgeforge_amd import _lib as L
from edgeforge_amd import hip as H
from edgeforge_amd.model import LAYER_MATS, TINYLLAMA_Q8, Config, DeviceModel, Engine

EPS = 1e-5


# ---- the cases ---------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call of a decode step: one token's q/k/v projections (latency and launch bound)
        {"name": "qkv_b1", "kind": "qkv", "D": 2048, "heads": 32, "kv": 4, "batch": 1},
        # one token's feed-forward block: interactive decode
        {"name": "mlp_b1", "kind": "mlp", "D": 2048, "F": 5632, "batch": 1},
        # a few concurrent users, an odd number of them
        {"name": "mlp_b7", "kind": "mlp", "D": 2048, "F": 5632, "batch": 7},
        # a serving batch
        {"name": "mlp_b64", "kind": "mlp", "D": 2048, "F": 5632, "batch": 64},
        # a prompt's rows, not a multiple of any tile
        {"name": "mlp_rows1500", "kind": "mlp", "D": 2048, "F": 5632, "batch": 1500},
        # interactive decode: the whole model, one sequence, a short context
        {"name": "decode_b1", "kind": "decode", "layers": 22, "batch": 1, "pos": 55, "V": 32000},
        # serving: a full batch well into its context
        {"name": "decode_b64_long", "kind": "decode", "layers": 4, "batch": 64, "pos": 900, "V": 32000},
        # a long prompt
        {"name": "prefill_1999", "kind": "prefill", "layers": 4, "batch": 1, "n": 1999, "V": 32000},
        # one chunk of a perplexity run
        {"name": "score_511", "kind": "score", "layers": 2, "n": 511, "V": 32000},
        # the chat loop's sampler settings (top-k 40, top-p 0.95)
        {"name": "sample_topk_b1", "kind": "sample", "V": 32000, "batch": 1, "temperature": 0.8, "top_k": 40,
         "top_p": 0.95, "penalty": 1.1, "hist": 64, "sigma": 3.0},
        # nucleus sampling of a serving batch
        {"name": "sample_topp_b64", "kind": "sample", "V": 32000, "batch": 64, "temperature": 0.8, "top_k": 0,
         "top_p": 0.95, "penalty": 1.1, "hist": 64, "sigma": 3.0},
        # packing one feed-forward matrix
        {"name": "quantize_q4", "kind": "quantize", "rows": 5632, "cols": 2048, "q8": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["qkv", "mlp", "mlp", "decode", "prefill", "score", "sample", "quantize"])
    if kind == "qkv":
        kv = rng.choice([1, 2, 4, 8, 32])
        return {"kind": kind, "D": 2048, "heads": 32, "kv": kv, "batch": _log_int(rng, 1, 1024)}
    if kind == "mlp":
        D = rng.choice([512, 1024, 2048, 2048, 4096])
        F = 32 * _log_int(rng, 24, 5632 * 2048 // D // 32)
        return {"kind": kind, "D": D, "F": min(F, 14336), "batch": _log_int(rng, 1, 1500)}
    if kind == "decode":
        return {"kind": kind, "layers": 2, "batch": _log_int(rng, 1, 64), "pos": _log_int(rng, 8, 900),
                "V": rng.choice([32000, 8009])}
    if kind == "prefill":
        batch = _log_int(rng, 1, 24)
        return {"kind": kind, "layers": 2, "batch": batch, "n": _log_int(rng, 8, 1999 // batch),
                "V": rng.choice([32000, 8009])}
    if kind == "score":
        return {"kind": kind, "layers": 2, "n": _log_int(rng, 40, 511), "V": rng.choice([32000, 8009])}
    if kind == "sample":
        top_k = rng.choice([0, 0, 20, 40, 300])
        return {"kind": kind, "V": _log_int(rng, 3000, 32768), "batch": _log_int(rng, 1, 64),
                "temperature": rng.choice([0.0, 0.7, 0.8, 1.0]), "top_k": top_k,
                "top_p": rng.choice([0.9, 0.95, 1.0]), "penalty": rng.choice([1.0, 1.1]), "hist": _log_int(rng, 1, 500),
                "sigma": rng.choice([1.0, 2.0, 3.0])}
    return {"kind": kind, "rows": _log_int(rng, 500, 5632), "cols": 32 * _log_int(rng, 16, 64),
            "q8": rng.random() < 0.4}


# ---- inputs ------------------------------------------------------------------------------------------
class Buffer:
    """Device memory of a torch tensor, as the hip module's calls take it."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = self.t.data_ptr()
        self.nbytes = self.t.numel() * self.t.element_size()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 17)
    return g


def _randn(g, *shape, mean=0.0, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale + mean


def _pack(g, rows, cols, q8):
    """N(0, 0.02) weights as rows of Q8_0 (scale, 32 codes) or Q4_0 (scale, 16 bytes of two codes) blocks."""
    w = _randn(g, rows, cols // 32, 32, scale=0.02)
    d = (w.abs().amax(-1, keepdim=True) / (127.0 if q8 else 7.0)).half()
    q = torch.round(w / d.float())
    db = d.view(torch.uint8)
    if q8:
        codes = q.clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        u = (q.clamp(-8, 7) + 8).to(torch.uint8)
        codes = u[..., :16] | (u[..., 16:] << 4)
    return torch.cat([db, codes], -1).reshape(rows, -1).contiguous()


def _unpack(b, cols, q8):
    """The packed rows' values in float64."""
    b = b.view(b.shape[0], cols // 32, 34 if q8 else 18)
    d = b[..., :2].contiguous().view(torch.float16).double()
    c = b[..., 2:].contiguous()
    if q8:
        q = c.view(torch.int8).double()
    else:
        q = torch.cat([c & 15, c >> 4], -1).double() - 8.0
    return (q * d).reshape(b.shape[0], cols)


def _weight(b, cols, q8):
    return H.Weight(L.Q8_0 if q8 else L.Q4_0, b.shape[0], cols, device=Buffer(b))


def _config(case):
    n = case["pos"] + 1 if case["kind"] == "decode" else case["n"]
    return Config(V=case["V"], L=case["layers"], max_pos=max(64, n))


def _model_tensors(case, seed):
    """Packed matrices, norms and the BF16 embedding of one synthetic model, and the prompt ids."""
    cfg, g = _config(case), _gen(seed)
    mats = {}
    for l in range(cfg.L):
        for m in LAYER_MATS:
            r, c = cfg.shape(m)
            q8 = (l, m) in TINYLLAMA_Q8
            mats[(l, m)] = (_pack(g, r, c, q8), c, q8)
    mats["lm_head"] = (_pack(g, cfg.V, cfg.D, True), cfg.D, True)
    norms = {(l, n): _randn(g, cfg.D, mean=1.0, scale=0.1) for l in range(cfg.L) for n in ("attn", "ffn")}
    norms["final"] = _randn(g, cfg.D, mean=1.0, scale=0.1)
    embed = _randn(g, cfg.V, cfg.D, scale=0.02).bfloat16()
    n = case["pos"] + 1 if case["kind"] == "decode" else case["n"]
    ids = torch.randint(0, cfg.V, (case.get("batch", 1), n), generator=g, device="cuda").cpu().numpy().astype(np.int32)
    return cfg, mats, norms, embed, ids


def _prepare_engine(case, seed):
    cfg, mats, norms, embed, ids = _model_tensors(case, seed)
    torch.cuda.synchronize()
    m = DeviceModel(cfg, seed)
    m.weights = {k: _weight(b, c, q8) for k, (b, c, q8) in mats.items()}
    m.weights["embed"] = H.Weight(L.BF16, cfg.V, cfg.D, device=Buffer(embed))
    m.norms = {k: Buffer(v) for k, v in norms.items()}
    e = Engine(m, cfg.max_pos, batch=case.get("batch", 1))
    s = {"case": case, "engine": e, "ids": ids}
    if case["kind"] == "score":
        s["logits"] = Buffer(torch.empty(case["n"] - 1, cfg.V, device="cuda"))
        return s
    s["logits"] = torch.empty(case["batch"], cfg.V, device="cuda")
    if case["kind"] == "decode":
        if case["pos"] > 0:
            e.prefill(ids[:, :-1], 0, compute_logits=False)
        s["tokens"] = np.ascontiguousarray(ids[:, -1])
    return s


def _block_inputs(case, seed):
    g, D, batch = _gen(seed), case["D"], case["batch"]
    x, nw = _randn(g, batch, D), _randn(g, D, mean=1.0, scale=0.1)
    if case["kind"] == "qkv":
        kvd = D // case["heads"] * case["kv"]
        mats = [(_pack(g, D, D, False), D, False), (_pack(g, kvd, D, False), D, False), (_pack(g, kvd, D, True), D, True)]
    else:
        F = case["F"]
        mats = [(_pack(g, F, D, False), D, False), (_pack(g, F, D, False), D, False), (_pack(g, D, F, False), F, False)]
    return x, nw, mats


def _sample_inputs(case, seed):
    g = _gen(seed)
    logits = _randn(g, case["batch"], case["V"], scale=case["sigma"])
    hist = torch.randint(0, case["V"], (case["batch"], case["hist"]), generator=g, device="cuda", dtype=torch.int32)
    return logits, hist


def prepare(case, seed):
    H.init()
    kind = case["kind"]
    if kind in ("decode", "prefill", "score"):
        return _prepare_engine(case, seed)
    s = {"case": case}
    if kind in ("qkv", "mlp"):
        x, nw, mats = _block_inputs(case, seed)
        s["x"], s["norm"] = Buffer(x), Buffer(nw)
        s["w"] = [_weight(*m) for m in mats]
        # q, k and v rows share one row stride (D), as the block calls take it
        rows = [case["D"]] * 3 if kind == "qkv" else [case["F"], case["D"]]
        s["y"] = [Buffer(torch.zeros(case["batch"], r, device="cuda")) for r in rows]
    elif kind == "sample":
        logits, hist = _sample_inputs(case, seed)
        s["logits"], s["hist"] = Buffer(logits), Buffer(hist)
        s["hist_len"] = Buffer(torch.full((case["batch"],), case["hist"], dtype=torch.int32, device="cuda"))
        s["rng"] = H.RngStates([seed * 1000 + i for i in range(case["batch"])])
        s["out"] = Buffer(torch.zeros(case["batch"], dtype=torch.int32, device="cuda"))
        nbytes = L.lib().ef_hip_sample_workspace_bytes(case["V"], case["batch"])
        s["ws"] = Buffer(torch.empty(nbytes, dtype=torch.uint8, device="cuda"))
        s["cfg"] = dict(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                        repetition_penalty=case["penalty"])
    else:
        s["w"] = Buffer(_randn(_gen(seed), case["rows"], case["cols"], scale=0.02))
        s["qtype"] = L.Q8_0 if case["q8"] else L.Q4_0
        s["out"] = Buffer(torch.zeros(case["rows"] * H.row_bytes(s["qtype"], case["cols"]), dtype=torch.uint8,
                                      device="cuda"))
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "qkv":
        D, kvd = case["D"], case["D"] // case["heads"] * case["kv"]
        H.matvec_jobs_rmsnorm([(w, s["x"], y) for w, y in zip(s["w"], s["y"])], s["norm"], EPS, batch=case["batch"],
                              ldx=D, ldy=D)
        return [s["y"][0].t, s["y"][1].t[:, :kvd], s["y"][2].t[:, :kvd]]
    if kind == "mlp":
        gate, up, down = s["w"]
        act, out = s["y"]
        H.matvec_swiglu(gate, up, s["x"], act, s["norm"], EPS, batch=case["batch"])
        H.matvec(down, act, out, batch=case["batch"])
        return out.t
    if kind == "decode" or kind == "prefill":
        e = s["engine"]
        if kind == "decode":
            e.forward(s["tokens"], case["pos"])
        else:
            e.prefill(s["ids"], 0)
        p = ctypes.c_void_p()
        L.call("ef_hip_engine_logits", e.h, ctypes.byref(p))
        t = s["logits"]
        L.call("ef_hip_memcpy_d2d", t.data_ptr(), p.value, t.numel() * 4, None)
        return t
    if kind == "score":
        nll = s["engine"].score(s["ids"], 0, s["logits"])
        return [nll, s["logits"].t]
    if kind == "sample":
        H.sample(s["logits"], case["V"], s["cfg"], s["out"], batch=case["batch"], hist=s["hist"],
                 hist_len=s["hist_len"], hist_ld=case["hist"], rng=s["rng"], ws=s["ws"])
        return s["out"].t
    L.call("ef_hip_quantize", s["qtype"], s["w"].ptr, case["rows"], case["cols"], 1, s["out"].ptr, None)
    return s["out"].t


# ---- what a pass cannot do without ---------------------------------------------------------------------
def _qbytes(rows, cols, q8):
    return rows * (cols // 32) * (34 if q8 else 18)


def work(case):
    kind = case["kind"]
    if kind == "qkv":
        D, B = case["D"], case["batch"]
        kvd = D // case["heads"] * case["kv"]
        wb = _qbytes(D + kvd, D, False) + _qbytes(kvd, D, True)
        return {"bytes": wb + 4 * (B * (2 * D + 2 * kvd) + D), "flops": 2 * B * D * (D + 2 * kvd)}
    if kind == "mlp":
        D, F, B = case["D"], case["F"], case["batch"]
        return {"bytes": 2 * _qbytes(F, D, False) + _qbytes(D, F, False) + 4 * (2 * B * D + D), "flops": 6 * B * D * F}
    if kind in ("decode", "prefill", "score"):
        cfg, B = _config(case), case.get("batch", 1)
        kvd, per = cfg.KV * cfg.hd, 0
        params = 2 * cfg.D * cfg.D + 2 * kvd * cfg.D + 3 * cfg.F * cfg.D
        for l in range(cfg.L):
            for m in LAYER_MATS:
                r, c = cfg.shape(m)
                per += _qbytes(r, c, (l, m) in TINYLLAMA_Q8)
        if kind == "decode":
            rows, logit_rows, scores, kv_read = B, B, B * (case["pos"] + 1), B * case["pos"]
        else:
            n = case["n"] - (1 if kind == "score" else 0)
            rows, logit_rows, scores, kv_read = B * n, (n if kind == "score" else B), B * n * (n + 1) // 2, 0
        flops = rows * cfg.L * 2 * params + cfg.L * scores * cfg.H * cfg.hd * 4 + 2 * logit_rows * cfg.D * cfg.V
        kv = 4 * cfg.L * 2 * kvd * (rows + kv_read)
        byts = per + _qbytes(cfg.V, cfg.D, True) + kv + 2 * rows * cfg.D + 4 * logit_rows * cfg.V
        return {"bytes": byts, "flops": flops}
    if kind == "sample":
        return {"bytes": 4 * case["batch"] * (case["V"] + case["hist"] + 1), "flops": 4 * case["batch"] * case["V"]}
    n = case["rows"] * case["cols"]
    # the scale search tries six scales and refines up to twice: about six operations per weight and try
    return {"bytes": 4 * n + _qbytes(case["rows"], case["cols"], case["q8"]), "flops": (4 if case["q8"] else 48) * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "quantize"):
        return "exact"  # token ids and packed bytes are defined to the bit
    if kind in ("qkv", "mlp"):
        return {"rel": 2e-6, "max": 2e-5}  # FP32 sums in another order (2e-7 to 4.4e-7 against 64 bits)
    return {"rel": 8e-6, "max": 8e-5}  # a whole model in FP32 (up to 2e-6 against 64 bits)


# ---- the same in 64 bits ---------------------------------------------------------------------------------
def _rms(x, w):
    return w.double() * (x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS))


def _rope_tables(cfg, n):
    """cos / sin of the model's float32 angles (position times float32 inverse frequency)."""
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    half = cfg.hd // 2
    inv = np.array([np.float32(1.0) / np.float32(powf(cfg.rope_theta, np.float32(2 * i) / np.float32(cfg.hd)))
                    for i in range(half)], np.float32)
    ang = torch.from_numpy(np.arange(n, dtype=np.float32)[:, None] * inv[None, :]).cuda().double()
    return ang.cos(), ang.sin()


def _rope(x, cos, sin):
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_hidden(cfg, mats, norms, embed, ids):
    """Final-norm output [n][D] of every sequence in float64."""
    n = ids.shape[1]
    cos, sin = _rope_tables(cfg, n)
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    xs = [embed[torch.from_numpy(row.astype(np.int64)).cuda()].double() for row in ids]
    group = cfg.H // cfg.KV
    for l in range(cfg.L):
        W = {m: _unpack(*mats[(l, m)]).t() for m in LAYER_MATS}
        for i, x in enumerate(xs):
            h = _rms(x, norms[(l, "attn")])
            q = _rope((h @ W["wq"]).view(n, cfg.H, cfg.hd), cos, sin)
            k = _rope((h @ W["wk"]).view(n, cfg.KV, cfg.hd), cos, sin)
            v = (h @ W["wv"]).view(n, cfg.KV, cfg.hd)
            ctx = torch.empty(n, cfg.H, cfg.hd, dtype=torch.float64, device="cuda")
            for hd in range(cfg.H):
                sc = (q[:, hd] @ k[:, hd // group].t()) / math.sqrt(cfg.hd)
                ctx[:, hd] = torch.softmax(sc.masked_fill_(mask, -math.inf), -1) @ v[:, hd // group]
            x = x + ctx.reshape(n, -1) @ W["wo"]
            h = _rms(x, norms[(l, "ffn")])
            xs[i] = x + (torch.nn.functional.silu(h @ W["w_gate"]) * (h @ W["w_up"])) @ W["w_down"]
    return [_rms(x, norms["final"]) for x in xs]


def exact(case, seed):
    kind = case["kind"]
    if kind == "qkv":
        x, nw, mats = _block_inputs(case, seed)
        h = _rms(x.double(), nw)
        return [h @ _unpack(*m).t() for m in mats]
    if kind == "mlp":
        x, nw, mats = _block_inputs(case, seed)
        h = _rms(x.double(), nw)
        gate, up, down = [_unpack(*m).t() for m in mats]
        return (torch.nn.functional.silu(h @ gate) * (h @ up)) @ down
    if kind in ("decode", "prefill", "score"):
        cfg, mats, norms, embed, ids = _model_tensors(case, seed)
        head = _unpack(*mats["lm_head"]).t()
        if kind == "score":
            logits = _exact_hidden(cfg, mats, norms, embed, ids[:, :-1])[0] @ head
            target = torch.from_numpy(ids[0, 1:].astype(np.int64)).cuda()
            nll = torch.logsumexp(logits, -1) - logits.gather(1, target[:, None])[:, 0]
            return [nll, logits]
        return torch.stack([h[-1] @ head for h in _exact_hidden(cfg, mats, norms, embed, ids)])
    return None
