"""Attention over scores with a large common part, as trained models have: the matrix-core prefill and
large-batch decode kernels (one pass with a running maximum) against a float64 softmax
(kern::attention_heads, src/kernels.cpp:153-174).

One-layer models whose q, k and v are exact in float32 whatever the order of the sums, so that the
attention is all that rounds: embedding rows of +-1 (RMSNorm with eps 0 leaves them), Q8_0 matrices of
small codes with a power of two as scale, RoPE with a base so large that the dims in use do not turn,
an identity o projection and an empty feed-forward block.  Even heads have flat scores around the
offset (their maximum comes early and stays), odd heads rise along the positions (a new maximum in
every chunk, so the wave that the heads share rescales all along)."""
import numpy as np
import pytest

import oracle as O
from edgeforge_amd.model import Config, DeviceModel, Engine
from tests import _data as D

pytestmark = pytest.mark.gpu

H, HD, DIM, F, VARIANTS = 8, 64, 512, 256, 2
CONST, RAMP = 16, 64  # embedding columns that are always 1, and that spell the position
# Relative 2-norm per head.  Terms: 2^-24 for the exponent's last rounding, for c2 (times the distance to the
# maximum, about 1 on average under the softmax's weights), 2^-23 for exp2, 2^-24 for each of up to 64
# additions of chunk sums (at random: 8 x 2^-24 / 2), 2^-23 for the o projection's operand split, 2^-23 for the
# residual and the final norm: together below 16 x 2^-24.
REL_ERR = 16 * 2.0 ** -24


def _q8(codes: np.ndarray, scale: float) -> np.ndarray:
    r, c = codes.shape
    out = np.empty((r, c // 32, 34), np.uint8)
    out[:, :, :2] = np.full(1, scale, np.float16).view(np.uint8)
    out[:, :, 2:] = codes.astype(np.int8).view(np.uint8).reshape(r, c // 32, 32)
    return out.reshape(r, -1)


def _model(hip, n, offset, seed):
    """(DeviceModel, embedding [n][VARIANTS][DIM], q / k / v matrices in float64)."""
    g = D.rng(seed)
    x = g.choice([-1.0, 1.0], size=(n, VARIANTS, DIM)).astype(np.float32)
    x[:, :, :CONST] = 1.0
    x[:, :, CONST:CONST + RAMP] = np.where((np.arange(n) * RAMP // n)[:, None, None] > np.arange(RAMP), 1.0, -1.0)
    used = [j for j in range(HD) if j % 32 >= 16 and j not in (30, 31)]  # dims that RoPE leaves
    free = DIM - CONST - RAMP
    wq, wk = np.zeros((DIM, DIM), np.int64), np.zeros((HD, DIM), np.int64)
    wk[used, -free:] = g.integers(-5, 6, size=(len(used), free))
    wk[31, :CONST] = 96               # k[31] = 24, the common part
    wk[30, CONST:CONST + RAMP] = 2    # k[30] = -2 .. 2 along the positions
    for h in range(H):
        wq[64 * h + np.array(used), -free:] = g.integers(-5, 6, size=(len(used), free))
        wq[64 * h + 31, :CONST] = round(offset * (1 + h / 8) / 0.75)  # q[31] k[31] / 8: 1 to 1.9 times the offset
        wq[64 * h + 30, :CONST] = 64 if h % 2 else 0                  # odd heads rise by 8 over the positions
    wv = g.integers(-8, 9, size=(HD, DIM))
    cfg = Config(D=DIM, F=F, H=H, KV=1, hd=HD, V=n * VARIANTS, L=1, max_pos=n, eps=0.0, rope_theta=1e38)
    m = DeviceModel(cfg, seed)
    mats = {"wq": (wq, 2.0 ** -6), "wk": (wk, 2.0 ** -6), "wv": (wv, 1.0), "wo": (np.eye(DIM), 1.0),
            "w_gate": (np.zeros((F, DIM)), 1.0), "w_up": (np.zeros((F, DIM)), 1.0), "w_down": (np.zeros((DIM, F)), 1.0)}
    m.weights = {(0, k): hip.Weight(O.Q8_0, *w.shape, host=_q8(w, d)) for k, (w, d) in mats.items()}
    m.weights["lm_head"] = hip.Weight(O.Q8_0, cfg.V, DIM, host=_q8(np.zeros((cfg.V, DIM)), 1.0))
    bf16 = (x.reshape(-1, DIM).view(np.uint32) >> 16).astype(np.uint16)
    m.weights["embed"] = hip.Weight(O.BF16, cfg.V, DIM, host=bf16.view(np.uint8))
    ones = hip.DeviceArray.from_host(np.ones(DIM, np.float32))
    m.norms = {(0, "attn"): ones, (0, "ffn"): ones, "final": ones}
    return m, x, [w * d for w, d in (mats["wq"], mats["wk"], mats["wv"])]


def _want(x, mats, ids, last):
    """Final-norm output (DIM) of position `last` in float64."""
    h = x.reshape(-1, DIM)[ids[:last + 1]].astype(np.float64)
    q, k, v = mats[0] @ h[last], h @ mats[1].T, h @ mats[2].T
    s = k @ q.reshape(H, HD).T / 8.0
    p = np.exp(s - s.max(0))
    out = h[last] + ((p / p.sum(0)).T @ v).reshape(-1)
    return out / np.sqrt((out * out).mean())


def _errors(got, want):
    d = (got.astype(np.float64) - want).reshape(H, HD)
    return np.linalg.norm(d, axis=1) / np.linalg.norm(want.reshape(H, HD), axis=1)


@pytest.mark.parametrize("offset", [0, 10, 40])
def test_prefill_attention_with_offset_scores(hip, monkeypatch, offset):
    monkeypatch.setenv("EF_HIP_PREFILL_ATTENTION", "tiled")
    n = 1999
    print(f"[case] prefill attention, scores around {offset}", flush=True)
    m, x, mats = _model(hip, n, offset, seed=offset + 1)
    ids = (np.arange(n) * VARIANTS + D.rng(5).integers(0, VARIANTS, n)).astype(np.int32)
    eng = Engine(m, max_seq=n)
    eng.prefill([ids], 0)
    err = _errors(eng.hidden()[0], _want(x, mats, ids, n - 1))
    eng.close()
    print(f"offset {offset}: relative error per head {err}", flush=True)
    assert err.max() < REL_ERR, err


@pytest.mark.parametrize("offset", [0, 10, 40])
def test_large_batch_attention_with_offset_scores(hip, monkeypatch, offset):
    monkeypatch.delenv("EF_HIP_ATTENTION", raising=False)
    n, B = 1999, 128
    print(f"[case] large-batch attention, scores around {offset}", flush=True)
    m, x, mats = _model(hip, n, offset, seed=offset + 2)
    ids = (np.arange(n) * VARIANTS + D.rng(6).integers(0, VARIANTS, (B, n))).astype(np.int32)
    eng = Engine(m, max_seq=n, batch=B)
    eng.prefill(ids[:, :-1], 0, compute_logits=False)
    eng.forward(ids[:, -1], n - 1)
    got = eng.hidden()
    eng.close()
    err = np.array([_errors(got[b], _want(x, mats, ids[b], n - 1)) for b in (0, 63, 127)])
    print(f"offset {offset}: relative error per head {err}", flush=True)
    assert err.max() < REL_ERR, err
