"""GPU parity of the batched (2+ sequences) packed GEMV on the matrix cores (C-ABI calls).

Every sequence of a batch must meet the single-vector gates:
|gpu - exact| <= 1e-5 * sum|w x| per row (tests/test_qinfer.cpp:95) and max |gpu - cpu fp32| <= 1e-4
against the oracle's AVX2 kernel (src/qkernels.cpp:131-180) on that sequence alone.  Shapes cover
batches that are not a multiple of the 16-sequence tile, many tiles in one launch, more than 1024
sequences (several launches), row counts that leave a partial workgroup, Q8_0, a K split (K = 5632
at B = 64) and mixed-type launches; epilogues and the fused RMSNorm are checked against the oracle's separate operations.
"""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

import oracle as O
from edgeforge_amd import _lib as L
from tests import _data as D

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ABS_TOL = 1e-4
REL_TOL = 1e-5


def _batch_x(seed, batch, cols):
    return np.stack([D.activations_with_outliers(seed + b, cols) for b in range(batch)]).astype(np.float32)



@pytest.mark.parametrize("qtype,rows,cols,batch", [
    (O.Q4_0, 512, 2048, 5),      # one partial sequence tile
    (O.Q8_0, 300, 2048, 16),     # Q8_0, rows leave a partial workgroup
    (O.Q4_0, 2048, 5632, 64),    # K split across workgroups
    (O.Q4_0, 37, 256, 70),       # tiny K, a partial last tile
    (O.Q4_0, 96, 512, 300),      # 19 sequence tiles in one launch
    (O.Q8_0, 37, 256, 1100),     # two launches (1024 + 76 sequences)
    (O.Q8_0, 64, 512, 2),
    (O.Q4_0, 5632, 2048, 16),    # TinyLlama gate / up shape at B = 16
    (O.Q4_0, 2048, 5632, 16),    # down shape (K = 5632)
    (O.Q8_0, 256, 2048, 16),     # a Q8_0 k / v override
    (O.Q4_0, 2048, 2048, 16),    # q / o shape
    (O.Q4_0, 5632, 2048, 64),    # the same at B = 64
    (O.Q8_0, 256, 2048, 64),
])
def test_batched_gemv_each_sequence_meets_the_gates(hip, qtype, rows, cols, batch):
    print(f"[case] batched gemv qtype={qtype} {rows}x{cols} B={batch}", flush=True)
    packed = D.random_rows(qtype, rows, cols, seed=rows + cols + batch)
    X = _batch_x(1000 + batch, batch, cols)
    W = hip.Weight(qtype, rows, cols, host=packed)
    dx = hip.DeviceArray.from_host(X)
    dy = hip.DeviceArray((batch, rows))
    hip.matvec(W, dx, dy, batch=batch)
    got = dy.numpy()
    w64 = D.dequant_exact(qtype, packed, cols)
    for b in range(batch):
        assert D.rel_dot_error(w64, X[b], got[b]).max() < REL_TOL, b
        cpu = O.matvec(qtype, packed.reshape(-1), X[b], backend=O.AVX2)
        assert np.abs(got[b] - cpu).max() <= ABS_TOL + 1e-5 * np.abs(cpu).max(), b
    hip.matvec(W, dx, dy, batch=batch)
    assert np.array_equal(dy.numpy().view(np.uint32), got.view(np.uint32))  # reproducible bits


@pytest.mark.parametrize("B", [64, 300])  # 300: the many-sequence kernel (a batched prefill's shape)
def test_batched_swiglu_and_residual_chain(hip, B):
    """Transformer::forward's FFN chain (src/model.cpp:249-262) for 64 and 300 sequences at once."""
    print(f"[case] ffn chain B={B}", flush=True)
    D_, F = 2048, 5632
    X = np.stack([D.normal(40 + b, D_) for b in range(B)]).astype(np.float32)
    nw = (1.0 + 0.1 * D.normal(41, D_)).astype(np.float32)
    g = O.quantize(O.Q4_0, D.normal(42, (F, D_), 0.02))
    u = O.quantize(O.Q4_0, D.normal(43, (F, D_), 0.02))
    dn = O.quantize(O.Q4_0, D.normal(44, (D_, F), 0.02))
    G, U, Dn = (hip.Weight(O.Q4_0, F, D_, host=g), hip.Weight(O.Q4_0, F, D_, host=u),
                hip.Weight(O.Q4_0, D_, F, host=dn))
    dx = hip.DeviceArray.from_host(X)
    dnw = hip.DeviceArray.from_host(nw)
    dact = hip.DeviceArray((B, F))
    hip.matvec_swiglu(G, U, dx, dact, norm_w=dnw, eps=1e-5, batch=B)
    hip.matvec_residual(Dn, dact, dx, batch=B)  # K = 5632 at B = 64: split-K with a finalize pass
    got_act, got = dact.numpy(), dx.numpy()
    L = O.lib()
    for b in list(range(0, B, 9)) + [B - 1]:
        h = np.empty(D_, np.float32)
        L.efo_rmsnorm(O.ptr(h, O._f32p), O.ptr(X[b], O._f32p), O.ptr(nw, O._f32p), D_, 1e-5)
        gate, up = O.matvec_jobs([(O.Q4_0, g, h), (O.Q4_0, u, h)])
        act = np.empty_like(gate)
        L.efo_swiglu(O.ptr(act, O._f32p), O.ptr(gate, O._f32p), O.ptr(up, O._f32p), F)
        assert np.abs(got_act[b] - act).max() <= ABS_TOL, b
        ref = X[b] + O.matvec(O.Q4_0, dn.reshape(-1), got_act[b])
        assert np.abs(got[b] - ref).max() <= ABS_TOL, b


@pytest.mark.parametrize("B", [8, 270])
def test_batched_mixed_type_jobs_with_norm(hip, B):
    """q/k/v with k, v stored Q8_0 in one launch for 8 and 270 sequences, input RMSNorm fused."""
    print(f"[case] mixed q/k/v B={B}", flush=True)
    cols = 2048
    X = np.stack([D.normal(60 + b, cols) for b in range(B)]).astype(np.float32)
    nw = (1.0 + 0.05 * D.normal(61, cols)).astype(np.float32)
    shapes = [(O.Q4_0, 2048), (O.Q8_0, 256), (O.Q8_0, 256)]
    keep, ws, outs = [], [], []
    for i, (qt, rows) in enumerate(shapes):
        packed = O.quantize(qt, D.normal(70 + i, (rows, cols), 0.02))
        keep.append(packed)
        ws.append(hip.Weight(qt, rows, cols, host=packed))
        outs.append(hip.DeviceArray((B, 2048)))  # one output stride for the launch (the C-ABI's ldy)
    dx = hip.DeviceArray.from_host(X)
    hip.matvec_jobs_rmsnorm([(ws[i], dx, outs[i]) for i in range(3)], hip.DeviceArray.from_host(nw), 1e-5, batch=B,
                            ldx=cols, ldy=2048)
    L = O.lib()
    for b in range(0, B, 1 if B <= 16 else 7):
        h = np.empty(cols, np.float32)
        L.efo_rmsnorm(O.ptr(h, O._f32p), O.ptr(X[b], O._f32p), O.ptr(nw, O._f32p), cols, 1e-5)
        for i, (qt, rows) in enumerate(shapes):
            cpu = O.matvec(qt, keep[i].reshape(-1), h)
            assert np.abs(outs[i].numpy()[b, :rows] - cpu).max() <= ABS_TOL, (b, i)


@pytest.mark.parametrize("qtype", [O.Q4_0, O.Q8_0])
def test_batched_gemv_dynamic_range(hip, qtype):
    """Sequences 12 decades apart, one block 1e5 above the rest of its sequence and an all-zero
    sequence in one launch: each sequence meets the gates on its own (every sequence has its own
    power-of-two scale), and the zero sequence gives exact zeros."""
    rows, cols, B = 96, 2048, 20
    print(f"[case] batched gemv dynamic range qtype={qtype}", flush=True)
    packed = D.random_rows(qtype, rows, cols, seed=91)
    X = _batch_x(500, B, cols) * (10.0 ** np.linspace(-6.0, 6.0, B))[:, None]
    X[3, 64:96] *= 1e5
    X[7, :] = 0.0
    X = X.astype(np.float32)
    W = hip.Weight(qtype, rows, cols, host=packed)
    dx = hip.DeviceArray.from_host(X)
    dy = hip.DeviceArray((B, rows))
    hip.matvec(W, dx, dy, batch=B)
    got = dy.numpy()
    w64 = D.dequant_exact(qtype, packed, cols)
    for b in range(B):
        assert D.rel_dot_error(w64, X[b], got[b]).max() < REL_TOL, b
    assert not got[7].any()


def test_batched_norm_long_rows(hip):
    """An RMSNorm fused into a product whose rows are longer than one workgroup's blocks (K = 4096,
    a K split): the results meet the gates against the oracle's norm + matvec."""
    B, cols, rows = 6, 4096, 128
    X = np.stack([D.normal(80 + b, cols) for b in range(B)]).astype(np.float32)
    nw = (1.0 + 0.05 * D.normal(81, cols)).astype(np.float32)
    packed = O.quantize(O.Q4_0, D.normal(82, (rows, cols), 0.02))
    W = hip.Weight(O.Q4_0, rows, cols, host=packed)
    out = hip.DeviceArray((B, rows))
    hip.matvec_jobs_rmsnorm([(W, hip.DeviceArray.from_host(X), out)], hip.DeviceArray.from_host(nw), 1e-5,
                            batch=B, ldx=cols, ldy=rows)
    L = O.lib()
    for b in range(B):
        h = np.empty(cols, np.float32)
        L.efo_rmsnorm(O.ptr(h, O._f32p), O.ptr(X[b], O._f32p), O.ptr(nw, O._f32p), cols, 1e-5)
        assert np.abs(out.numpy()[b] - O.matvec(O.Q4_0, packed.reshape(-1), h)).max() <= ABS_TOL, b


@pytest.mark.parametrize("qtype", [O.Q4_0, O.Q8_0])
def test_refresh_after_rewriting_device_bytes(hip, qtype):
    """Batched products read a tile-order copy made on first use; ef_hip_weight_refresh rewrites it
    from the handle's current bytes, so a caller that rewrites the bytes sees the new matrix."""
    rows, cols, batch = 96, 512, 16
    print(f"[case] refresh qtype={qtype} {rows}x{cols} B={batch}", flush=True)
    first = D.random_rows(qtype, rows, cols, seed=11)
    second = D.random_rows(qtype, rows, cols, seed=12)
    buf = hip.DeviceArray.from_host(first.reshape(-1))
    W = hip.Weight(qtype, rows, cols, device=buf)
    X = _batch_x(77, batch, cols)
    dx = hip.DeviceArray.from_host(X)
    dy = hip.DeviceArray((batch, rows))
    hip.matvec(W, dx, dy, batch=batch)
    y_first = dy.numpy()
    buf.upload(second.reshape(-1))
    hip.matvec(W, dx, dy, batch=batch)
    assert np.array_equal(dy.numpy(), y_first)  # the copy still holds the former bytes
    W.refresh()
    hip.matvec(W, dx, dy, batch=batch)
    got = dy.numpy()
    w64 = D.dequant_exact(qtype, second, cols)
    for b in range(batch):
        assert D.rel_dot_error(w64, X[b], got[b]).max() < REL_TOL, b
    # batch 1 reads the bytes in place: the same matrix either way
    y1 = hip.DeviceArray((rows,))
    hip.matvec(W, hip.DeviceArray.from_host(X[0]), y1, batch=1)
    assert np.abs(y1.numpy() - got[0]).max() <= ABS_TOL + 1e-5 * np.abs(got[0]).max()


def _exact_close(W64, X, got, what):
    """|got - exact| <= 1e-5 * sum|w x| for every output (the single-vector gate)."""
    x = X.astype(np.float64)
    err = np.abs(got - x @ W64.T) / np.maximum(np.abs(x) @ np.abs(W64).T, 1e-30)
    assert err.max() < REL_TOL, (what, float(err.max()))


@pytest.mark.parametrize("qtype,rows,cols,batch", [
    (O.Q4_0, 2001, 2080, 900),   # an odd count of K blocks (65), a partial row tile, 57 sequence tiles
    (O.Q8_0, 2001, 2048, 900),
    (O.Q4_0, 600, 5632, 1100),   # long rows, few row groups: K shares
    (O.Q4_0, 3401, 256, 4100),   # two launches, the second of 4 sequences; 8 K blocks (one flush)
    (O.Q8_0, 15000, 2048, 129),  # one sequence past a tile
])
def test_many_sequence_kernel_edges(hip, qtype, rows, cols, batch):
    """The many-sequence kernel (3.5G multiply-adds or more in a call) at the edges of its tiles."""
    print(f"[case] many-sequence gemv qtype={qtype} {rows}x{cols} B={batch}", flush=True)
    packed = D.random_rows(qtype, rows, cols, seed=rows + batch)
    X = (D.rng(rows).standard_normal((batch, cols)) * np.exp(D.rng(cols).normal(size=(batch, 1)))).astype(np.float32)
    W = hip.Weight(qtype, rows, cols, host=packed)
    dx, dy = hip.DeviceArray.from_host(X), hip.DeviceArray((batch, rows))
    hip.matvec(W, dx, dy, batch=batch)
    got = dy.numpy()
    w64 = D.dequant_exact(qtype, packed, cols)
    _exact_close(w64, X, got, "store")
    base = D.rng(3).standard_normal((batch, rows)).astype(np.float32)
    dy.upload(base)
    hip.matvec_residual(W, dx, dy, batch=batch)
    # the same sums added to y: one more rounding of the result
    assert np.abs(dy.numpy() - (base + got)).max() <= 2.0 ** -23 * (np.abs(base) + np.abs(got)).max()
    # rows of x and y further apart than their lengths: the same bits, and nothing between the rows of y
    ldx, ldy = cols + 4, rows + 3
    wide = np.zeros((batch, ldx), np.float32)
    wide[:, :cols] = X
    dx2, dy2 = hip.DeviceArray.from_host(wide), hip.DeviceArray.from_host(np.full((batch, ldy), 7.0, np.float32))
    L.call("ef_hip_matvec", W.handle, dx2.ptr, dy2.ptr, batch, ldx, ldy, None)
    got2 = dy2.numpy()
    assert np.array_equal(got2[:, :rows].view(np.uint32), got.view(np.uint32))
    assert (got2[:, rows:] == 7.0).all()


def test_many_sequence_kernel_swiglu_and_mixed_jobs(hip):
    K, F, B = 2048, 1000, 900
    rng = D.rng(77)
    X = rng.standard_normal((B, K)).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    x64 = X.astype(np.float64)
    h = nw * (x64 / np.sqrt((x64 * x64).mean(1, keepdims=True) + 1e-5))
    dx, dn = hip.DeviceArray.from_host(X), hip.DeviceArray.from_host(nw)
    pk = [D.random_rows(O.Q4_0, F, K, seed=90 + i) for i in range(2)]
    G, U = [hip.Weight(O.Q4_0, F, K, host=p) for p in pk]
    dy = hip.DeviceArray((B, F))
    hip.matvec_swiglu(G, U, dx, dy, dn, 1e-5, batch=B)
    g, u = [h @ D.dequant_exact(O.Q4_0, p, K).T for p in pk]
    sg, su = [np.abs(h) @ np.abs(D.dequant_exact(O.Q4_0, p, K)).T for p in pk]
    want = g / (1 + np.exp(-g)) * u
    # each factor within 1e-5 of its sum of |w x| (|silu'| < 1.1), plus the FP32 rounding of the product
    bound = 1e-5 * (1.1 * sg * np.abs(u) + np.abs(g) * su) + 1e-6 * np.abs(want) + 1e-10 * sg * su
    assert (np.abs(dy.numpy() - want) <= bound).all()
    jobs, mats = [], []
    for i, (qt, rows) in enumerate([(O.Q4_0, 2048), (O.Q8_0, 130), (O.Q4_0, 70)]):
        p = D.random_rows(qt, rows, K, seed=95 + i)
        y = hip.DeviceArray((B, 2048))
        jobs.append((hip.Weight(qt, rows, K, host=p), dx, y))
        mats.append(D.dequant_exact(qt, p, K))
    hip.matvec_jobs_rmsnorm(jobs, dn, 1e-5, batch=B, ldx=K, ldy=2048)
    for (W, _, y), w64 in zip(jobs, mats):
        err = np.abs(y.numpy()[:, :W.rows] - h @ w64.T) / np.maximum(np.abs(h) @ np.abs(w64).T, 1e-30)
        assert err.max() < REL_TOL


def _in_new_thread(f):
    """f() in a thread of its own, which plans its launches anew (EF_HIP_GEMV_ROWS is read there)."""
    box = []

    def run():
        try:
            box.append((f(), None))
        except BaseException as e:  # re-raised below
            box.append((None, e))

    t = threading.Thread(target=run)
    t.start()
    t.join()
    if box[0][1] is not None:
        raise box[0][1]
    return box[0][0]


@pytest.mark.parametrize("stages", [1, 3, 17])  # a single one, an odd count, two flushes and one stage more
@pytest.mark.parametrize("qtype,ns,kw", [(qt, *s) for s in ((4, 1), (3, 1), (4, 2), (3, 2), (2, 2), (4, 4), (2, 4))
                                         for qt in (O.Q4_0, O.Q8_0)
                                         if (qt, *s) != (O.Q8_0, 4, 4)])  # whose stages do not fit the LDS
def test_many_sequence_kernel_every_shape(hip, monkeypatch, qtype, ns, kw, stages):
    """Each instantiated shape of the many-sequence kernel (ns sequence tiles, kw K shares), forced by
    EF_HIP_GEMV_ROWS: a partial row tile and workgroup (150 rows), a partial sequence tile and group, and more
    than 8 sequence groups (600 sequences); store and residual of one matrix, SwiGLU of two."""
    rows, K = 150, 32 * kw * stages
    print(f"[case] many-sequence kernel ns={ns} kw={kw} qtype={qtype} K={K}", flush=True)
    monkeypatch.setenv("EF_HIP_GEMV_ROWS", f"{ns},{kw}")
    pk = [D.random_rows(qtype, rows, K, seed=150 + K + i) for i in range(2)]
    w64 = [D.dequant_exact(qtype, p, K) for p in pk]
    G, U = [hip.Weight(qtype, rows, K, host=p) for p in pk]
    for batch in (35, 600):
        X = (D.rng(batch).standard_normal((batch, K)) * np.exp(D.rng(K).normal(size=(batch, 1)))).astype(np.float32)
        base = D.rng(3).standard_normal((batch, rows)).astype(np.float32)
        dx, ds, dr, dg = hip.DeviceArray.from_host(X), *[hip.DeviceArray.from_host(base) for _ in range(3)]

        def calls():
            hip.matvec(G, dx, ds, batch=batch)
            hip.matvec_residual(G, dx, dr, batch=batch)
            hip.matvec_swiglu(G, U, dx, dg, batch=batch)

        _in_new_thread(calls)
        got = ds.numpy()
        _exact_close(w64[0], X, got, "store")
        assert np.abs(dr.numpy() - (base + got)).max() <= 2.0 ** -23 * (np.abs(base) + np.abs(got)).max()
        x = X.astype(np.float64)
        g, u = [x @ w.T for w in w64]
        sg, su = [np.abs(x) @ np.abs(w).T for w in w64]
        with np.errstate(over="ignore"):
            want = g / (1 + np.exp(-g)) * u
        bound = 1e-5 * (1.1 * sg * np.abs(u) + np.abs(g) * su) + 1e-6 * np.abs(want) + 1e-10 * sg * su  # as above
        assert (np.abs(dg.numpy() - want) <= bound).all()


def test_kept_workspace_is_shared_in_order(hip):
    """Calls on the library's stream keep one workspace: calls of different shapes in turn and from two
    threads give the bits of calls on a stream of their own (which allocate)."""
    shapes = [(128, 1024, 5), (64, 2048, 40), (256, 5632, 64), (96, 4096, 300), (128, 1024, 5)]
    work = []
    for i, (rows, cols, batch) in enumerate(shapes):
        W = hip.Weight(O.Q4_0, rows, cols, host=D.random_rows(O.Q4_0, rows, cols, seed=120 + i))
        x = hip.DeviceArray.from_host(_batch_x(2000 + i, batch, cols))
        work.append((W, x, batch))
    s = hip.Stream()
    want = []
    for W, x, batch in work:
        y = hip.DeviceArray((batch, W.rows))
        hip.matvec(W, x, y, batch=batch, stream=s)
        want.append(y.numpy(s))
    outs = [[hip.DeviceArray((b, W.rows)) for W, _, b in work] for _ in range(2)]

    def enqueue(k):
        for _ in range(20):
            for (W, x, batch), y in zip(work, outs[k]):
                hip.matvec(W, x, y, batch=batch)

    threads = [threading.Thread(target=enqueue, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    hip.sync()
    for k in range(2):
        for y, w in zip(outs[k], want):
            assert np.array_equal(y.numpy().view(np.uint32), w.view(np.uint32))


def _grow_kept_workspace():
    """(In a process of its own, where nothing is kept yet.)  Workspaces of 0.1 to 70 MB, each call one that
    replaces the kept buffer while the launches that use the old one are still queued."""
    from edgeforge_amd import hip
    hip.init(0)
    work = []
    for i, (rows, cols, batch) in enumerate([(64, 1024, 5), (64, 2048, 200), (96, 4096, 300), (64, 5632, 600),
                                             (64, 5632, 1000), (64, 14336, 1000)]):
        W = hip.Weight(O.Q4_0, rows, cols, host=D.random_rows(O.Q4_0, rows, cols, seed=140 + i))
        x = hip.DeviceArray.from_host(_batch_x(2100 + i, batch, cols))
        work.append((W, x, batch))
    s = hip.Stream()
    want = []
    for W, x, batch in work:  # also makes the tile-order copies
        y = hip.DeviceArray((batch, W.rows))
        hip.matvec(W, x, y, batch=batch, stream=s)
        want.append(y.numpy(s))
    outs = [(i, hip.DeviceArray((batch, W.rows))) for i, (W, x, batch) in enumerate(work) for _ in range(30)]
    for i, y in outs:  # queued behind each other; the first of each shape replaces the kept workspace
        hip.matvec(work[i][0], work[i][1], y, batch=work[i][2])
    hip.sync()
    for i, y in outs:
        assert np.array_equal(y.numpy().view(np.uint32), want[i].view(np.uint32)), i
    print("grown", flush=True)


def test_kept_workspace_grows_under_queued_launches():
    print("[case] kept workspace growth in a process of its own", flush=True)
    r = subprocess.run([sys.executable, "-c", "from tests import test_gpu_gemv_batched as t; t._grow_kept_workspace()"],
                       cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "grown" in r.stdout, (r.returncode, r.stdout, r.stderr)
