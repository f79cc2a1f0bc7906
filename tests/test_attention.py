"""attention (src/ops/attention.js:168), head size 128 — the consumer of the `heads` epilogue's output.

CPU: the oracle (a restatement of the test suite's cpuAttn, test/kernels.test.js:30-49) against an independent numpy
formulation (masked softmax(Q K^T scale) V per head), the three mask modes, GQA and the soft cap.
GPU: the HIP kernel against the oracle on the reference's own cases (test/kernels.test.js:148-152, seeds and scales
as attnSetup at :153-157) plus ragged lengths, GQA 8:1, an offset O with ld > Hq * 128, and the soft cap.
Tolerance (fp16 output): |got - want| <= 2^-8 * max|want| + 2^-9 |want|, and the reference's cos > 0.9995; P is
rounded to fp16 before the P.V products, as in the reference kernels (pv16)."""
import ctypes as C

import numpy as np
import pytest

import oracle
import p0k

ATT = [  # test/kernels.test.js:148-152
    dict(label="no mask", Hq=2, Hkv=2, Lq=96, Lk=96, mode=0),
    dict(label="causal + valid length 80, GQA 4:2", Hq=4, Hkv=2, Lq=96, Lk=96, mode=1, nvalid=80),
    dict(label="valid length 77 of 100 keys, 64 queries", Hq=2, Hkv=2, Lq=64, Lk=100, mode=2, nvalid=77),
]
MORE = [
    dict(label="ragged 300 x 257, GQA 8:1", Hq=8, Hkv=1, Lq=300, Lk=257, mode=0),
    dict(label="causal 200, valid 150", Hq=2, Hkv=1, Lq=200, Lk=200, mode=1, nvalid=150),
    dict(label="one query", Hq=3, Hkv=3, Lq=1, Lk=130, mode=2, nvalid=129),
    dict(label="soft cap 1.0", Hq=2, Hkv=2, Lq=70, Lk=90, mode=0, cap=1.0),
]


def setup(c, seed, qs=0.5):
    """attnSetup (test/kernels.test.js:153-157): Q, K = f16(randn * 0.5), V = f16(randn)."""
    D = 128
    q = oracle.f16_bits(oracle.randn(c["Hq"] * c["Lq"] * D, seed, qs))
    k = oracle.f16_bits(oracle.randn(c["Hkv"] * c["Lk"] * D, seed + 1, qs))
    v = oracle.f16_bits(oracle.randn(c["Hkv"] * c["Lk"] * D, seed + 2))
    return q, k, v


def numpy_attention(q, k, v, c):
    D, Hq, Hkv, Lq, Lk = 128, c["Hq"], c["Hkv"], c["Lq"], c["Lk"]
    Q = oracle.h2f(q).astype(np.float64).reshape(Hq, Lq, D)
    K = oracle.h2f(k).astype(np.float64).reshape(Hkv, Lk, D)
    V = oracle.h2f(v).astype(np.float64).reshape(Hkv, Lk, D)
    nv = c.get("nvalid", Lk)
    i, j = np.arange(Lq)[:, None], np.arange(Lk)[None, :]
    vis = {0: np.ones((Lq, Lk), bool), 1: j <= np.minimum(i, nv - 1), 2: np.broadcast_to(j < nv, (Lq, Lk))}[c["mode"]]
    out = np.zeros((Lq, Hq, D))
    for h in range(Hq):
        s = Q[h] @ K[h // (Hq // Hkv)].T / np.sqrt(128.0)
        if c.get("cap"):
            s = c["cap"] * np.tanh(s / c["cap"])
        s = np.where(vis, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ V[h // (Hq // Hkv)]
    return out.reshape(Lq, Hq * D)


@pytest.mark.parametrize("c", ATT + MORE, ids=lambda c: c["label"])
def test_oracle_is_masked_softmax(c):
    q, k, v = setup(c, 21)
    got = oracle.h2f(oracle.attention(q, k, v, c["Lq"], c["Lk"], c["Hq"], c["Hkv"], c["mode"], c.get("nvalid"),
                                      cap=c.get("cap", 0.0))).reshape(c["Lq"], -1)
    want = numpy_attention(q, k, v, c)
    np.testing.assert_allclose(got, want, rtol=2 ** -10, atol=2 ** -14)


def test_attention_checks():
    base = dict(Lq=4, Lk=4, Hq=2, Hkv=2)
    bufs = {n: np.zeros(4096, np.uint16) for n in "qkvo"}

    def check(**kw):
        a = {n: {"buf": bufs[n]} for n in "qkvo"}
        a.update(base)
        a.update(kw)
        return p0k.lib().p0k_attention_check(p0k.C.byref(p0k.attn_args(a, p0k.numpy_resolve)))
    assert check() == 0
    assert check(Hkv=3) == 1 and "multiple of Hkv" in p0k.lib().p0k_last_error().decode()
    assert check(mode=3) == 1
    assert check(mode=2, nvalid=9) == 1
    assert check(Lq=64) == 1 and "needs" in p0k.lib().p0k_last_error().decode()


# ------------------------------------------------------------------------------------------------ GPU
def cos_and_err(got, want):
    g, w = got.astype(np.float64).ravel(), want.astype(np.float64).ravel()
    return g @ w / (np.linalg.norm(g) * np.linalg.norm(w) + 1e-30), np.abs(g - w)


@pytest.mark.gpu
@pytest.mark.parametrize("bq", [128, 256])
@pytest.mark.parametrize("c", ATT + MORE, ids=lambda c: c["label"])
def test_attention_matches_oracle(dev, c, bq, monkeypatch):
    """Both workgroup sizes on every case (the library takes 128 queries; 256 are a tuning switch)."""
    monkeypatch.setenv("P0K_ATTN_BQ", str(bq))
    print(f"attention bq={bq} {c}", flush=True)
    q, k, v = setup(c, 21, 1.0 if c.get("cap") else 0.5)
    Lq, Hq = c["Lq"], c["Hq"]
    ld = Hq * 128 + (8 if c["mode"] == 2 else 0)                       # a padded O row for one case
    dq, dk, dv = dev.upload(q), dev.upload(k), dev.upload(v)
    do = dev.buffer(Lq * ld * 2 + 16)
    try:
        flops = dev.attention({"q": {"buf": dq}, "k": {"buf": dk}, "v": {"buf": dv}, "o": {"buf": do, "off": 16, "ld": ld},
                               "Lq": Lq, "Lk": c["Lk"], "Hq": Hq, "Hkv": c["Hkv"], "mode": c["mode"],
                               "nvalid": c.get("nvalid", 0), "cap": c.get("cap", 0.0)})
        assert flops == 4 * Lq * c["Lk"] * 128 * Hq
        o = dev.read(do, np.uint16, (Lq * ld * 2 + 16) // 2)
        assert np.all(o[:8] == 0)
        got = o[8:8 + Lq * ld].reshape(Lq, ld)
        if ld > Hq * 128:
            assert np.all(got[:, Hq * 128:] == 0)
        got = oracle.h2f(got[:, :Hq * 128].ravel())
        want = oracle.h2f(oracle.attention(q, k, v, Lq, c["Lk"], Hq, c["Hkv"], c["mode"], c.get("nvalid"),
                                           cap=c.get("cap", 0.0)))
        cos, err = cos_and_err(got, want)
        assert cos > 0.9995
        bound = 2 ** -8 * np.abs(want).max() + 2 ** -9 * np.abs(want)
        assert np.all(err <= bound), f"max err {err.max()} (bound {bound.max()})"
    finally:
        for d in (dq, dk, dv, do):
            dev.free(d)


# Causal grids of more blocks than CUs, longest blocks first: heads a multiple of 8 (an XCD's own) and not, all blocks
# resident at once (the second on each CU in the opposite order) and more, a valid length that levels the work
@pytest.mark.gpu
# (cap: the soft-capped kernels; bq 256: the blocks of the tuning switch)
@pytest.mark.parametrize("Hq,Hkv,L,nvalid,cap,bq", [(40, 8, 900, 900, 0, 0), (35, 7, 1000, 990, 0, 0), (48, 6, 1500, 700, 0, 0), (72, 9, 513, 513, 0, 0),
                                                    (40, 8, 900, 880, 2.0, 0), (48, 6, 1500, 1500, 2.0, 0), (72, 9, 1000, 990, 0, 256), (35, 7, 2000, 1999, 2.0, 256)])
def test_attention_causal_block_order(dev, Hq, Hkv, L, nvalid, cap, bq, monkeypatch):
    """Sampled rows of every head and block against float64 numpy, with the file's fp16 tolerance (every block of the
    grid computes some of them, so a block taken twice and another never would show)."""
    print(f"causal order Hq={Hq} L={L} nvalid={nvalid} cap={cap} bq={bq}", flush=True)
    if bq:
        monkeypatch.setenv("P0K_ATTN_BQ", str(bq))
    assert (L + (bq or 128) - 1) // (bq or 128) * Hq > dev.cus()
    c = dict(Hq=Hq, Hkv=Hkv, Lq=L, Lk=L, mode=1, nvalid=nvalid)
    q, k, v = setup(c, 23)
    bufs = [dev.upload(a) for a in (q, k, v)] + [dev.buffer(L * Hq * 256)]
    try:
        dev.attention({"q": {"buf": bufs[0]}, "k": {"buf": bufs[1]}, "v": {"buf": bufs[2]}, "o": {"buf": bufs[3]}, "Lq": L,
                       "Lk": L, "Hq": Hq, "Hkv": Hkv, "mode": 1, "nvalid": nvalid, "cap": cap})
        got = oracle.h2f(dev.read(bufs[3], np.uint16, L * Hq * 128)).reshape(L, Hq, 128)
    finally:
        for b in bufs:
            dev.free(b)
    Q, K, V = (oracle.h2f(a).astype(np.float64).reshape(n, L, 128) for a, n in ((q, Hq), (k, Hkv), (v, Hkv)))
    rows = sorted({min(L - 1, 128 * b + o) for b in range((L + 127) // 128) for o in (0, 31, 127)})
    for h in range(Hq):
        s = Q[h, rows] @ K[h // (Hq // Hkv)].T / np.sqrt(128.0)
        s = cap * np.tanh(s / cap) if cap else s
        s = np.where(np.arange(L)[None, :] <= np.minimum(np.array(rows), nvalid - 1)[:, None], s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        want = (p / p.sum(1, keepdims=True)) @ V[h // (Hq // Hkv)]
        err = np.abs(got[rows, h] - want)
        assert np.all(err <= 2 ** -8 * np.abs(want).max() + 2 ** -9 * np.abs(want)), f"head {h}: max err {err.max()}"


# The few-queries kernel (32-row blocks of a kv head's packed query heads, runs of 32-key tiles over 4 waves): rows and
# keys at the edges of its blocks, tiles and 128-key sets, one run and several, every mask mode
FEW = [dict(Hq=h, Hkv=k, Lq=q, Lk=n, mode=m, nvalid=v, cap=cap) for h, k, q, n, m, v, cap in [
    (1, 1, 1, 1, 0, 1, 0), (3, 3, 1, 31, 0, 31, 0), (8, 2, 1, 32, 2, 32, 0), (8, 2, 1, 33, 2, 33, 0),
    (4, 4, 1, 128, 2, 127, 0), (32, 8, 1, 1000, 2, 129, 0), (32, 8, 1, 1000, 2, 999, 0), (5, 1, 2, 700, 0, 700, 0),
    (2, 2, 16, 520, 2, 517, 0), (8, 2, 8, 300, 0, 300, 0), (3, 1, 11, 385, 2, 385, 0), (8, 2, 16, 260, 2, 255, 0),
    (2, 1, 32, 200, 1, 20, 0), (4, 2, 16, 64, 1, 64, 0), (6, 2, 100, 333, 1, 80, 0), (2, 2, 700, 700, 1, 700, 0),
    (3, 1, 70, 1500, 0, 1500, 0), (8, 2, 1, 900, 2, 890, 1.0), (300, 300, 1, 200, 2, 180, 0)]]


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["eager", "graph", "caller's capture"])
@pytest.mark.parametrize("c", FEW, ids=lambda c: "Hq{Hq} Hkv{Hkv} Lq{Lq} Lk{Lk} mode{mode} nvalid{nvalid} cap{cap}".format(**c))
def test_attention_few_queries(dev, c, how):
    """Against the oracle with the file's fp16 tolerance; twice with the same bits (the runs merge in order, counters
    are left at zero), replayed from the library's graph, and under a capture begun by the caller (no workspace)."""
    print(f"few queries {how} {c}", flush=True)
    q, k, v = setup(c, 21, 1.0 if c["cap"] else 0.5)
    Lq, Hq = c["Lq"], c["Hq"]
    n, ld = Lq * (Hq * 128 + 4), Hq * 128 + 4
    bufs = [dev.upload(q), dev.upload(k), dev.upload(v), dev.buffer(n * 2)]
    a = {"q": {"buf": bufs[0]}, "k": {"buf": bufs[1]}, "v": {"buf": bufs[2]}, "o": {"buf": bufs[3], "ld": ld}, "Lq": Lq,
         "Lk": c["Lk"], "Hq": Hq, "Hkv": c["Hkv"], "mode": c["mode"], "nvalid": c["nvalid"], "cap": c["cap"]}
    got = []
    try:
        if how == "eager":
            for _ in range(2):
                dev.attention(a)
                got.append(dev.read(bufs[3], np.uint16, n))
        elif how == "graph":
            dev.graph_begin()
            dev.attention(a)
            g = dev.graph_end()
            for _ in range(3):
                dev.upload(np.zeros(n, np.uint16), bufs[3])
                dev.graph_launch(g)
                got.append(dev.read(bufs[3], np.uint16, n))
            dev.graph_destroy(g)
        else:
            hip, s = C.CDLL("libamdhip64.so"), C.c_void_p(p0k.lib().p0k_ctx_stream(dev.ctx))
            graph, exe = C.c_void_p(), C.c_void_p()
            dev.done()
            assert hip.hipStreamBeginCapture(s, 1) == 0          # thread-local capture mode
            try:
                dev.attention(a)
            finally:
                assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            for _ in range(2):
                assert hip.hipGraphLaunch(exe, s) == 0
                got.append(dev.read(bufs[3], np.uint16, n))
            hip.hipGraphExecDestroy(exe)
            hip.hipGraphDestroy(graph)
    finally:
        for b in bufs:
            dev.free(b)
    assert all(np.array_equal(g, got[0]) for g in got)
    o = got[0].reshape(Lq, ld)
    assert np.all(o[:, Hq * 128:] == 0)
    want = oracle.h2f(oracle.attention(q, k, v, Lq, c["Lk"], Hq, c["Hkv"], c["mode"], c["nvalid"], cap=c["cap"]))
    err = np.abs(oracle.h2f(o[:, :Hq * 128].ravel()) - want)
    bound = 2 ** -8 * np.abs(want).max() + 2 ** -9 * np.abs(want)
    assert np.all(err <= bound), f"max err {err.max()} (bound {bound.max()})"


@pytest.mark.gpu
@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("Lq,Lk,nvalid", [(1, 3000, 2500), (16, 700, 389), (40, 300, 200)])
def test_attention_values_that_are_not_finite(dev, Lq, Lk, nvalid, split, monkeypatch):
    """Both kernels. NaN in the cache past the last tile of 64 keys that the valid length reaches: not seen. Keys whose score
    is -inf: as if they were not there. A key whose score is +inf: NaN, in every row that sees it."""
    monkeypatch.setenv("P0K_ATTN_SPLIT", split)
    print(f"not finite Lq={Lq} Lk={Lk} nvalid={nvalid} split={split}", flush=True)
    c = dict(Hq=4, Hkv=2, Lq=Lq, Lk=Lk, mode=2, nvalid=nvalid)
    rng = np.random.default_rng(Lk)
    Q = np.abs(rng.standard_normal((4, Lq, 128)) * 0.5).astype(np.float16) + np.float16(0.01)     # (positive)
    K = (rng.standard_normal((2, Lk, 128)) * 0.5).astype(np.float16)
    V = rng.standard_normal((2, Lk, 128)).astype(np.float16)

    def run(K, V):
        bufs = [dev.upload(a) for a in (Q, K, V)] + [dev.buffer(Lq * 4 * 256)]
        try:
            dev.attention({"q": {"buf": bufs[0]}, "k": {"buf": bufs[1]}, "v": {"buf": bufs[2]}, "o": {"buf": bufs[3]}, **c})
            return oracle.h2f(dev.read(bufs[3], np.uint16, Lq * 512)).reshape(Lq, 4, 128)
        finally:
            for b in bufs:
                dev.free(b)

    clean = run(K, V)
    Kn, Vn = K.copy(), V.copy()
    Kn[:, (nvalid + 63) // 64 * 64:] = Vn[:, (nvalid + 63) // 64 * 64:] = np.nan
    assert np.array_equal(run(Kn, Vn), clean) and np.isfinite(clean).all()
    gone = [0, 31, 32, 100, nvalid - 1]
    Ki = K.copy()
    Ki[:, gone] = -np.inf
    keep = np.setdiff1d(np.arange(nvalid), gone)
    want = numpy_attention(Q.view(np.uint16), np.ascontiguousarray(K[:, keep]).view(np.uint16), np.ascontiguousarray(V[:, keep]).view(np.uint16),
                           dict(c, Lk=keep.size, mode=0)).reshape(Lq, 4, 128)
    err = np.abs(run(Ki, V) - want)
    assert np.all(err <= 2 ** -8 * np.abs(want).max() + 2 ** -9 * np.abs(want)), f"max err {err.max()}"
    Kp = K.copy()
    Kp[0, 150] = np.inf                                   # kv head 0: query heads 0 and 1
    got = run(Kp, V)
    assert np.isnan(got[:, :2]).all() and np.array_equal(got[:, 2:], clean[:, 2:])


@pytest.mark.gpu
@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("pattern", ["slow ramp", "fast ramp", "late spike", "falling"])
def test_attention_moving_maximum(dev, pattern, split, monkeypatch):
    """Scores whose row maximum keeps moving across the 64-key tiles: the kernel keeps the subtracted maximum until a
    row's maximum outgrows it by more than 8 in the log2 domain (P up to 2^8 meanwhile) and rescales O and l when it
    moves. Every query sees s_j = g(j) + noise: a slow ramp (about 4 log2 units per tile: the maximum moves every other
    tile), a fast ramp (16 per tile: every tile), one late spike (25 units in one tile) and a falling ramp (the maximum
    is set by the first tile and never moves); against float64 numpy with the file's fp16 tolerance. Both kernels: the
    one over 128-query blocks (split 0) and the one over runs of keys, whose runs and waves each have their own."""
    monkeypatch.setenv("P0K_ATTN_SPLIT", split)
    Hq, Lq, Lk, D = 2, 128, 512, 128
    j = np.arange(Lk, dtype=np.float64)
    g = {"slow ramp": 0.5 * j, "fast ramp": 2.0 * j, "late spike": np.where(j == 300, 200.0, 0.0),
         "falling": 60.0 - 0.1 * j}[pattern]
    rng = np.random.default_rng(7)
    # q = (1, ..., 1) + noise, k_j = g(j) / 128 (1, ..., 1) + noise: q . k_j = g(j) + O(noise)
    Q = np.ones((Hq, Lq, D)) + 0.05 * rng.standard_normal((Hq, Lq, D))
    K = np.repeat((g / 128.0)[None, :, None], D, axis=2).repeat(Hq, axis=0) + 0.05 * rng.standard_normal((Hq, Lk, D))
    V = rng.standard_normal((Hq, Lk, D))
    q, k, v = (oracle.f16_bits(a.astype(np.float32).ravel()) for a in (Q, K, V))
    c = dict(Hq=Hq, Hkv=Hq, Lq=Lq, Lk=Lk, mode=0)
    dq, dk, dv, do = dev.upload(q), dev.upload(k), dev.upload(v), dev.buffer(Lq * Hq * D * 2)
    try:
        dev.attention({"q": {"buf": dq}, "k": {"buf": dk}, "v": {"buf": dv}, "o": {"buf": do}, "Lq": Lq, "Lk": Lk,
                       "Hq": Hq, "Hkv": Hq})
        got = oracle.h2f(dev.read(do, np.uint16, Lq * Hq * D))
    finally:
        for d in (dq, dk, dv, do):
            dev.free(d)
    want = numpy_attention(q, k, v, c).ravel()
    err = np.abs(got - want)
    bound = 2 ** -8 * np.abs(want).max() + 2 ** -9 * np.abs(want)
    assert np.all(err <= bound), f"{pattern}: max err {err.max()} (bound {bound.max()})"
