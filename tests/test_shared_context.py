"""One context used by several threads, and graphs replayed through a context other than the one that captured them:
calls that hand data from one launch to the next in the context's workspaces must not meet there (GPU)."""
import ctypes as C
import threading

import numpy as np
import pytest

import p0k
from cases import make_case

pytestmark = pytest.mark.gpu

# calls of several launches: X' and a decode, X' and slices of K, slices alone, X' and one GEMM
SHARED_CALLS = [
    dict(enc="q8g64s.t64", xmode="rms", epi="f16", M=12, N=512, K=4096, wscale=0.02, seed=41),
    dict(enc="q4g32a.t64", xmode="lnmod", epi="f16", M=77, N=512, K=4096, wscale=0.02, seed=42),
    dict(enc="f16", epi="f16", M=40, N=256, K=4096, wscale=0.02, seed=43),
    dict(enc="q8g64s.t64", xmode="rms", epi="f16", M=300, N=256, K=512, wscale=0.02, seed=44),
]


def test_threads_share_a_context():
    """Four threads, each enqueueing its own call again and again into buffers of its own, get the bits that each call
    gives alone (the first calls also grow the workspaces under the other threads)."""
    cs = [make_case(**kw) for kw in SHARED_CALLS]
    dev, alone = p0k.Device(0), p0k.Device(0)
    try:
        want = [c.run_device(alone) for c in cs]
        ins = [{k: dev.upload(v) for k, v in c.bufs.items() if k != "y"} for c in cs]
        outs = [[dev.buffer(c.bufs["y"].nbytes) for _ in range(16)] for c in cs]
        start, errs = threading.Barrier(len(cs)), []

        def work(i):
            try:
                start.wait()
                for y in outs[i]:
                    dev.gemm(cs[i].args(lambda n: y if n == "y" else ins[i][n]))
            except Exception as e:                       # noqa: BLE001 (shown by the main thread)
                errs.append((i, e))

        ts = [threading.Thread(target=work, args=(i,)) for i in range(len(cs))]
        print("[p0k-test] four threads on one context", flush=True)
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not errs, errs
        for i, c in enumerate(cs):
            for y in outs[i]:
                assert np.array_equal(dev.read(y, np.uint16, c.bufs["y"].size), want[i]), SHARED_CALLS[i]
    finally:
        dev.close()
        alone.close()


@pytest.mark.parametrize("what", ["attention over runs of keys", "X' and slices of K"])
def test_graph_launched_through_another_context(what):
    """A graph whose calls use workspaces, replayed through a second context while the first one's own calls use the same
    workspaces: both keep the bits they have alone, again and again, and the second context refuses the graph once the
    first is gone."""
    own, other = p0k.Device(0), p0k.Device(0)
    print(f"[p0k-test] graph through another context: {what}", flush=True)
    try:
        if what.startswith("attention"):
            Hq, Hkv, Lk = 32, 8, 3777
            rng = np.random.default_rng(5)
            calls, outs, size = [], [], Hq * 128
            for _ in range(2):
                q, k, v = (own.upload((rng.standard_normal(n * 128)).astype(np.float16)) for n in (Hq, Hkv * Lk, Hkv * Lk))
                o = own.buffer(size * 2)
                a = {"q": {"buf": q}, "k": {"buf": k}, "v": {"buf": v}, "o": {"buf": o}, "Lq": 1, "Lk": Lk, "Hq": Hq,
                     "Hkv": Hkv, "mode": 2, "nvalid": Lk}
                calls.append(lambda a=a: own.attention(a))
                outs.append(o)
        else:
            cs = [make_case(enc="q4g32a.t64", xmode="rms", epi="f16", M=77, N=512, K=4096, wscale=0.02, seed=s) for s in (45, 46)]
            ds = [{k: own.upload(v) for k, v in c.bufs.items()} for c in cs]
            calls = [lambda c=c, d=d: own.gemm(c.args(lambda n: d[n])) for c, d in zip(cs, ds)]
            outs, size = [d["y"] for d in ds], cs[0].bufs["y"].size
        want = []
        for call, o in zip(calls, outs):
            call()
            want.append(own.read(o, np.uint16, size))
        own.graph_begin()
        calls[0]()
        g = own.graph_end()
        zero = np.zeros(size, np.uint16)
        for rep in range(10):
            for o in outs:
                own.upload(zero, o)
            for _ in range(4):
                calls[1]()
                other.graph_launch(g)
            calls[1]()
            for o, w in zip(outs, want):                 # (the read waits for the other context's replays too)
                assert np.array_equal(own.read(o, np.uint16, size), w), f"repetition {rep}"
        own.graph_launch(g)
        assert np.array_equal(own.read(outs[0], np.uint16, size), want[0])
        own.graph_begin()
        with pytest.raises(p0k.P0kError, match="is captured"):
            other.graph_launch(g)
        own.graph_destroy(own.graph_end())
        own.close()
        with pytest.raises(p0k.P0kError, match="destroyed"):
            other.graph_launch(g)
        p0k.Device.graph_destroy(g)
    finally:
        own.close()
        other.close()


def test_capture_ended_by_the_caller_is_forgotten():
    """p0k_graph_begin's capture ended with the HIP API, then a capture begun by the caller: its attention call takes no
    workspace (one run of keys: the bits of any other caller's capture, not those of the runs)."""
    hip, dev = C.CDLL("libamdhip64.so"), p0k.Device(0)
    s = C.c_void_p(p0k.lib().p0k_ctx_stream(dev.ctx))
    rng = np.random.default_rng(6)
    Hq, Hkv, Lk = 32, 8, 3777
    q, k, v = (dev.upload(rng.standard_normal(n * 128).astype(np.float16)) for n in (Hq, Hkv * Lk, Hkv * Lk))
    o = dev.buffer(Hq * 256)
    a = {"q": {"buf": q}, "k": {"buf": k}, "v": {"buf": v}, "o": {"buf": o}, "Lq": 1, "Lk": Lk, "Hq": Hq, "Hkv": Hkv}

    def captured():
        graph, exe = C.c_void_p(), C.c_void_p()
        dev.done()
        assert hip.hipStreamBeginCapture(s, 1) == 0
        try:
            dev.attention(a)
        finally:
            assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
        assert hip.hipGraphLaunch(exe, s) == 0
        got = dev.read(o, np.uint16, Hq * 128)
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)
        return got

    print("[p0k-test] a capture ended by the caller", flush=True)
    try:
        dev.attention(a)
        runs, one = dev.read(o, np.uint16, Hq * 128), captured()
        assert not np.array_equal(runs, one)
        graph = C.c_void_p()
        dev.graph_begin()
        assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
        hip.hipGraphDestroy(graph)
        assert np.array_equal(captured(), one)
    finally:
        dev.close()


def test_graph_without_workspaces_is_launched_freely():
    """A graph none of whose calls took a workspace (a prompt captured before the workspace for its slices of K was there
    among them) has no order to keep: another context launches it also while the first is being captured."""
    own, other = p0k.Device(0), p0k.Device(0)
    print("[p0k-test] graph without workspaces", flush=True)
    try:
        cs = [make_case(enc="q4g32a.t64", epi="f16", M=M, N=512, K=4096, wscale=0.02, seed=47) for M in (1, 77)]
        ds = [{k: own.upload(v) for k, v in c.bufs.items()} for c in cs]
        own.graph_begin()
        for c, d in zip(cs, ds):
            own.gemm(c.args(lambda n: d[n]))
        g = own.graph_end()
        own.graph_begin()
        other.graph_launch(g)
        own.graph_destroy(own.graph_end())
        other.done()
        for c, d in zip(cs, ds):
            got, size = own.read(d["y"], np.uint16, c.bufs["y"].size), c.bufs["y"].size
            own.upload(np.zeros(size, np.uint16), d["y"])
            own.graph_launch(g)
            assert got.any() and np.array_equal(own.read(d["y"], np.uint16, size), got)
        own.graph_destroy(g)
    finally:
        own.close()
        other.close()
