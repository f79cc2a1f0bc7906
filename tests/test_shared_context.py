"""One context used by several threads, and graphs replayed through a context other than the one that captured them:
calls that hand data from one launch to the next in the context's workspaces must not meet there (GPU)."""
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
