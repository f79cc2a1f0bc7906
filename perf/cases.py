"""Performance cases of the `gemm` path and its neighbours: what a program that runs a quantised language model, a
diffusion transformer or an image / video decoder on this library asks of it, through the Python binding of the C ABI.

A case is a dict of plain values. Its "op" names the part of such a program:

  linear   one projection: [rowstats ->] gemm
  mlp      a feed-forward block: residual copy -> rowstats -> up-projection with its gated activation -> down-projection
           added to the residual
  attn     attention over head-major Q / K / V (a decode step over a KV cache, a causal prompt, a full image)
  block    a transformer's attention block: rowstats -> QKV with norm + RoPE into heads -> attention -> output
           projection, gated, added to the residual
  conv3    a 3x3x3 convolution over a clip (video decoder), with or without its PixelNorm + SiLU prologue
  conv2d   a 2-D convolution over an image (image decoder): GroupNorm statistics -> convolution with GroupNorm + SiLU
           applied on the way in, bias, optionally 2x up-sampling

"graph": the program captures its calls once and replays them (a decode loop, a serving bucket); otherwise it enqueues
each call. Weights are N(0, scale) in the library's own encodings, activations fp16 N(0, 1).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath(os.path.join("p0pc0rn-kernels_amd", "python")))
import p0k  # noqa: E402

Q4, Q8, F16 = "q4g32a.t64", "q8g64s.t64", "f16"
_dev = None


def _device():
    global _dev
    if _dev is None:
        torch.cuda.init()
        _dev = p0k.Device(0)
    return _dev


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call there is: one token through an attention projection of an 8B-sized language model
        {"name": "decode_proj", "op": "linear", "enc": Q4, "M": 1, "N": 4096, "K": 4096, "x": "f16", "epi": "f16",
         "graph": False},
        # one token through that model's feed-forward block, replayed as a decode loop does
        {"name": "decode_mlp", "op": "mlp", "enc": Q4, "M": 1, "K": 4096, "F": 14336, "x": "rms", "act": "silu",
         "graph": True},
        # a dozen sequences decoded together, 8-bit weights
        {"name": "decode_mlp_batch", "op": "mlp", "enc": Q8, "M": 12, "K": 4096, "F": 14336, "x": "rms",
         "act": "silu", "graph": True},
        # one token attending to a long KV cache, 4 query heads to a key head
        {"name": "decode_attn", "op": "attn", "Lq": 1, "Lk": 4096, "Hq": 32, "Hkv": 8, "mode": 2, "nvalid": 3777,
         "graph": False},
        # a short prompt of odd length: QKV with RMSNorm in front and norm + RoPE behind
        {"name": "prompt_qkv", "op": "linear", "enc": Q4, "M": 77, "N": 6144, "K": 4096, "x": "rms", "epi": "heads",
         "graph": True},
        # an ordinary prompt through the feed-forward block
        {"name": "prompt_mlp", "op": "mlp", "enc": Q4, "M": 300, "K": 4096, "F": 14336, "x": "rms", "act": "silu",
         "graph": True},
        # a long prompt through a projection, 8-bit weights, added to the residual
        {"name": "prefill_q8", "op": "linear", "enc": Q8, "M": 2048, "N": 4096, "K": 4096, "x": "rms",
         "epi": "resadd", "graph": False},
        # causal attention of a long prompt, its length no multiple of anything
        {"name": "prefill_attn", "op": "attn", "Lq": 1999, "Lk": 1999, "Hq": 32, "Hkv": 8, "mode": 1, "nvalid": 1999,
         "graph": False},
        # the attention block of a diffusion transformer, 64 x 64 latent patches
        {"name": "dit_attn_block", "op": "block", "enc": Q4, "M": 4096, "K": 3072, "H": 24, "graph": False},
        # its feed-forward block (GeGLU): the largest matrix products
        {"name": "dit_mlp", "op": "mlp", "enc": Q4, "M": 4096, "K": 3072, "F": 12288, "x": "lnmod", "act": "gelu",
         "graph": False},
        # a video decoder's convolution at full latent size
        {"name": "video_conv3", "op": "conv3", "T": 13, "H": 92, "W": 160, "C": 128, "N": 128, "pn": False,
         "graph": False},
        # an image decoder's convolution with its GroupNorm
        {"name": "image_conv2d", "op": "conv2d", "H": 128, "W": 128, "C": 256, "N": 256, "stride": 1, "up2": False,
         "graph": False},
    ]


def _log(rng, lo, hi, step=1):
    """a size between lo and hi, even over its logarithm, a multiple of step"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "attn", "attn", "block", "conv3", "conv2d"])
    if op == "linear":
        x, epi = rng.choice(["f16", "rms", "lnmod"]), rng.choice(["f16", "f32", "bias", "resadd", "swiglu", "heads"])
        K = _log(rng, 1024, 14336, 64)
        N = _log(rng, 1024, 28672, 128)
        if epi in ("f16", "bias") and rng.random() < 0.3:
            N -= rng.choice([1, 7, 40])
        M = rng.choice([_log(rng, 1, 16), _log(rng, 17, 512), _log(rng, 512, 4096)])
        M = min(M, max(1, int(2e11 / (N * K))))
        return {"op": op, "enc": rng.choice([Q4, Q4, Q8, F16]), "M": M, "N": N, "K": K, "x": x, "epi": epi,
                "graph": M <= 512}
    if op == "mlp":
        M = rng.choice([_log(rng, 1, 16), _log(rng, 17, 4096)])
        K = _log(rng, 1024, 4096, 128)
        x = rng.choice(["rms", "lnmod"])
        return {"op": op, "enc": rng.choice([Q4, Q8]), "M": M, "K": K, "F": _log(rng, 2048, 14336 if M <= 2048 else 12288, 128),
                "x": x, "act": "silu" if x == "rms" else "gelu", "graph": M <= 512}
    if op == "attn":
        Hkv, rep = rng.choice([4, 8, 16]), rng.choice([1, 2, 4])
        if rng.random() < 0.5:
            Lk = _log(rng, 128, 16384)
            return {"op": op, "Lq": rng.choice([1, 1, rng.randint(2, 16)]), "Lk": Lk, "Hq": Hkv * rep, "Hkv": Hkv,
                    "mode": 2, "nvalid": rng.randint(Lk // 2, Lk), "graph": False}
        Lq, mode = _log(rng, 64, 4096), rng.choice([0, 1])
        Lk = Lq if mode == 1 else rng.choice([Lq, _log(rng, 64, 4096)])
        return {"op": op, "Lq": Lq, "Lk": Lk, "Hq": Hkv * rep, "Hkv": Hkv, "mode": mode, "nvalid": Lk, "graph": False}
    if op == "block":
        H = rng.choice([8, 12, 16, 24])
        M = _log(rng, 64, 4096)
        return {"op": op, "enc": rng.choice([Q4, Q8]), "M": M, "K": H * 128, "H": H, "graph": M <= 512}
    if op == "conv3":
        C = rng.choice([64, 96, 128, 256])
        N = rng.choice([64, 128, 256])
        H, W = _log(rng, 12, 92), _log(rng, 12, 160)
        T = min(rng.randint(1, 13), max(1, int(3e9 / (H * W * C * N))))
        return {"op": op, "T": T, "H": H, "W": W, "C": C, "N": N, "pn": rng.random() < 0.5,
                "graph": False}
    H, W = _log(rng, 16, 256), _log(rng, 16, 256)
    stride, up2 = rng.choice([(1, False), (1, False), (2, False), (1, True)])
    return {"op": op, "H": H if not up2 else max(16, H // 2), "W": W, "C": rng.choice([64, 128, 256, 512]),
            "N": rng.choice([64, 128, 256]), "stride": stride, "up2": up2, "graph": False}


# ------------------------------------------------------------------------------------------------------- buffers
class _Memory:
    """One device buffer of the library, given back when its last user is gone; torch sees it as a tensor."""

    def __init__(self, dev, shape, typestr, itemsize):
        self.dev, self.buf = dev, dev.buffer(math.prod(shape) * itemsize)
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (self.buf.ptr, False),
                                         "version": 2, "strides": None}

    def __del__(self):
        self.dev.free(self.buf)


_TYPES = {torch.float32: ("<f4", 4), torch.float16: ("<f2", 2), torch.int32: ("<i4", 4)}


class _State:
    """Buffers by name (`t`: as tensors, `b`: as the library's), the call list and, where captured, its graph."""

    def __init__(self, dev):
        self.dev, self.t, self.b, self.calls, self.graph, self.out = dev, {}, {}, [], None, None

    def new(self, name, shape, dtype):
        m = _Memory(self.dev, shape, *_TYPES[dtype])
        self.b[name], self.t[name] = m.buf, torch.as_tensor(m, device="cuda")
        return self.t[name]

    def put(self, name, value):
        value = value.contiguous()
        self.new(name, value.shape, value.dtype)
        self.dev.done()                          # the buffer's clear is queued on the library's stream
        self.t[name].copy_(value)

    def go(self):
        for c in self.calls:
            c()

    def __del__(self):
        if self.graph is not None:
            self.dev.done()
            self.dev.graph_destroy(self.graph)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


# ------------------------------------------------------------------------------------------------------- weights
def _encode(enc, w):
    """fp32 [rows][K] -> the encoding's bytes as int32 words (or fp16 rows)"""
    rows, K = w.shape
    if enc == F16:
        return w.half()
    if enc == Q4:
        v = w.view(rows // 64, 64, K // 32, 32).transpose(1, 2)                       # tile, group, row, k
        mn = v.amin(-1).half()
        s = ((v.amax(-1) - mn.float()) / 15.0).half()
        s = torch.where(s == 0, torch.ones_like(s), s)
        q = ((v - mn.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, 15).to(torch.int32)
        q = q.view(*q.shape[:3], 4, 8)
        code = q[..., 0].clone()
        for i in range(1, 8):
            code |= q[..., i] << (4 * i)
        sm = torch.stack([s, mn], -1).contiguous().view(torch.int32).squeeze(-1)      # low half scale, high half minimum
        return torch.cat([code.flatten(2), sm], -1)
    v = w.view(rows // 64, 64, K // 64, 64).transpose(1, 2)
    s = (v.abs().amax(-1) / 127.0).half()
    s = torch.where(s == 0, torch.ones_like(s), s)
    q = (v / s.float()[..., None]).round_().clamp_(-128, 127).to(torch.int8).contiguous()
    return torch.cat([q.view(torch.int32).flatten(2), s.contiguous().view(torch.int32)], -1)


def _decode(enc, b, rows, K):
    """the weights the bytes stand for, in 64 bits"""
    if enc == F16:
        return b.double()
    if enc == Q4:
        code, sm = b[..., :256].reshape(*b.shape[:2], 64, 4), b[..., 256:].contiguous().view(torch.float16)
        s, mn = sm[..., 0::2].double(), sm[..., 1::2].double()
        q = torch.stack([(code >> (4 * i)) & 15 for i in range(8)], -1).flatten(3)
        v = q.double() * s[..., None] + mn[..., None]
    else:
        q = b[..., :1024].contiguous().view(torch.int8).view(*b.shape[:2], 64, 64)
        s = b[..., 1024:].contiguous().view(torch.float16)
        v = q.double() * s.double()[..., None]
    return v.transpose(1, 2).reshape(rows, K)


def _rows(enc, n):
    return n if enc == F16 else (n + 63) // 64 * 64


def _weight(s, name, enc, g, n, K, scale):
    s.put(name, _encode(enc, _randn(g, _rows(enc, n), K) * scale))
    return {"enc": enc, "buf": s.b[name], "rows": _rows(enc, n), "cols": K}


def _heads(N):
    """query and key / value heads of a QKV projection of N columns, about four query heads to a key head"""
    h = N // 128
    hkv = max(1, h // 6)
    return h - 2 * hkv, hkv


def _rope(L):
    """a table of rotary angles, theta 10000: [L][64][cos, sin]"""
    a = torch.arange(L, device="cuda")[:, None] * 10000.0 ** (-torch.arange(64, device="cuda") / 64.0)[None, :]
    return torch.stack([a.cos(), a.sin()], -1).float()


def _act_rows(s, g, M, K, mode):
    """fp16 rows, or the fp32 residual with what its norm needs"""
    if mode == "f16":
        s.put("x", _randn(g, M, K).half())
        return
    s.put("x", _randn(g, M, K).half().float())
    s.new("st", (M, 2), torch.float32)
    s.put("pv", 1.0 + 0.1 * _randn(g, K) if mode == "rms" else 0.5 * _randn(g, 2 * K))


def _norm_args(s, x, mode, K):
    a = {"x": {"buf": s.b[x], "mode": mode}}
    if mode != "f16":
        a["stats"] = {"buf": s.b["st"]}
        a["pv"] = {"buf": s.b["pv"], "stride": K if mode == "lnmod" else 0}
    return a


# ------------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    dev = _device()
    s, g = _State(dev), _gen(seed)
    s.case = case
    _PREPARE[case["op"]](s, case, g)
    torch.cuda.synchronize()
    if case["graph"]:
        s.go()                                   # once, so that the library's workspaces have their size
        dev.done()
        dev.graph_begin()
        s.go()
        s.graph = dev.graph_end()
    return s


def _gemm_call(s, a):
    """the call as a program that repeats it makes it: the argument struct is flattened once"""
    args = p0k.gemm_args(a, s.dev.resolve)
    s.calls.append(lambda: s.dev.gemm_raw(args))


def _prepare_linear(s, c, g):
    M, N, K, epi = c["M"], c["N"], c["K"], c["epi"]
    _act_rows(s, g, M, K, c["x"])
    a = {"w": _weight(s, "w", c["enc"], g, N, K, 0.02), "M": M, "N": N, "K": K, "epi": epi}
    a.update(_norm_args(s, "x", c["x"], K))
    no = N // 2 if epi == "swiglu" else N
    if epi == "heads":
        hq, hkv = _heads(N)
        s.new("y", (N // 128, M, 128), torch.float16)
        s.put("ev", 1.0 + 0.1 * _randn(g, 256))
        s.put("rope", _rope(M))
        a["ev"] = {"buf": s.b["ev"]}
        a["heads"] = {"Ltot": M, "Hq": hq, "Hkv": hkv, "rope": {"buf": s.b["rope"]}}
    else:
        s.new("y", (M, no), torch.float32 if epi in ("f32", "resadd") else torch.float16)
    if epi == "swiglu":
        a["wr0"], a["wr1"] = 0, N // 2
    if epi == "bias":
        s.put("ev", 0.5 * _randn(g, N))
        a["ev"] = {"buf": s.b["ev"]}
    if epi == "resadd":
        s.put("res", _randn(g, M, N).half().float())
        n = M * N * 4
        s.calls.append(lambda: s.dev.copy(s.b["y"], 0, s.b["res"], 0, n))
    a["y"] = {"buf": s.b["y"], "ld": 0 if epi == "heads" else no}
    _rowstats_call(s, "x", M, K, c["x"])
    _gemm_call(s, a)
    s.out = {"y": s.t["y"]}


def _rowstats_call(s, x, M, K, mode):
    if mode != "f16":
        s.calls.append(lambda: s.dev.rowstats(s.b[x], M, K, "rms" if mode == "rms" else "ln", 1e-6, s.b["st"]))


def _prepare_mlp(s, c, g):
    M, K, F = c["M"], c["K"], c["F"]
    _act_rows(s, g, M, K, c["x"])
    s.new("h", (M, K), torch.float32)
    s.new("a", (M, F), torch.float16)
    wu, wd = _weight(s, "wu", c["enc"], g, 2 * F, K, 0.02), _weight(s, "wd", c["enc"], g, K, F, 0.02)
    up = {"w": wu, "M": M, "N": 2 * F, "K": K, "epi": "swiglu", "act": c["act"], "wr0": 0, "wr1": F,
          "y": {"buf": s.b["a"], "ld": F}}
    up.update(_norm_args(s, "h", c["x"], K))
    down = {"w": wd, "x": {"buf": s.b["a"]}, "y": {"buf": s.b["h"]}, "M": M, "N": K, "K": F, "epi": "resadd"}
    if c["x"] == "lnmod":
        s.put("ev", 0.5 * _randn(g, K))
        down["ev"] = {"buf": s.b["ev"]}
    n = M * K * 4
    s.calls.append(lambda: s.dev.copy(s.b["h"], 0, s.b["x"], 0, n))
    _rowstats_call(s, "h", M, K, c["x"])
    _gemm_call(s, up)
    _gemm_call(s, down)
    s.out = {"h": s.t["h"]}


def _prepare_attn(s, c, g):
    s.put("q", _randn(g, c["Hq"], c["Lq"], 128).half())
    s.put("k", _randn(g, c["Hkv"], c["Lk"], 128).half())
    s.put("v", _randn(g, c["Hkv"], c["Lk"], 128).half())
    s.new("o", (c["Lq"], c["Hq"] * 128), torch.float16)
    args = p0k.attn_args({"q": {"buf": s.b["q"]}, "k": {"buf": s.b["k"]}, "v": {"buf": s.b["v"]},
                          "o": {"buf": s.b["o"]}, "Lq": c["Lq"], "Lk": c["Lk"], "Hq": c["Hq"], "Hkv": c["Hkv"],
                          "mode": c["mode"], "nvalid": c["nvalid"]}, s.dev.resolve)
    s.calls.append(lambda: s.dev.attention_raw(args))
    s.out = {"o": s.t["o"]}


def _prepare_block(s, c, g):
    M, K, H = c["M"], c["K"], c["H"]
    _act_rows(s, g, M, K, "lnmod")
    s.new("h", (M, K), torch.float32)
    s.new("qkv", (3 * H, M, 128), torch.float16)
    s.new("o", (M, K), torch.float16)
    s.put("nw", 1.0 + 0.1 * _randn(g, 256))
    s.put("rope", _rope(M))
    s.put("gate", 0.5 * _randn(g, K))
    qkv = {"w": _weight(s, "wqkv", c["enc"], g, 3 * K, K, 0.02), "M": M, "N": 3 * K, "K": K, "epi": "heads",
           "y": {"buf": s.b["qkv"]}, "ev": {"buf": s.b["nw"]},
           "heads": {"Ltot": M, "Hq": H, "Hkv": H, "rope": {"buf": s.b["rope"]}}}
    qkv.update(_norm_args(s, "h", "lnmod", K))
    part = H * M * 256
    at = p0k.attn_args({"q": {"buf": s.b["qkv"]}, "k": {"buf": s.b["qkv"], "off": part},
                        "v": {"buf": s.b["qkv"], "off": 2 * part}, "o": {"buf": s.b["o"]}, "Lq": M, "Hq": H},
                       s.dev.resolve)
    proj = {"w": _weight(s, "wo", c["enc"], g, K, K, 0.02), "x": {"buf": s.b["o"]}, "y": {"buf": s.b["h"]}, "M": M,
            "N": K, "K": K, "epi": "resadd", "ev": {"buf": s.b["gate"]}}
    n = M * K * 4
    s.calls.append(lambda: s.dev.copy(s.b["h"], 0, s.b["x"], 0, n))
    _rowstats_call(s, "h", M, K, "lnmod")
    _gemm_call(s, qkv)
    s.calls.append(lambda: s.dev.attention_raw(at))
    _gemm_call(s, proj)
    s.out = {"h": s.t["h"], "qkv": s.t["qkv"]}


def _prepare_conv3(s, c, g):
    T, H, W, C, N = c["T"], c["H"], c["W"], c["C"], c["N"]
    K = 27 * C
    s.put("x", _randn(g, T, H, W, C).half())
    s.new("y", (T, H, W, N), torch.float16)
    s.put("ev", 0.5 * _randn(g, N))
    a = {"w": _weight(s, "w", F16, g, N, K, 0.02), "x": {"buf": s.b["x"]}, "y": {"buf": s.b["y"]}, "M": T * H * W,
         "N": N, "K": K, "epi": "bias", "ev": {"buf": s.b["ev"]},
         "conv": {"kind": "conv3", "Hi": H, "Wi": W, "Ci": C, "Ho": H, "Wo": W, "stride": T, "pn": c["pn"]}}
    if c["pn"]:
        s.new("st", (T * H * W,), torch.float32)
        a["stats"] = {"buf": s.b["st"]}
        s.calls.append(lambda: s.dev.pixstats(s.b["x"], T * H * W, C, s.b["st"]))
    _gemm_call(s, a)
    s.out = {"y": s.t["y"]}


def _conv2d_size(c):
    H, W = (2 * c["H"], 2 * c["W"]) if c["up2"] else (c["H"], c["W"])
    return (H - 1) // c["stride"] + 1, (W - 1) // c["stride"] + 1


def _prepare_conv2d(s, c, g):
    H, W, C, N = c["H"], c["W"], c["C"], c["N"]
    Ho, Wo = _conv2d_size(c)
    K = 9 * C
    s.put("x", _randn(g, H, W, C).half())
    s.new("y", (Ho, Wo, N), torch.float16)
    s.put("ev", 0.5 * _randn(g, N))
    s.put("gb", torch.cat([1.0 + 0.2 * _randn(g, C), 0.3 * _randn(g, C)]))
    s.new("part", ((H * W + 63) // 64 * 128,), torch.float32)
    s.new("ab", (2 * C,), torch.float32)
    a = {"w": _weight(s, "w", F16, g, N, K, 0.02), "x": {"buf": s.b["x"]}, "y": {"buf": s.b["y"]}, "M": Ho * Wo,
         "N": N, "K": K, "epi": "bias", "ev": {"buf": s.b["ev"]}, "pv": {"buf": s.b["ab"], "stride": C},
         "conv": {"kind": "conv", "Hi": H, "Wi": W, "Ci": C, "Ho": Ho, "Wo": Wo, "stride": c["stride"], "padT": 1,
                  "padL": 1, "ks": 3, "up2": c["up2"], "gn": True}}
    s.calls.append(lambda: s.dev.groupnorm_stats(s.b["x"], H * W, C, s.b["part"], s.b["gb"], 0, 4 * C, s.b["ab"]))
    _gemm_call(s, a)
    s.out = {"y": s.t["y"]}


_PREPARE = {"linear": _prepare_linear, "mlp": _prepare_mlp, "attn": _prepare_attn, "block": _prepare_block,
            "conv3": _prepare_conv3, "conv2d": _prepare_conv2d}


def run(state):
    if state.graph is not None:
        state.dev.graph_launch(state.graph)
    else:
        state.go()
    return state.out


# ------------------------------------------------------------------------------------------------------- work
def _wbytes(enc, n, K):
    return {Q4: 5 / 8, Q8: 1.03125, F16: 2}[enc] * _rows(enc, n) * K


def work(case):
    c, op = case, case["op"]
    if op == "linear":
        M, N, K, epi = c["M"], c["N"], c["K"], c["epi"]
        no = N // 2 if epi == "swiglu" else N
        b = _wbytes(c["enc"], N, K) + M * K * (2 if c["x"] == "f16" else 4)
        b += M * no * {"f32": 4, "resadd": 8}.get(epi, 2)
        return {"bytes": b, "flops": 2 * M * N * K}
    if op == "mlp":
        M, K, F = c["M"], c["K"], c["F"]
        return {"bytes": _wbytes(c["enc"], 2 * F, K) + _wbytes(c["enc"], K, F) + 8 * M * K, "flops": 6 * M * F * K}
    if op == "attn":
        pairs = c["Lq"] * (c["nvalid"] if c["mode"] == 2 else c["Lk"])
        if c["mode"] == 1:
            pairs = c["Lq"] * (c["Lq"] + 1) // 2
        keys = c["nvalid"] if c["mode"] == 2 else c["Lk"]
        return {"bytes": 512 * (c["Hq"] * c["Lq"] + c["Hkv"] * keys), "flops": 512 * c["Hq"] * pairs}
    if op == "block":
        M, K = c["M"], c["K"]
        return {"bytes": _wbytes(c["enc"], 4 * K, K) + 8 * M * K + 6 * M * K, "flops": 8 * M * K * K + 4 * M * M * K}
    if op == "conv3":
        v = c["T"] * c["H"] * c["W"]
        return {"bytes": 2 * v * (c["C"] + c["N"]) + 54 * c["C"] * c["N"], "flops": 54 * v * c["C"] * c["N"]}
    Ho, Wo = _conv2d_size(c)
    return {"bytes": 2 * (c["H"] * c["W"] * c["C"] + Ho * Wo * c["N"]) + 18 * c["C"] * c["N"],
            "flops": 18 * Ho * Wo * c["C"] * c["N"]}


def tolerance(case):
    # Measured between kernels, tiles and K splits of the library: 1e-5 where only the order of fp32 sums changes (a
    # prologue's or a result's fp16 rounding then tips here and there). Quantised weights may be rounded to fp16 or
    # kept in fp32 (both are right): 1.5e-4 apart. Attention's probabilities are fp16 beside a row maximum that depends
    # on the order of the keys: 3e-4 apart.
    if case["op"] in ("attn", "block"):
        return {"rel": 1.2e-3}
    if case["op"] == "mlp" or (case["op"] == "linear" and case["enc"] != F16):
        return {"rel": 6e-4}
    return {"rel": 1e-4}


# ------------------------------------------------------------------------------------------------------- exact
def _norm64(s, x, mode, K):
    if mode == "f16":
        return x
    pv = s.t["pv"].double()
    if mode == "rms":
        return x * (x.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * pv
    d = x - x.mean(-1, keepdim=True)
    return d * (d.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (1 + pv[:K]) + pv[K:]


def _glu64(y, act):
    a, b = y.chunk(2, -1)
    if act == "silu":
        return a * torch.sigmoid(a) * b
    return a * torch.sigmoid(2 * 0.7978845608 * (a + 0.044715 * a ** 3)) * b


def _heads64(y, hq, hkv, nw, rope):
    """[M][heads * 128] -> head-major with norm + RoPE (interleaved pairs) on the query and key heads"""
    M = y.shape[0]
    y = y.view(M, -1, 128).transpose(0, 1)
    n = y * (y.square().mean(-1, keepdim=True) + 1e-6).rsqrt()
    nw, rope = nw.double(), rope.double()
    n = torch.cat([n[:hq] * nw[:128], n[hq:] * nw[128:]])
    cs, sn = rope[..., 0], rope[..., 1]
    e, o = n[..., 0::2], n[..., 1::2]
    r = torch.stack([e * cs - o * sn, e * sn + o * cs], -1).flatten(2)
    return torch.cat([r[:hq + hkv], y[hq + hkv:]])


def _attn64(q, k, v, mode, nvalid):
    """[H][L][128] each -> [Lq][Hq * 128], a head at a time"""
    hq, lq = q.shape[:2]
    lk, rep = k.shape[1], q.shape[0] // k.shape[0]
    j = torch.arange(lk, device="cuda")
    see = None
    if mode == 1:
        see = j[None, :] <= torch.arange(lq, device="cuda")[:, None].clamp(max=nvalid - 1)
    elif mode == 2:
        see = (j < nvalid)[None, :]
    out = []
    for h in range(hq):
        p = q[h] @ k[h // rep].t().contiguous() / math.sqrt(128.0)
        if see is not None:
            p = p.masked_fill(~see, -math.inf)
        out.append(torch.softmax(p, -1) @ v[h // rep])
    return torch.cat(out, -1)


def _conv64(x, w, offsets, size, stride):
    """sum over taps of x shifted by the tap (x padded so that every shift is inside) times the tap's weights"""
    C = x.shape[-1]
    y = 0
    for i, o in enumerate(offsets):
        v = x
        for d, (at, n) in enumerate(zip(o, size)):
            v = v.narrow(d, at, (n - 1) * stride[d] + 1)
        v = v[tuple(slice(None, None, st) for st in stride)]
        y = y + (v.reshape(-1, C) @ w[:, i * C:(i + 1) * C].t().contiguous())
    return y.view(*size, -1)


def exact(case, seed):
    c, op = dict(case, graph=False), case["op"]
    s = prepare(c, seed)
    t = s.t
    if op == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        y = _norm64(s, t["x"].double(), c["x"], K) @ _decode(c["enc"], t["w"], _rows(c["enc"], N), K)[:N].t().contiguous()
        if c["epi"] == "swiglu":
            y = _glu64(y, "silu")
        elif c["epi"] == "bias":
            y = y + t["ev"].double()
        elif c["epi"] == "resadd":
            y = y + t["res"].double()
        elif c["epi"] == "heads":
            y = _heads64(y, *_heads(N), t["ev"], t["rope"])
        return {"y": y}
    if op == "mlp":
        M, K, F = c["M"], c["K"], c["F"]
        x = t["x"].double()
        y = _glu64(_norm64(s, x, c["x"], K) @ _decode(c["enc"], t["wu"], 2 * F, K).t().contiguous(), c["act"])
        y = y @ _decode(c["enc"], t["wd"], K, F).t().contiguous()
        return {"h": x + (y * t["ev"].double() if c["x"] == "lnmod" else y)}
    if op == "attn":
        return {"o": _attn64(t["q"].double(), t["k"].double(), t["v"].double(), c["mode"], c["nvalid"])}
    if op == "block":
        M, K, H = c["M"], c["K"], c["H"]
        x = t["x"].double()
        y = _norm64(s, x, "lnmod", K) @ _decode(c["enc"], t["wqkv"], 3 * K, K).t().contiguous()
        qkv = _heads64(y, H, H, t["nw"], t["rope"])
        o = _attn64(qkv[:H], qkv[H:2 * H], qkv[2 * H:], 0, M)
        o = o @ _decode(c["enc"], t["wo"], K, K).t().contiguous()
        return {"h": x + t["gate"].double() * o, "qkv": qkv}
    if op == "conv3":
        T, H, W = c["T"], c["H"], c["W"]
        x = t["x"].double()
        if c["pn"]:
            x = x * (x.square().mean(-1, keepdim=True) + 1e-8).rsqrt()
            x = x * torch.sigmoid(x)
        x = torch.cat([x[:1], x, x[-1:]])                                   # time repeats its ends, space is zero
        x = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        taps = [(a, b, d) for a in range(3) for b in range(3) for d in range(3)]
        return {"y": _conv64(x, t["w"].double(), taps, (T, H, W), (1, 1, 1)) + t["ev"].double()}
    C = c["C"]
    x = t["x"].double()
    v = x.view(-1, 32, C // 32)
    mean = v.mean((0, 2), keepdim=True)
    x = ((v - mean) * ((v - mean).square().mean((0, 2), keepdim=True) + 1e-6).rsqrt()).view(x.shape)
    gb = t["gb"].double()
    x = x * gb[:C] + gb[C:]
    x = x * torch.sigmoid(x)
    if c["up2"]:
        x = x.repeat_interleave(2, 0).repeat_interleave(2, 1)
    st = c["stride"]
    x = torch.nn.functional.pad(x, (0, 0, 1, 1 + st, 1, 1 + st))
    y = _conv64(x, t["w"].double(), [(a, b) for a in range(3) for b in range(3)], _conv2d_size(c), (st, st))
    return {"y": y + t["ev"].double()}
