"""Performance cases of the decode path: what a program that runs SSF, GPTQ or
AWQ weights through this library spends its time on.

The single layers and blocks come first (a product with its activation
quantization, a feed-forward block, the vocabulary head with the greedy pick,
decode and prompt attention, the batched products, a mixture-of-experts layer,
the re-quantization of a copy), then whole calls of the decoder (a step, a
prompt, a step of several sequences) on a few layers of the Llama-3-8B and
Qwen2.5-1.5B shapes. Weights are synthetic. Device buffers are torch tensors,
handed to the library as plain device pointers.

A case is a dict of plain values; "kind" says which path it takes.
"""
import hashlib
import math
import os
import tempfile

import numpy as np
import torch

import sheep_amd as sa
from sheep_amd import gptq, ingest

DEV = "cuda"
EPS = 1e-5

# the decoder shapes of the benchmark; the layer count is the case's
SHAPES = {
    "llama": dict(n_embd=4096, n_head=32, n_head_kv=8, n_ff=14336, n_vocab=128256, rope_theta=5e5, rms_eps=1e-5),
    "qwen": dict(n_embd=1536, n_head=12, n_head_kv=2, n_ff=8960, n_vocab=151936, rope_theta=1e6, rms_eps=1e-6,
                 qkv_bias=True),
}
N_CTX = 4096


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest product of a decode step (the attention output of the
        # 1.5B shape): two launches, all latency
        dict(name="gemv_q4_1536x1536", kind="gemv", rows=1536, cols=1536, bits=4, norm=False),
        # a dense feed-forward block at batch 1, the bulk of a decode step's
        # weight bytes
        dict(name="ffn_decode_q4_4096x14336", kind="ffn", cols=4096, ff=14336, bits=4, perm=False),
        # the vocabulary head at 8 bits and the greedy pick
        dict(name="head_q8_151936x1536", kind="head", rows=151936, cols=1536, bits=8),
        # a GPTQ file's matrix used as it is
        dict(name="gptq_gemv_14336x4096", kind="gptq", rows=14336, cols=4096, act_order=False),
        # attention of one decode step at the end of a 4096-position context
        dict(name="attn_decode_32x8_at_4095", kind="attn", heads=32, kv=8, n_ctx=4096, pos=4095),
        # attention of a prompt chunk behind a prefix, a ragged row count
        dict(name="attn_prompt_509_at_1531", kind="attn_prompt", heads=32, kv=8, n_ctx=4096, pos=1531, n=509),
        # the feed-forward products of a prompt chunk on the matrix cores
        dict(name="ffn_rows_q4_509", kind="ffn_rows", cols=4096, ff=14336, bits=4, n=509, per256=True),
        # a mixture-of-experts layer for 16 sequences
        dict(name="moe_8x14336_16_tokens", kind="moe", cols=4096, ff=14336, experts=8, used=2, n=16, per256=True),
        # the encode direction: a float tensor into 4-bit planes and fields
        dict(name="requant_q4_4096x14336", kind="requant", rows=4096, cols=14336, bits=4),
        # one decode step near the end of the context, logits on the host
        dict(name="step_llama_at_3968", kind="step", model="llama", layers=4, bits=4, exact=False, pos=3968),
        # a prompt as the server reads it by default
        dict(name="prompt_llama_1021", kind="prompt", model="llama", layers=4, bits=4, level=1, exact=False, pos=0,
             n=1021),
        # one step of 16 sequences at about a thousand positions
        dict(name="batch_llama_16_at_1024", kind="batch", model="llama", layers=4, bits=4, pos=1024, n=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "ffn", "head", "gptq", "attn", "attn_prompt", "ffn_rows", "ffn_rows", "moe",
                       "requant", "step", "prompt", "prompt", "batch"])
    bits = rng.choice([2, 3, 4, 4, 4, 4, 5, 6, 8])
    heads, kv = rng.choice([(32, 8), (12, 2), (16, 8), (8, 8), (28, 4)])
    if kind == "gemv":
        return dict(kind=kind, rows=_log(rng, 257, 20001), cols=128 * _log(rng, 8, 112), bits=bits,
                    norm=rng.random() < 0.5)
    if kind == "ffn":
        return dict(kind=kind, cols=128 * _log(rng, 6, 32), ff=128 * _log(rng, 16, 112), bits=rng.choice([4, 4, 6, 8]),
                    perm=rng.random() < 0.5)
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 30001, 151936), cols=128 * _log(rng, 8, 24), bits=rng.choice([4, 6, 8]))
    if kind == "gptq":
        return dict(kind=kind, rows=8 * _log(rng, 64, 1792), cols=128 * _log(rng, 8, 112), act_order=rng.random() < 0.5)
    if kind == "attn":
        return dict(kind=kind, heads=heads, kv=kv, n_ctx=4096, pos=_log(rng, 30, 4095))
    if kind == "attn_prompt":
        n = _log(rng, 17, 512)
        return dict(kind=kind, heads=heads, kv=kv, n_ctx=4096, pos=rng.randrange(0, 4096 - n), n=n)
    if kind == "ffn_rows":
        per256 = rng.random() < 0.7
        return dict(kind=kind, cols=256 * _log(rng, 4, 16), ff=256 * _log(rng, 8, 56), bits=rng.choice([4, 4, 4, 6, 8]),
                    n=_log(rng, 2, 512 if per256 else 64), per256=per256)
    if kind == "moe":
        small = rng.random() < 0.5
        return dict(kind=kind, cols=1024 if small else 4096, ff=3584 if small else 14336, experts=16 if small else 8,
                    used=4 if small else 2, n=rng.randint(1, 16), per256=rng.random() < 0.5)
    if kind == "requant":
        return dict(kind=kind, rows=_log(rng, 257, 4096), cols=256 * _log(rng, 4, 56), bits=bits)
    model = rng.choice(["llama", "qwen"])
    if kind == "step":
        return dict(kind=kind, model=model, layers=rng.randint(2, 4), bits=4, exact=rng.random() < 0.4,
                    pos=_log(rng, 40, 4000))
    if kind == "prompt":
        exact = rng.random() < 0.3
        return dict(kind=kind, model=model, layers=2, bits=rng.choice([4, 4, 8]), exact=exact,
                    level=1 if exact else rng.choice([1, 2]), pos=rng.choice([0, 0, rng.randint(1, 1000)]),
                    n=_log(rng, 20, 1000))
    return dict(kind=kind, model=model, layers=rng.randint(2, 4), bits=4, pos=_log(rng, 40, 2000), n=rng.randint(2, 16))


# ---------------------------------------------------------------- inputs

class Buf:
    """A torch tensor as one of the library's device buffers."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


class Act:
    def __init__(self, q, scale, sums):
        self.q, self.scale, self.sums, self.n = Buf(q), Buf(scale), Buf(sums), q.shape[-1]


def _gen(seed, salt):
    h = hashlib.sha256(f"{seed}:{salt}".encode()).digest()
    return torch.Generator(device=DEV).manual_seed(int.from_bytes(h[:7], "little"))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEV)


def _act(n, rows=None):
    sh = () if rows is None else (rows,)
    return Act(_empty(*sh, n, dtype=torch.int8), _empty(*sh, n // 32), _empty(*sh, n // 32, dtype=torch.int32))


# the planes of a width in storage order: (bits, the code bit they start at)
PLANES = {2: [(2, 0)], 3: [(2, 0), (1, 2)], 4: [(4, 0)], 5: [(4, 0), (1, 4)], 6: [(2, 4), (4, 0)],
          7: [(4, 0), (2, 4), (1, 6)], 8: [(4, 0), (4, 4)]}


def _pack(codes, b):
    """Codes [rows][cols] of b bits as the file's plane of that width, uint8 [rows][cols * b / 8]."""
    r, n = codes.shape
    c = codes.view(r, n // 128, 4, 32)
    if b == 4:
        return torch.stack([c[:, :, 0] | c[:, :, 1] << 4, c[:, :, 2] | c[:, :, 3] << 4], 2).reshape(r, -1)
    if b == 2:
        return (c[:, :, 0] | c[:, :, 1] << 2 | c[:, :, 2] << 4 | c[:, :, 3] << 6).reshape(r, -1)
    w = (1 << torch.arange(8, device=codes.device, dtype=torch.int32)).to(torch.uint8)
    return (codes.view(r, n // 8, 8) * w).sum(-1, dtype=torch.uint8)


class Weights:
    """A quantized matrix of uniform codes and mean-zero weights of variance about 1 / cols."""

    def __init__(self, g, rows, cols, bits, upload=True):
        ng, ns = cols // 32, (cols + 255) // 256
        self.rows, self.cols, self.bits = rows, cols, bits
        self.codes = torch.randint(0, 1 << bits, (rows, cols), generator=g, device=DEV, dtype=torch.uint8)
        self.sq = torch.randint(96, 256, (rows, ng), generator=g, device=DEV, dtype=torch.uint8)
        step = math.sqrt(12.0) / (1 << bits) / math.sqrt(cols) / 180.0
        self.sd = (step * (0.75 + 0.5 * torch.rand(rows, ns, generator=g, device=DEV))).half()
        # the group's min is -(2^bits - 1) / 2 of its steps
        self.md = (self.sd.float() * ((1 << bits) - 1) / 2 * 2).half()
        self.mq = (127.0 - self.sq.float() / 2).round().clamp(0, 255).to(torch.uint8)
        self.mat = self.upload() if upload else None
        if upload:
            del self.codes, self.sq, self.mq, self.sd, self.md

    def upload(self):
        planes = [_pack((self.codes >> sh) & ((1 << b) - 1), b).cpu().numpy() for b, sh in PLANES[self.bits]]
        ptrs = (sa.c_void_p * 4)(*([p.ctypes.data for p in planes] + [None] * (4 - len(planes))))
        f = [t.cpu().contiguous().numpy() for t in (self.sd, self.sq, self.md, self.mq)]
        return sa.Mat(sa.lib().sml_hip_mat_upload(ptrs, f[0].ctypes.data, f[1].ctypes.data, f[2].ctypes.data,
                                                  f[3].ctypes.data, self.rows, self.cols, self.bits, 0, 0))

    def dense(self):
        ng = self.cols // 32
        sup = torch.arange(ng, device=DEV) // 8
        step = self.sd.double()[:, sup] * self.sq.double()
        low = self.md.double()[:, sup] * (self.mq.double() - 127)
        w = self.codes.view(self.rows, ng, 32).double() * step[:, :, None] + low[:, :, None]
        return w.view(self.rows, self.cols)


def _quant64(x, width):
    """The int8 quantization of x [..., n] per `width` values, in 64 bits: codes and scales per group of 32."""
    v = x.reshape(*x.shape[:-1], -1, width) if x.shape[-1] % width == 0 else None
    if v is None:
        pad = -x.shape[-1] % width
        v = torch.nn.functional.pad(x, (0, pad)).reshape(*x.shape[:-1], -1, width)
    s = v.abs().amax(-1, keepdim=True) / 127.0
    q = torch.where(s > 0, (v / s.clamp_min(1e-300)).round().clamp(-127, 127), torch.zeros_like(v))
    n = x.shape[-1]
    codes = q.reshape(*x.shape[:-1], -1)[..., :n]
    scale = s.expand(*s.shape[:-1], width // 32).reshape(*x.shape[:-1], -1)[..., : n // 32]
    return codes, scale


def _deq(codes, scale):
    return (codes.view(*scale.shape, 32) * scale[..., None]).reshape(codes.shape)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu64(g):
    return g / (1 + torch.exp(-g))


def _x(g, n):
    """A residual-stream row: normal values with a few large channels."""
    x = _randn(g, n)
    x[:: max(1, n // 6)] *= 8.0
    return x


def _rope(theta, half, n_ctx):
    f = theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    a = torch.arange(n_ctx, device=DEV, dtype=torch.float64)[:, None] * f
    return torch.cos(a).float(), torch.sin(a).float()


def _rotate64(x, c, s):
    """Halved-pair rotation of x [..., hd] by c, s [..., hd / 2]."""
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


# ---------------------------------------------------------------- decoders

_OPEN = {"key": None, "dec": None}


def _file(tag, write):
    """A synthetic model file by content tag, written once per machine."""
    path = os.path.join(tempfile.gettempdir(), f"sml_perf_{hashlib.sha256(tag.encode()).hexdigest()[:16]}.ssf")
    if not os.path.exists(path):
        tmp = f"{path}.{os.getpid()}"
        write(tmp)
        os.replace(tmp, path)
    return path


def _model_file(case):
    spec = dict(SHAPES[case["model"]], n_layer=case["layers"], nbits=case["bits"], seed=41, n_ctx_train=N_CTX)
    return _file(repr(sorted(spec.items())), lambda p: sa.synth_model(p, **spec))


def _ids(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


def _decoder(case):
    """The open decoder of this case (one per process), its caches holding the same prefix for every seed."""
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if _OPEN["key"] == key:
        return _OPEN["dec"]
    _OPEN["key"] = None
    d = sa.Decoder(_model_file(case), n_ctx=N_CTX, exact=case.get("exact", False))
    V = SHAPES[case["model"]]["n_vocab"]
    d.prompt_mode(2)
    if case["kind"] == "batch":
        d.slots(case["n"])
        for b, p in enumerate(_batch_pos(case)):
            if p:
                d.prefill_slot(b, _ids(900 + b, p, V), 0, V)
    elif case["pos"]:
        d.prefill(_ids(900, case["pos"], V), 0, V)
    d.prompt_mode(case.get("level", 1))
    _OPEN.update(key=key, dec=d)
    return d


def _batch_pos(case):
    return [max(1, case["pos"] - 13 * b) for b in range(case["n"])]


_MOE = {"key": None, "moe": None}


def _moe(case):
    spec = dict(n_layer=1, n_embd=case["cols"], n_head=32, n_head_kv=8, n_ff=case["ff"], n_vocab=1024,
                n_expert=case["experts"], n_expert_used=case["used"], moe_flags=1, rope_theta=1e6, seed=1005)
    key = repr(sorted(spec.items()))
    if _MOE["key"] != key:
        if _MOE["moe"]:
            _MOE["moe"].free()
        _MOE.update(key=None, moe=None)
        _MOE["moe"] = sa.MoE(_file(key, lambda p: sa.synth_model(p, **spec)), 0, 16)
        _MOE["key"] = key
    _MOE["moe"].regime(case["per256"])
    return _MOE["moe"]


# ---------------------------------------------------------------- prepare

def _gptq_arrays(case, seed):
    g = _gen(seed, "gptq")
    rows, cols = case["rows"], case["cols"]
    qweight = torch.randint(-(1 << 31), 1 << 31, (cols // 8, rows), generator=g, device=DEV, dtype=torch.int64).int()
    qzeros = torch.randint(-(1 << 31), 1 << 31, (cols // 128, rows // 8), generator=g, device=DEV, dtype=torch.int64)
    qzeros = ((qzeros & 0x11111111) + 0x77777777).int()         # zero points 8 and 9, stored less one
    scales = (0.3 / math.sqrt(cols) * (0.5 + torch.rand(cols // 128, rows, generator=g, device=DEV))).half()
    gidx = None
    if case["act_order"]:
        gidx = (torch.randperm(cols, generator=g, device=DEV) // 128).int()
    return qweight, qzeros, scales, gidx, _randn(g, cols)


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed, kind)
    s = dict(case=case, kind=kind)
    if kind in ("gemv", "head"):
        s["m"] = Weights(g, case["rows"], case["cols"], case["bits"]).mat
        s["x"] = Buf(_x(g, case["cols"]))
        s["w"] = Buf(1 + 0.1 * _randn(g, case["cols"])) if kind == "head" or case["norm"] else None
        s["act"], s["y"] = _act(case["cols"]), Buf(_empty(case["rows"]))
        s["tok"] = Buf(_empty(1, dtype=torch.int32))
    elif kind == "ffn":
        s["gate"], s["up"] = (Weights(g, case["ff"], case["cols"], case["bits"]).mat for _ in range(2))
        s["down"] = Weights(g, case["cols"], case["ff"], case["bits"]).mat
        s["x"], s["w"] = Buf(_x(g, case["cols"])), Buf(1 + 0.1 * _randn(g, case["cols"]))
        s["perm"] = Buf(torch.randperm(case["cols"], generator=g, device=DEV).int()) if case["perm"] else None
        s["h"], s["hact"], s["y"] = Buf(_empty(case["ff"])), _act(case["ff"]), Buf(_empty(case["cols"]))
    elif kind == "gptq":
        qw, qz, sc, gi, x = _gptq_arrays(case, seed)
        s["m"] = gptq.GptqMat(qw.cpu().numpy(), qz.cpu().numpy(), sc.cpu().numpy(), case["rows"], case["cols"],
                              g_idx=None if gi is None else gi.cpu().numpy())
        s["x"], s["y"] = Buf(x), Buf(_empty(case["rows"]))
    elif kind in ("attn", "attn_prompt"):
        H, KV, n_ctx, hd = case["heads"], case["kv"], case["n_ctx"], 128
        n = case.get("n", 1)
        s["qkv"] = _randn(g, n, (H + 2 * KV) * hd)
        s["kc"], s["vc"] = _randn(g, n_ctx, KV * hd).half(), _randn(g, n_ctx, KV * hd).half()
        s["cos"], s["sin"] = _rope(5e5, hd // 2, n_ctx)
        s["pos"] = torch.tensor([case["pos"]], dtype=torch.int32, device=DEV)
        nf = sa.lib().sml_hip_attn_part_floats(H, hd, n_ctx)
        s["part"] = _empty(max(nf, n * H * ((n_ctx + 127) // 128) * (hd + 2)))
        s["out"], s["oact"] = _empty(n, H * hd), _act(H * hd)
    elif kind == "ffn_rows":
        s["gate"], s["up"] = (Weights(g, case["ff"], case["cols"], case["bits"]).mat for _ in range(2))
        s["down"] = Weights(g, case["cols"], case["ff"], case["bits"]).mat
        for k, n in (("a", case["cols"]), ("b", case["ff"])):
            q, sc = _quant64(_randn(g, case["n"], n).double(), 256 if case["per256"] else 32)
            s[k] = Act(q.to(torch.int8), sc.float(), q.view(case["n"], -1, 32).sum(-1).int())
        s["h"], s["y"] = Buf(_empty(case["n"], case["ff"])), Buf(_empty(case["n"], case["cols"]))
    elif kind == "moe":
        s["moe"] = _moe(case)
        n, k = case["n"], case["used"]
        s["x"], s["out"] = Buf(_randn(g, n, case["cols"])), Buf(_empty(n, case["cols"]))
        s["sel"], s["w"] = Buf(_empty(n, k, dtype=torch.int32)), Buf(_empty(n, k))
        s["logits"] = Buf(_empty(n, case["experts"]))
    elif kind == "requant":
        rows, cols = case["rows"], case["cols"]
        # columns of different sizes, as a layer's inputs have
        s["x"] = Buf(_randn(g, rows, cols) * (0.02 * torch.exp(0.3 * _randn(g, cols))))
        s["planes"] = [_empty(rows, cols * b // 8, dtype=torch.uint8) for b, _ in PLANES[case["bits"]]]
        s["sd"], s["md"] = (_empty(rows, cols // 256, dtype=torch.int16) for _ in range(2))
        s["sq"], s["mq"] = (_empty(rows, cols // 32, dtype=torch.uint8) for _ in range(2))
        s["perm"] = _empty(cols, dtype=torch.int32)
    else:
        V = SHAPES[case["model"]]["n_vocab"]
        s["dec"], s["V"] = _decoder(case), V
        n = case["n"] if kind in ("prompt", "batch") else 1
        s["ids"] = _ids(seed, n, V)
    return s


# ---------------------------------------------------------------- run

def run(s):
    kind, case = s["kind"], s["case"]
    if kind in ("gemv", "head"):
        sa.normq(s["x"], s["act"], w=s["w"], eps=EPS)
        sa.matvec(s["m"], s["act"], s["y"])
        if kind == "gemv":
            return {"y": s["y"].t}
        sa._chk(sa.lib().sml_hip_argmax(s["y"].ptr, case["rows"], s["tok"].ptr), "argmax")
        return {"y": s["y"].t, "tok": s["tok"].t}
    if kind == "ffn":
        sa.matvec_swiglu_fused(s["gate"], s["up"], s["h"], x=s["x"], w=s["w"], perm=s["perm"], eps=EPS, hact=s["hact"])
        sa.matvec(s["down"], s["hact"], s["y"])
        return {"h": s["h"].t, "y": s["y"].t}
    if kind == "gptq":
        s["m"].matvec(s["x"], s["y"])
        return {"y": s["y"].t}
    if kind == "attn":
        H, KV, hd = case["heads"], case["kv"], 128
        q = s["qkv"].data_ptr()
        o = s["oact"]
        sa._chk(sa.lib().sml_hip_attention_q(
            q, q + H * hd * 4, q + (H + KV) * hd * 4, s["kc"].data_ptr(), s["vc"].data_ptr(), s["cos"].data_ptr(),
            s["sin"].data_ptr(), s["pos"].data_ptr(), H, KV, hd, case["n_ctx"], s["part"].data_ptr(),
            s["out"].data_ptr(), o.q.ptr, o.scale.ptr, o.sums.ptr), "attention")
        p = case["pos"]
        return {"out": s["out"], "codes": o.q.t, "scale": o.scale.t, "k": s["kc"][p], "v": s["vc"][p]}
    if kind == "attn_prompt":
        p, n = case["pos"], case["n"]
        sa._chk(sa.lib().sml_hip_attention_prompt(
            s["qkv"].data_ptr(), n, p, s["kc"].data_ptr(), s["vc"].data_ptr(), s["cos"].data_ptr(),
            s["sin"].data_ptr(), case["heads"], case["kv"], 128, case["n_ctx"], s["part"].data_ptr(),
            s["out"].data_ptr()), "prompt attention")
        return {"out": s["out"], "k": s["kc"][p:p + n], "v": s["vc"][p:p + n]}
    if kind == "ffn_rows":
        a, b, n = s["a"], s["b"], case["n"]
        sa.gemm_swiglu(s["gate"], s["up"], a.q, a.scale, a.sums, n, s["h"], per256=case["per256"])
        sa.gemm(s["down"], b.q, b.scale, b.sums, n, s["y"], per256=case["per256"])
        return {"h": s["h"].t, "y": s["y"].t}
    if kind == "moe":
        s["moe"].ffn(s["x"], case["n"], s["out"], sel=s["sel"], w=s["w"], logits=s["logits"])
        return {"out": s["out"].t, "sel": s["sel"].t, "w": s["w"].t, "logits": s["logits"].t}
    if kind == "requant":
        pl = (sa.c_void_p * 3)(*([p.data_ptr() for p in s["planes"]] + [None] * (3 - len(s["planes"]))))
        sa._chk(ingest._lib().sml_hip_requant(
            s["x"].ptr, case["rows"], case["cols"], case["bits"], None, None, 2, pl, s["sd"].data_ptr(),
            s["sq"].data_ptr(), s["md"].data_ptr(), s["mq"].data_ptr(), s["perm"].data_ptr(), None), "requant")
        return {k: s[k] for k in ("planes", "sd", "sq", "md", "mq", "perm")}
    d, ids, V = s["dec"], s["ids"], s["V"]
    if kind == "step":
        return {"logits": d.step(int(ids[0]), case["pos"], V)}
    if kind == "prompt":
        return {"logits": d.prefill(ids, case["pos"], V)}
    return {"logits": d.step_multi(ids, _batch_pos(case), list(range(case["n"])), V)}


# ---------------------------------------------------------------- work and tolerance

def _mat_bytes(rows, cols, bits):
    return rows * cols * bits / 8 + rows * (cols // 32) * 2 + rows * ((cols + 255) // 256) * 4


def _act_bytes(n):
    return n + n // 32 * 8


def _model_work(case, rows, keys, heads):
    """`rows` positions through the layers, attending to `keys` positions in all; logits of `heads` of them."""
    p = SHAPES[case["model"]]
    E, F, V, hd = p["n_embd"], p["n_ff"], p["n_vocab"], 128
    kvd, L, b = p["n_head_kv"] * hd, case["layers"], case["bits"]
    shapes = [(p["n_head"] * hd + 2 * kvd, E), (E, p["n_head"] * hd), (2 * F, E), (E, F)]
    weights = L * sum(_mat_bytes(r, c, b) for r, c in shapes) + _mat_bytes(V, E, b)
    flops = 2 * rows * L * sum(r * c for r, c in shapes) + 2 * heads * V * E + 4 * L * p["n_head"] * hd * keys
    return dict(weights=weights, flops=flops, kv=L * 2 * kvd * 2, out=heads * V * 4)


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "head"):
        r, c = case["rows"], case["cols"]
        return {"bytes": _mat_bytes(r, c, case["bits"]) + 8 * c + 4 * r, "flops": 2 * r * c}
    if kind == "ffn":
        c, f, b = case["cols"], case["ff"], case["bits"]
        return {"bytes": 2 * _mat_bytes(f, c, b) + _mat_bytes(c, f, b) + 12 * c + 4 * f, "flops": 6 * c * f}
    if kind == "gptq":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * c / 2 + c / 128 * r * 2.5 + 4 * (r + c), "flops": 2 * r * c}
    if kind in ("attn", "attn_prompt"):
        H, KV, p, n = case["heads"], case["kv"], case["pos"], case.get("n", 1)
        keys = n * p + n * (n + 1) // 2
        io = n * ((H + 2 * KV) * 128 * 4 + H * 128 * 4)
        return {"bytes": 2 * (p + n) * KV * 128 * 2 + io, "flops": 4 * 128 * H * keys}
    if kind == "ffn_rows":
        c, f, b, n = case["cols"], case["ff"], case["bits"], case["n"]
        return {"bytes": 2 * _mat_bytes(f, c, b) + _mat_bytes(c, f, b) + n * (_act_bytes(c) + _act_bytes(f) + 4 * (c + f)),
                "flops": 6 * c * f * n}
    if kind == "moe":
        c, f, n, E, k = case["cols"], case["ff"], case["n"], case["experts"], case["used"]
        touched = E * (1 - (1 - k / E) ** n)                    # experts some token chose, on average
        return {"bytes": touched * (2 * _mat_bytes(f, c, 4) + _mat_bytes(c, f, 4)) + E * c * 4 + 8 * n * c,
                "flops": 6 * c * f * n * k + 2 * n * c * E}
    if kind == "requant":
        r, c = case["rows"], case["cols"]
        # 20 ranges, each fitted 3 times, about 10 operations a weight
        return {"bytes": 4 * r * c + _mat_bytes(r, c, case["bits"]), "flops": 20 * 4 * 10 * r * c}
    if kind == "step":
        w = _model_work(case, 1, case["pos"] + 1, 1)
        return {"bytes": w["weights"] + w["kv"] * (case["pos"] + 1) + w["out"], "flops": w["flops"]}
    if kind == "prompt":
        p, n = case["pos"], case["n"]
        w = _model_work(case, n, n * p + n * (n + 1) // 2, 1)
        return {"bytes": w["weights"] + w["kv"] * (p + n) + w["out"], "flops": w["flops"]}
    keys = sum(p + 1 for p in _batch_pos(case))
    w = _model_work(case, case["n"], keys, case["n"])
    return {"bytes": w["weights"] + w["kv"] * keys + w["out"], "flops": w["flops"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "requant":
        return "exact"
    if kind in ("gemv", "head"):
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}       # fp32 sums over exact integers
    if kind == "gptq":
        # the input's 15-bit fixed point against float products: 5e-5, 2e-4
        return {"rel": 2e-4, "max": 1e-3}
    if kind == "ffn":
        return {"rel": 2e-3, "max": 2e-2}                       # a code of h may round the other way (3e-4)
    if kind in ("attn", "attn_prompt"):
        # fp32 sums in another order: 7e-7, 8e-6; an fp16 cache entry may round the other way
        return {"rel": 1e-5, "max": 2e-3, "differ": 0.01}
    if kind == "ffn_rows":
        return {"rel": 1e-5, "max": 1e-4}                       # two orders of the fp32 sums: 3e-7, 2e-5
    if kind == "moe":
        return {"rel": 2e-3, "max": 3e-2}                       # as the dense block
    # Several layers: the int8 codes of every layer's inputs round the other
    # way where another order of a sum moves them, and the logits then differ
    # by the quantization's own noise: 0.015 and 0.15 over 4 layers for two
    # correct orders, where a wrong term shows at 1.
    return {"rel": 3e-2, "max": 0.5}


# ---------------------------------------------------------------- the same in 64 bits

def exact(case, seed):
    kind = case["kind"]
    g = _gen(seed, kind)
    if kind in ("gemv", "head"):
        m = Weights(g, case["rows"], case["cols"], case["bits"], upload=False)
        x = _x(g, case["cols"]).double()
        if kind == "head" or case["norm"]:
            x = _norm64(x, (1 + 0.1 * _randn(g, case["cols"])).double())
        y = m.dense() @ _deq(*_quant64(x, 32))
        return {"y": y} if kind == "gemv" else {"y": y, "tok": None}
    if kind == "ffn":
        gate, up = (Weights(g, case["ff"], case["cols"], case["bits"], upload=False) for _ in range(2))
        down = Weights(g, case["cols"], case["ff"], case["bits"], upload=False)
        x, w = _x(g, case["cols"]).double(), (1 + 0.1 * _randn(g, case["cols"])).double()
        x = _norm64(x, w)
        if case["perm"]:
            x = x[torch.randperm(case["cols"], generator=g, device=DEV)]
        a = _deq(*_quant64(x, 32))
        h = _silu64(gate.dense() @ a) * (up.dense() @ a)
        return {"h": h, "y": down.dense() @ _deq(*_quant64(h, 32))}
    if kind == "gptq":
        qw, qz, sc, gi, x = _gptq_arrays(case, seed)
        rows, cols = case["rows"], case["cols"]
        sh = torch.arange(0, 32, 4, device=DEV, dtype=torch.int32)
        codes = ((qw[:, None, :] >> sh[None, :, None]) & 15).reshape(cols, rows)
        zeros = ((qz[:, :, None] >> sh) & 15).reshape(cols // 128, rows) + 1
        grp = torch.arange(cols, device=DEV) // 128 if gi is None else gi.long()
        w = (codes - zeros[grp]).double() * sc.double()[grp]
        return {"y": x.double() @ w}
    if kind in ("attn", "attn_prompt"):
        H, KV, n_ctx, hd, p, n = case["heads"], case["kv"], case["n_ctx"], 128, case["pos"], case.get("n", 1)
        qkv = _randn(g, n, (H + 2 * KV) * hd).double()
        kc, vc = _randn(g, n_ctx, KV * hd).half(), _randn(g, n_ctx, KV * hd).half()
        c, s = (t[p:p + n, None].double() for t in _rope(5e5, hd // 2, n_ctx))
        q = _rotate64(qkv[:, : H * hd].view(n, H, hd), c, s)
        k = _rotate64(qkv[:, H * hd:(H + KV) * hd].view(n, KV, hd), c, s)
        kc[p:p + n], vc[p:p + n] = k.reshape(n, -1).half(), qkv[:, (H + KV) * hd:].half()
        K, V = (t[: p + n].double().view(p + n, KV, hd) for t in (kc, vc))
        dead = torch.arange(p + n, device=DEV)[None] > torch.arange(p, p + n, device=DEV)[:, None]
        out = torch.empty(n, H, hd, dtype=torch.float64, device=DEV)
        for h in range(H):
            sc = (q[:, h] @ K[:, h // (H // KV)].T.contiguous() / math.sqrt(hd)).masked_fill(dead, -math.inf)
            out[:, h] = torch.softmax(sc, -1) @ V[:, h // (H // KV)]
        out = out.view(n, H * hd)
        if kind == "attn":
            return {"out": out, "codes": None, "scale": _quant64(out[0], 32)[1], "k": kc[p].double(),
                    "v": vc[p].double()}
        return {"out": out, "k": kc[p:p + n].double(), "v": vc[p:p + n].double()}
    if kind == "ffn_rows":
        gate, up = (Weights(g, case["ff"], case["cols"], case["bits"], upload=False) for _ in range(2))
        down = Weights(g, case["cols"], case["ff"], case["bits"], upload=False)
        a, b = (_quant64(_randn(g, case["n"], n).double(), 256 if case["per256"] else 32)
                for n in (case["cols"], case["ff"]))
        a, b = (_deq(q, sc.float().double()) for q, sc in (a, b))
        h = _silu64(a @ gate.dense().T.contiguous()) * (a @ up.dense().T.contiguous())
        return {"h": h, "y": b @ down.dense().T.contiguous()}
    return None
