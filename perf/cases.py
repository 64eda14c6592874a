"""The work that a user of this engine has it do, as cases that can be timed and checked.

Kinds:
  quant      minfer.quant_q8 of one activation vector (before every projection)
  gemv       minfer.quant_q8 + minfer.gemv_q4: one projection of one token
  attn       minfer.attn_decode: one token's attention over its context
  attn_mfma  minfer.attn_decode_mfma: the same with matrix-core chunk records
  prefill    Engine.prefill of a prompt but its last token, then Engine.step of that token
             with its logits
  teacher    Engine.teacher over a token sequence (every position's prediction and margin),
             then Engine.step of its last token with the logits
  chat       Engine.prefill, Engine.generate, then one Engine.step with its logits
  spec       the same with speculative decoding (mi_opts.spec = 1)

Model shapes are minfer.SHAPES (the 0.5B, 1.5B and 3B shapes of the benchmark). The models are
seeded random-init GGUF files written once per machine, with norm weights around 1 and q/k
biases of order 1, so that attention scores and residuals have a trained model's magnitudes;
the seed of a case makes its prompt. A loaded engine is kept per (shape, options), as a
program that serves prompts keeps it: every pass starts from an empty context.
"""
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nano-inference_amd"))
import minfer  # noqa: E402

MAX_CTX = 4352
MODEL_SEED = 2000

# (rows, blocks of 32 columns, blocks per chunk, K segments): projections of the three shapes
# with the K splits the benchmark uses, and the row counts between them
HEADS = {"S05": (14, 2, 64), "S15": (12, 2, 128), "S3": (16, 2, 128)}


def listed():
    return [
        # one activation vector of the 1.5B model: the smallest call, launch latency only
        {"name": "quant_1536", "kind": "quant", "n": 1536},
        # the 0.5B model's o projection: 896 x 896, chunks of 4 blocks
        {"name": "gemv_o_896", "kind": "gemv", "rows": 896, "nb": 28, "cb": 4, "ks": 7},
        # the 1.5B model's down projection, K split in 7 as the benchmark does
        {"name": "gemv_down_1536x8960", "kind": "gemv", "rows": 1536, "nb": 280, "cb": 8, "ks": 7},
        # its lm_head: the largest matrix of a token
        {"name": "gemv_lm_head_151936x1536", "kind": "gemv", "rows": 151936, "nb": 48, "cb": 8, "ks": 1},
        # a short, ragged context on the 0.5B heads (14/2, head size 64)
        {"name": "attn_s05_777", "kind": "attn", "shape": "S05", "L": 777},
        # the benchmark's longest context on the 1.5B heads (12/2, head size 128)
        {"name": "attn_s15_32768", "kind": "attn", "shape": "S15", "L": 32768},
        # a middling context on the 3B heads (16/2), matrix-core form
        {"name": "attn_mfma_s3_8191", "kind": "attn_mfma", "shape": "S3", "L": 8191},
        # a short question and a short answer (the benchmark's 64-token prompt)
        {"name": "chat_s15_64_64", "kind": "chat", "shape": "S15", "n": 64, "gen": 64},
        # speculative decoding of a prompt that repeats itself
        {"name": "spec_s15_200_96", "kind": "spec", "shape": "S15", "n": 200, "gen": 96},
        # an ordinary prompt
        {"name": "prefill_s15_512", "kind": "prefill", "shape": "S15", "n": 512},
        # a long, ragged document
        {"name": "prefill_s15_3001", "kind": "prefill", "shape": "S15", "n": 3001},
        # scoring a text under teacher forcing, on the small model
        {"name": "teacher_s05_301", "kind": "teacher", "shape": "S05", "n": 301},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quant", "gemv", "gemv", "attn", "attn_mfma", "chat", "spec", "prefill", "prefill", "teacher"])
    if kind == "quant":
        return {"kind": kind, "n": 32 * _log(rng, 4, 352)}
    if kind == "gemv":
        cb = rng.choice([4, 8])
        nc = _log(rng, 1, 43)
        rows = 64 * _log(rng, 2, 2374 * 48 // max(48, cb * nc))
        return {"kind": kind, "rows": rows, "nb": cb * nc, "cb": cb, "ks": rng.randint(1, min(nc, 8))}
    if kind in ("attn", "attn_mfma"):
        return {"kind": kind, "shape": rng.choice(list(HEADS)), "L": _log(rng, 5, 32768)}
    shape = rng.choice(["S05", "S15"])
    if kind in ("chat", "spec"):
        return {"kind": kind, "shape": shape, "n": _log(rng, 4, 1000), "gen": rng.randint(8, 120)}
    return {"kind": kind, "shape": shape, "n": _log(rng, 3, 3001)}


# ---------------------------------------------------------------- models
def _dims(shape):
    s = minfer.SHAPES[shape]
    hd = s["n_embd"] // s["n_head"]
    kvd = s["n_head_kv"] * hd
    return dict(L=s["n_layer"], E=s["n_embd"], FF=s["n_ff"], NH=s["n_head"], NKV=s["n_head_kv"], HD=hd, KVD=kvd,
                V=s["n_vocab"])


def _model(shape):
    d = os.path.join(tempfile.gettempdir(), "minfer-perf-%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, "%s-%d.gguf" % (shape, MODEL_SEED))
    if not os.path.exists(path):
        tmp = "%s.%d" % (path, os.getpid())
        minfer.synth_gguf(tmp, shape, MODEL_SEED, emb_q4=True, qk_bias_std=1.0, norm_offset=1.0)
        os.replace(tmp, path)
    return path


_engines = {}


def _engine(shape, spec):
    key = (shape, spec)
    if key not in _engines:
        _engines[key] = minfer.Engine(_model(shape), max_ctx=MAX_CTX, spec=spec)
    return _engines[key]


def _ids(case, seed):
    """the case's tokens; a speculative prompt repeats a seeded pattern, as code and lists do"""
    n, V = case["n"], minfer.SHAPES[case["shape"]]["n_vocab"]
    if case["kind"] == "spec":
        pat = minfer.prompt_ids(seed, min(n, 40), V)
        return (pat * (n // len(pat) + 1))[:n]
    return minfer.prompt_ids(seed, n, V)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _gemv_inputs(case, seed):
    """GGUF q4_0 blocks (fp16 scale of a trained weight's size, 16 nibble bytes) and an
    activation vector of order 1 with a few large channels"""
    g = _gen(seed)
    rows, nb = case["rows"], case["nb"]
    src = torch.randint(0, 256, (rows, nb, 18), dtype=torch.uint8, generator=g)
    d = (torch.rand(rows, nb, generator=g) * 0.01 + 0.001).half()
    src[:, :, :2] = d.view(torch.uint8).reshape(rows, nb, 2)
    x = torch.randn(nb * 32, generator=g)
    x[:: 61] *= 8
    return src, x


def _attn_inputs(case, seed):
    nh, nkv, hd = HEADS[case["shape"]]
    g = torch.Generator("cuda").manual_seed(seed)
    L = case["L"]
    q = torch.randn(nh, hd, device="cuda", generator=g)
    kc = torch.randn(nkv, L, hd, device="cuda", generator=g).half()
    vc = torch.randn(nkv, L, hd, device="cuda", generator=g).half()
    return q, kc, vc


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case)
    if kind in ("quant", "gemv"):
        if kind == "gemv":
            src, x = _gemv_inputs(case, seed)
            rows, nb, cb, ks = case["rows"], case["nb"], case["cb"], case["ks"]
            s["w"] = torch.from_numpy(minfer.pack_q4(src.numpy().reshape(-1), rows, nb, cb)).cuda()
            s["part"] = torch.empty(ks * rows, device="cuda")
            s["y"] = torch.empty(rows, device="cuda")
        else:
            x = torch.randn(case["n"], generator=_gen(seed))
        s["x"] = x.cuda()
        n = x.numel()
        s["xq"] = torch.empty(n, dtype=torch.int8, device="cuda")
        s["xd"] = torch.empty(n // 32, device="cuda")
        s["xs8"] = torch.empty(n // 32, dtype=torch.int32, device="cuda")
    elif kind in ("attn", "attn_mfma"):
        nh, nkv, hd = HEADS[case["shape"]]
        s["q"], s["k"], s["v"] = _attn_inputs(case, seed)
        s["scratch"] = torch.empty(minfer.attn_scratch_floats(nh, hd, case["L"]), device="cuda")
        s["out"] = torch.empty(nh * hd, device="cuda")
    else:
        s["ids"] = _ids(case, seed)
        s["engine"] = _engine(case["shape"], 1 if kind == "spec" else 0)
    return s


def run(s):
    kind = s["kind"]
    if kind in ("quant", "gemv"):
        minfer.quant_q8(s["x"], s["xq"], s["xd"], s["xs8"])
        if kind == "quant":
            return {"codes": s["xq"], "scale": s["xd"], "sum8": s["xs8"]}
        minfer.gemv_q4(s["w"], s["rows"], s["nb"], s["cb"], s["ks"], s["xq"], s["xd"], s["xs8"], s["part"], s["y"])
        return {"y": s["y"]}
    if kind in ("attn", "attn_mfma"):
        nh, nkv, hd = HEADS[s["shape"]]
        f = minfer.attn_decode if kind == "attn" else minfer.attn_decode_mfma
        f(s["q"], s["k"], s["v"], nh, nkv, hd, s["L"], s["L"], 1.0 / hd ** 0.5, s["scratch"], s["out"])
        return {"out": s["out"]}
    e, ids = s["engine"], s["ids"]
    n = len(ids)
    if kind == "teacher":
        pred, margin = e.teacher(ids)
        _, _, logits = e.step(ids[-1], n - 1, want_logits=True)
        return {"pred": np.asarray(pred, np.int32), "margin": np.asarray(margin, np.float32), "logits": logits}
    if kind == "prefill":
        e.prefill(ids[:-1])
        tok, _, logits = e.step(ids[-1], n - 1, want_logits=True)
        return {"token": tok, "logits": logits}
    e.prefill(ids)
    toks, margins = e.generate(s["gen"])
    _, _, logits = e.step(toks[-1], n + s["gen"] - 1, want_logits=True)
    return {"tokens": np.asarray(toks, np.int32), "margins": np.asarray(margins, np.float32), "logits": logits}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "quant":
        n = case["n"]
        return {"bytes": 5 * n + n // 4, "flops": 3 * n}
    if kind == "gemv":
        r, k = case["rows"], case["nb"] * 32
        return {"bytes": r * case["nb"] * 18 + 4 * k + 4 * r, "flops": 2 * r * k}
    if kind in ("attn", "attn_mfma"):
        nh, nkv, hd = HEADS[case["shape"]]
        return {"bytes": 4 * nkv * case["L"] * hd + 8 * nh * hd, "flops": 4 * nh * hd * case["L"]}
    d = _dims(case["shape"])
    layer = (d["E"] + 2 * d["KVD"]) * d["E"] + d["E"] * d["E"] + 3 * d["E"] * d["FF"]
    head, layers = d["V"] * d["E"], d["L"] * layer
    kv, n = 4 * d["L"] * d["KVD"], case["n"]

    def attn(a, b):          # q.k and p.v of positions a..b-1 of a causal context
        return 4 * d["L"] * d["NH"] * d["HD"] * (b * (b + 1) - a * (a + 1)) // 2

    if kind == "teacher":
        return {"bytes": 2 * (layers + head) * 18 // 32 + n * (2 * kv + 4 * d["E"] + 8) + 4 * d["V"],
                "flops": 2 * n * (layers + head) + attn(0, n)}
    if kind == "prefill":
        return {"bytes": (2 * layers + head) * 18 // 32 + 2 * n * kv + 4 * n * d["E"] + 4 * d["V"],
                "flops": 2 * n * layers + 2 * head + attn(0, n)}
    m = case["gen"]          # the prompt, then a step per token; a speculative one verifies up to 8 at once
    steps = m if kind == "chat" else -(-m // 8)
    return {"bytes": (1 + steps) * (layers + head) * 18 // 32 + n * (kv + 4 * d["E"]) + steps * (n + m // 2) * kv
            + 4 * d["V"],
            "flops": 2 * (n + m) * layers + 2 * (m + 1) * head + attn(0, n + m)}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":        # fp16 scales of 32-bit quotients, codes at ties
        return {"rel": 1e-6, "max": 1e-3, "differ": 1e-3}
    if kind == "gemv":         # 32-bit sums of up to 344 scaled block products
        return {"rel": 2e-6, "max": 2e-5}
    if kind in ("attn", "attn_mfma"):
        return {"rel": 1e-5, "max": 1e-4}
    # int8 activations: a rounding in one layer moves codes in all that follow. Logits against
    # the 64-bit model: 2e-4 to 5e-4; margins are differences of two logits: up to 4e-3 on the
    # 1.5B shape and 0.1 on the 0.5B shape, where single positions hold most of it.
    if kind == "prefill":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 2e-2, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------- 64-bit results
class _Gguf:
    """tensors of a GGUF v3 file (F32 and q4_0) as 64-bit values on the GPU"""

    SIZE = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}

    def __init__(self, path):
        self.b = np.memmap(path, np.uint8, "r")
        self.o = 4
        self.rd("I")
        nt, nkv = self.rd("Q"), self.rd("Q")
        for _ in range(nkv):
            self.text()
            self.skip(self.rd("I"))
        self.t = {}
        for _ in range(nt):
            name = self.text()
            dims = [self.rd("Q") for _ in range(self.rd("I"))]
            ty, off = self.rd("I"), self.rd("Q")
            self.t[name] = (ty, dims, off)
        self.base = -(-self.o // 32) * 32

    def rd(self, f):
        n = struct.calcsize("<" + f)
        v = struct.unpack("<" + f, self.b[self.o:self.o + n].tobytes())[0]
        self.o += n
        return v

    def text(self):
        n = self.rd("Q")
        self.o += n
        return self.b[self.o - n:self.o].tobytes().decode("utf-8", "replace")

    def skip(self, t):
        if t == 8:
            self.text()
        elif t == 9:
            et, n = self.rd("I"), self.rd("Q")
            if et in self.SIZE:
                self.o += n * self.SIZE[et]
            else:
                for _ in range(n):
                    self.o += 8 + int.from_bytes(self.b[self.o:self.o + 8].tobytes(), "little")
        else:
            self.o += self.SIZE[t]

    def raw(self, name):
        ty, dims, off = self.t[name]
        cols, rows = dims[0], int(np.prod(dims[1:], dtype=np.int64)) if len(dims) > 1 else 1
        n = rows * cols * 4 if ty == 0 else rows * cols // 32 * 18
        return ty, rows, cols, torch.from_numpy(np.array(self.b[self.base + off:self.base + off + n])).cuda()

    def get(self, name):
        ty, rows, cols, raw = self.raw(name)
        if ty == 0:
            return raw.view(torch.float32).double().reshape(rows, cols).squeeze(0)
        return _q4(raw, rows, cols // 32)


def _q4(raw, rows, nb):
    b = raw.reshape(rows, nb, 18)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    q = torch.cat([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], dim=2).double() - 8
    return (q * d).reshape(rows, nb * 32)


def _int8(x):
    """x as the path's int8 activations: 32-element blocks, code = x * 127 / max, fp16 scale"""
    b = x.reshape(-1, 32)
    a = b.abs().amax(1, keepdim=True)
    codes = torch.round(b * torch.where(a > 0, 127 / a, torch.zeros_like(a)))
    return codes, (a / 127).half().double()


def _act(x):
    c, d = _int8(x)
    return (c * d).reshape(x.shape)


def _logits64(case, ids):
    """64-bit logits of the last position"""
    g, d = _Gguf(_model(case["shape"])), _dims(case["shape"])
    n, NH, NKV, HD = len(ids), d["NH"], d["NKV"], d["HD"]
    emb = g.get("token_embd.weight")
    h = emb[torch.tensor(ids, device="cuda")]
    del emb
    ang = torch.arange(n, device="cuda").double()[:, None] * (1e6 ** (-2 * torch.arange(HD // 2, device="cuda").double() / HD))
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    mask = torch.full((n, n), -math.inf, device="cuda", dtype=torch.float64).triu(1)

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * w

    def rope(x):
        a, b = x[..., :HD // 2], x[..., HD // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    for i in range(d["L"]):
        p = "blk.%d." % i
        x = _act(norm(h, g.get(p + "attn_norm.weight")))
        q, k, v = (x @ g.get(p + "attn_%s.weight" % c).T + g.get(p + "attn_%s.bias" % c) for c in "qkv")
        q = rope(q.reshape(n, NH, HD))
        k = rope(k.reshape(n, NKV, HD)).half().double()
        v = v.reshape(n, NKV, HD).half().double()
        o = torch.empty(n, NH, HD, dtype=torch.float64, device="cuda")
        for j in range(NH):
            kv = j * NKV // NH
            o[:, j] = torch.softmax(q[:, j] @ k[:, kv].T / math.sqrt(HD) + mask, -1) @ v[:, kv]
        h = h + _act(o.reshape(n, NH * HD)) @ g.get(p + "attn_output.weight").T
        x = _act(norm(h, g.get(p + "ffn_norm.weight")))
        a = torch.nn.functional.silu(x @ g.get(p + "ffn_gate.weight").T) * (x @ g.get(p + "ffn_up.weight").T)
        h = h + _act(a) @ g.get(p + "ffn_down.weight").T
    return (_act(norm(h[-1:], g.get("output_norm.weight"))) @ g.get("output.weight").T)[0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "quant":
        x = torch.randn(case["n"], generator=_gen(seed)).double()
        return {"codes": None, "scale": (x.reshape(-1, 32).abs().amax(1) / 127).half().double(), "sum8": None}
    if kind == "gemv":
        src, x = _gemv_inputs(case, seed)
        w = src.cuda()
        xa = _act(x.cuda().double())
        y = torch.cat([_q4(c, c.shape[0], case["nb"]) @ xa for c in w.split(8192)])
        return {"y": y}
    if kind in ("attn", "attn_mfma"):
        nh, nkv, hd = HEADS[case["shape"]]
        q, k, v = (t.double() for t in _attn_inputs(case, seed))
        o = [torch.softmax(k[h * nkv // nh] @ q[h] / math.sqrt(hd), 0) @ v[h * nkv // nh] for h in range(nh)]
        return {"out": torch.cat(o)}
    if case["n"] > 1024:
        return None
    if kind == "teacher":
        return {"pred": None, "margin": None, "logits": _logits64(case, _ids(case, seed))}
    if kind == "prefill":
        return {"token": None, "logits": _logits64(case, _ids(case, seed))}
    return None                               # later tokens depend on the ones chosen before
