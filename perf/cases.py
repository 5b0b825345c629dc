"""The calls this library is measured by: whole embedding calls through the host API, and the
forward's single layers through their device-memory entries.

listed() names the cases, draw() gives others of the same ranges, prepare() makes a case's inputs
on the GPU and the handles a program keeps (a loaded model, weight matrices, output buffers), run()
is one call. exact() states the same results in float64 with plain torch."""
import math
import os
import random
import struct
import sys
import tempfile
import zlib

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("gemma-embed-swift_amd"))
import gemma_embed as ge  # noqa: E402

EPS = 1e-6
# Synthetic weight files of the two text encoders and the image tower (seeded; no weights ship here).
MODELS = {"encoder": ge.CONFIG2, "reference": ge.REAL_SHAPES, "tower": ge.CONFIG5_VISION}
QUEUE = [4, 8, 15, 9, 12, 22, 17, 11, 31, 14, 6, 22]  # 171 tokens: lengths of a queue of search queries


def listed():
    return [
        # A search query typed by a user: one short text, where launches and latency set the time.
        dict(name="query", kind="embed", model="encoder", texts=1, low=12, high=12, dimensions=768),
        # A queue of twelve queries answered one call each, on the reference's own architecture
        # (per-layer inputs, head dims 256 and 512).
        dict(name="queries_reference", kind="queries", model="reference", texts=12, low=4, high=31, dimensions=768),
        # A page of short passages (titles, messages) in one call.
        dict(name="passages", kind="embed", model="encoder", texts=24, low=20, high=101, dimensions=512),
        # Indexing: 256 ragged texts, planned into packs by token count, Matryoshka prefix of 256.
        dict(name="ragged_256", kind="embed", model="encoder", texts=256, low=8, high=256, dimensions=256),
        # Bulk indexing: 32 documents of 512 tokens as one pack.
        dict(name="documents_32x512", kind="pack", model="encoder", texts=32, low=512, high=512),
        # Long documents: 4 texts of 8192 tokens (window 512 on sliding layers, full on global ones).
        dict(name="long_4x8192", kind="pack", model="encoder", texts=4, low=8192, high=8192),
        # Documents of about 1024 tokens on the reference's own architecture, at the default options.
        dict(name="documents_reference", kind="embed", model="reference", texts=8, low=901, high=1024, dimensions=768),
        # A batch of 8 images of 768 x 768 pixels through the image tower, from host pixels.
        dict(name="images_8", kind="images", images=8, grid_x=48, grid_y=48),
        # The feed-forward block's first half for a bulk pack: gate and up projections with GeGLU.
        dict(name="gate_up", kind="gate_up", rows=8192, width=768, features=1152),
        # A projection of a ragged mid-sized pack, fp32 out (the down projection's shape).
        dict(name="projection", kind="projection", rows=1419, width=1152, features=768, half=False),
        # One sliding-window attention layer over a ragged pack.
        dict(name="attention", kind="attention", texts=9, low=130, high=997, heads=3, kv_heads=1, head_dim=256,
             window=512),
        # The residual step with both norms after a sublayer, over a bulk pack.
        dict(name="residual_norm", kind="residual_norm", rows=16384, width=768),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["embed", "embed", "embed", "queries", "pack", "images", "gate_up", "projection", "attention",
                       "residual_norm"])
    model = rng.choice(["encoder", "encoder", "reference"])
    if kind == "queries":
        return dict(kind=kind, model=model, texts=rng.randint(2, 12), low=4, high=spread(8, 48), dimensions=768)
    if kind in ("embed", "pack"):
        high = spread(8, 2048)
        low = max(2, high // rng.choice([1, 2, 8]))
        texts = min(spread(1, 256), max(1, (24576 if kind == "embed" else 16384) // high))
        if kind == "pack":
            return dict(kind=kind, model="encoder", texts=texts, low=low, high=high)
        return dict(kind=kind, model=model, texts=texts, low=low, high=high, dimensions=rng.choice([768, 512, 256, 128]))
    if kind == "images":
        return dict(kind=kind, images=rng.randint(1, 6), grid_x=3 * rng.randint(4, 16), grid_y=3 * rng.randint(4, 16))
    if kind == "gate_up":
        width, features = rng.choice([(768, 1152), (512, 2048)])
        return dict(kind=kind, rows=spread(8, 16384), width=width, features=features)
    if kind == "projection":
        width, features = rng.choice([(768, 1280), (768, 768), (1152, 768), (512, 2048), (2048, 512), (1024, 512)])
        return dict(kind=kind, rows=spread(8, 16384), width=width, features=features, half=rng.random() < 0.5)
    if kind == "attention":
        heads, kv_heads, head_dim = rng.choice([(3, 1, 256), (4, 2, 256), (2, 1, 128)])
        high = spread(16, 2048)
        return dict(kind=kind, texts=min(spread(1, 64), max(1, 16384 // high)), low=max(8, high // 4), high=high,
                    heads=heads, kv_heads=kv_heads, head_dim=head_dim, window=rng.choice([0, 512, 1024]))
    return dict(kind=kind, rows=spread(8, 32768), width=rng.choice([512, 768, 1024]))


# ---------------------------------------------------------------------------- inputs


def lengths(case):
    """Text lengths of a case: fixed by the case, the same for every seed."""
    if case["kind"] == "queries" and case["texts"] == len(QUEUE) and case["high"] == 31:
        return list(QUEUE)
    rng = random.Random(zlib.crc32(repr(sorted(case.items())).encode()))
    return [rng.randint(case["low"], case["high"]) for _ in range(case["texts"])]


def texts(case, seed):
    """Token ids uniform over the vocabulary, framed by <bos> = 2 and <eos> = 1 as a tokenizer returns them."""
    rng = np.random.default_rng(seed)
    return [[2] + rng.integers(3, 262144, n - 2).tolist() + [1] for n in lengths(case)]


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def q8_rows(rng, rows, cols):
    """Q8_0 rows: blocks of an fp16 scale and 32 int8 values uniform in [-127, 127]."""
    blocks = np.zeros((rows * cols // 32, 34), np.uint8)
    q = rng.integers(-127, 128, (blocks.shape[0], 32)).astype(np.int8)
    scale = (np.abs(rng.normal(0.0, 0.02, blocks.shape[0])) * np.abs(q).max(axis=1) / 127).astype(np.float16)
    blocks[:, :2] = scale.view(np.uint8).reshape(-1, 2)
    blocks[:, 2:] = q.view(np.uint8)
    return blocks.reshape(rows, -1)


def dequantised(rows, cols):
    """float64 [rows][cols] on the GPU of Q8_0 bytes."""
    b = np.ascontiguousarray(rows).reshape(-1, 34)
    d = torch.from_numpy(b[:, :2].copy().view(np.float16).astype(np.float64)).cuda()
    return (d * torch.from_numpy(b[:, 2:].view(np.int8).copy()).cuda()).reshape(-1, cols)


def path_of(name):
    spec = MODELS[name]
    path = os.path.join(tempfile.gettempdir(), "gemma_embed_%d_%s_%08x.gguf" % (
        os.getuid(), name, zlib.crc32(repr(sorted(spec.items())).encode())))
    if not os.path.exists(path):
        write = ge.synth_write_vision_gguf if name == "tower" else ge.synth_write_gguf
        write("%s.%d" % (path, os.getpid()), **spec)
        os.replace("%s.%d" % (path, os.getpid()), path)
    return path


HELD = {}


def held(name):
    """The models and the context a program keeps loaded: one of each per process."""
    if name not in HELD:
        if name == "context":
            HELD[name] = ge.Context.create(0)
        elif name == "tower":
            HELD[name] = ge.Context.create(0)
            HELD[name].vision_load(path_of("tower"))
        else:
            HELD[name] = ge.EmbeddingModel.load(path_of(name))
    return HELD[name]


class Matrix:
    """A Q8_0 weight matrix in device memory, given back with its state."""

    def __init__(self, context, rows_q8, rows, cols):
        self.context, self.handle = context, context.q8_create(rows_q8, rows, cols)

    def __del__(self):
        self.context.q8_destroy(self.handle)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("embed", "queries", "pack"):
        options = ge.EmbedOptions(max_tokens=8192, dimensions=case.get("dimensions", 768))
        return dict(kind=kind, model=held(case["model"]), texts=texts(case, seed), options=options)
    if kind == "images":
        grids = [(case["grid_x"], case["grid_y"])] * case["images"]
        rng = np.random.default_rng(seed)
        pixels = rng.random((sum(x * y for x, y in grids), 768), dtype=np.float32) * np.float32(2) - np.float32(1)
        return dict(kind=kind, context=held("tower"), patches=pixels, grids=grids)
    c, g = held("context"), generator(seed)

    def half(*shape):
        return torch.randn(*shape, generator=g, device="cuda").half()

    if kind in ("gate_up", "projection"):
        rows, width, features = case["rows"], case["width"], case["features"]
        rng = np.random.default_rng(seed)
        w = [Matrix(c, q8_rows(rng, features, width), features, width) for _ in range(2 if kind == "gate_up" else 1)]
        out = torch.zeros(rows, features, device="cuda",
                          dtype=torch.float32 if kind == "projection" and not case["half"] else torch.float16)
        return dict(kind=kind, context=c, w=w, x=half(rows, width), out=out)
    if kind == "attention":
        n, start = lengths(case), 0
        ranges = []
        for length in n:
            ranges.append((start, length))
            start += length
        # unit-RMS rows and unscaled products, as the head norms leave them; 64 rows of slack
        q, k, v = (half(start + 64, h, case["head_dim"]) for h in (case["heads"], case["kv_heads"], case["kv_heads"]))
        items = torch.from_numpy(ge.attention_work(ranges).astype(np.int32)).cuda()
        out = torch.zeros(start, case["heads"], case["head_dim"], device="cuda", dtype=torch.float16)
        return dict(kind=kind, context=c, q=q, k=k, v=v, work=items, out=out, case=dict(case))
    rows, width = case["rows"], case["width"]
    x = torch.randn(rows, width, generator=g, device="cuda") * 20
    w, next_w = (1 + 0.1 * torch.randn(width, generator=g, device="cuda") for _ in range(2))
    return dict(kind=kind, context=c, x=x, t=half(rows, width), w=w, next_w=next_w,
                h=torch.zeros(rows, width, device="cuda", dtype=torch.float16))


def run(s):
    kind = s["kind"]
    if kind == "embed":
        return np.stack([e.vector for e in s["model"].embed(s["texts"], s["options"])])
    if kind == "queries":
        return [s["model"].embed([text], s["options"])[0].vector for text in s["texts"]]
    if kind == "pack":
        return s["model"].context.forward(s["texts"])[0]
    c = s["context"]
    if kind == "images":
        return c.vision_encode(s["patches"], s["grids"])[0]
    if kind == "gate_up":
        c.gemm_q8_geglu(s["w"][0].handle, s["w"][1].handle, s["x"].data_ptr(), s["x"].shape[0], s["out"].data_ptr())
        return s["out"]
    if kind == "projection":
        c.gemm_q8(s["w"][0].handle, s["x"].data_ptr(), s["x"].shape[0], s["out"].data_ptr(),
                  s["out"].dtype == torch.float16)
        return s["out"]
    if kind == "attention":
        k = s["case"]
        c.attention(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["out"].data_ptr(), s["work"].data_ptr(),
                    s["work"].shape[0], k["heads"], k["kv_heads"], k["head_dim"], k["window"] // 2)
        return s["out"]
    c.rmsnorm_residual(s["x"].data_ptr(), s["t"].data_ptr(), s["w"].data_ptr(), 1.0, s["next_w"].data_ptr(),
                       s["h"].data_ptr(), s["x"].shape[0], s["x"].shape[1], EPS)
    return [s["x"], s["h"]]


# ---------------------------------------------------------------------------- necessary work


def pairs(n, window):
    """Visible (query, key) pairs of one text of n tokens: all, or those with |i - j| <= window / 2."""
    h = window // 2 if window else n
    if h >= n:
        return n * n
    return n * (2 * h + 1) - h * (h + 1)


def work(case):
    kind = case["kind"]
    if kind in ("embed", "queries", "pack"):
        m, n = MODELS[case["model"]], lengths(case)
        d, ff, pl, tokens = m["hidden"], m["feed_forward"], m["per_layer_input"], sum(n)
        params, attention = pl * m["layers"] * d, 0
        for sliding in m["pattern"]:
            hd = m["head_dim_swa"] if sliding else m["head_dim_global"]
            kv = m["kv_heads_swa"] if sliding else m["kv_heads_global"]
            params += d * hd * (2 * m["heads"] + 2 * kv) + 3 * d * ff + 2 * d * pl
            attention += sum(pairs(i, m["sliding_window"] if sliding else 0) for i in n) * 4 * hd * m["heads"]
        calls = len(n) if kind == "queries" else 1
        return dict(bytes=calls * params * 34 / 32 + tokens * (d * 34 / 32 + 4) + len(n) * 768 * 4,
                    flops=2 * params * tokens + attention + 2 * len(n) * d * 768)
    if kind == "images":
        v, n = MODELS["tower"], case["grid_x"] * case["grid_y"]
        d, ff = v["hidden"], v["feed_forward"]
        params = v["layers"] * (4 * d * d * 34 / 32 + d * ff * (34 / 32 + 2)) + 2 * 768 * d * 34 / 32
        flops = n * (2 * 768 * d + v["layers"] * (8 * d * d + 4 * d * ff + 4 * n * d)) + n / 9 * 2 * d * 768
        return dict(bytes=params + case["images"] * n * (768 * 4 + 768 * 4 / 9), flops=case["images"] * flops)
    if kind in ("gate_up", "projection"):
        rows, k, f = case["rows"], case["width"], case["features"] * (2 if kind == "gate_up" else 1)
        out = case["features"] * (2 if kind == "gate_up" or case["half"] else 4)
        return dict(bytes=rows * (2 * k + out) + f * k * 34 / 32, flops=2 * rows * k * f)
    if kind == "attention":
        n, hd = lengths(case), case["head_dim"]
        return dict(bytes=sum(n) * hd * 2 * (2 * case["heads"] + 2 * case["kv_heads"]),
                    flops=4 * hd * case["heads"] * sum(pairs(i, case["window"]) for i in n))
    return dict(bytes=case["rows"] * case["width"] * (4 + 2 + 4 + 2), flops=case["rows"] * case["width"] * 10)


def tolerance(case):
    """About four times the distance from exact(): fp16 operands and stored activations, fp32 sums. Whole
    calls measure 2e-4 to 6.5e-4, single layers 2e-4 (gate_up 3.6e-4: its product is stored in fp16)."""
    return {"embed": {"rel": 3e-3}, "queries": {"rel": 3e-3}, "pack": {"rel": 3e-3}, "images": {"rel": 3e-3},
            "gate_up": {"rel": 1.5e-3}, "projection": {"rel": 1e-3}, "attention": {"rel": 1e-3},
            "residual_norm": {"rel": 1e-3}}[case["kind"]]


# ---------------------------------------------------------------------------- the same in 64 bits

SCALARS = {0: "<B", 1: "<b", 2: "<H", 3: "<h", 4: "<I", 5: "<i", 6: "<f", 7: "<?", 10: "<Q", 11: "<q", 12: "<d"}


class Weights:
    """A GGUF file's tensors, dequantised to float64 on the GPU as they are asked for."""

    def __init__(self, path):
        self.buf, self.pos = np.memmap(path, dtype=np.uint8, mode="r"), 8
        tensors, keys = self.take("<Q"), self.take("<Q")
        for _ in range(keys):
            self.text()
            self.value(self.take("<I"))
        self.at, self.kept = {}, {}
        for _ in range(tensors):
            name, nd = self.text(), self.take("<I")
            self.at[name] = ([self.take("<Q") for _ in range(nd)], self.take("<I"), self.take("<Q"))
        self.data = (self.pos + 31) // 32 * 32

    def take(self, fmt):
        v = struct.unpack_from(fmt, self.buf, self.pos)[0]
        self.pos += struct.calcsize(fmt)
        return v

    def text(self):
        n = self.take("<Q")
        self.pos += n
        return bytes(self.buf[self.pos - n:self.pos]).decode()

    def value(self, t):
        if t == 8:
            self.text()
        elif t == 9:
            of, n = self.take("<I"), self.take("<Q")
            for _ in range(n):
                self.value(of)
        else:
            self.take(SCALARS[t])

    def raw(self, name):
        shape, t, off = self.at[name]
        n = math.prod(shape)
        return self.buf[self.data + off:self.data + off + {0: 4 * n, 1: 2 * n, 30: 2 * n, 8: n // 32 * 34}[t]]

    def __getitem__(self, name):
        if name not in self.kept:
            (cols, *rest), t, _ = self.at[name]
            raw = self.raw(name)
            if t == 8:
                v = dequantised(raw, cols)
            elif t == 30:
                v = torch.from_numpy((raw.view(np.uint16).astype(np.uint32) << 16).view(np.float32).astype(np.float64)).cuda()
            else:
                v = torch.from_numpy(raw.view(np.float32 if t == 0 else np.float16).astype(np.float64)).cuda()
            self.kept[name] = v.reshape(-1, cols) if rest else v
        return self.kept[name]

    def rows(self, name, ids):
        cols = self.at[name][0][0]
        return dequantised(self.raw(name).reshape(-1, cols // 32 * 34)[np.asarray(ids)], cols)


def weights(name):
    if ("file", name) not in HELD:
        HELD["file", name] = Weights(path_of(name))
    return HELD["file", name]


def rms(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def attend(q, k, v, window, scale=1.0):
    """softmax(q k^T scale) v of one text, [n][heads][hd] over [n][kv_heads][hd]; |i - j| <= window / 2."""
    n, heads = q.shape[0], q.shape[1]
    out = torch.empty_like(q)
    for h in range(heads):
        j = h * k.shape[1] // heads
        s = (q[:, h] @ k[:, j].T.contiguous()) * scale
        if window:
            i = torch.arange(n, device=q.device)
            s.masked_fill_((i[:, None] - i[None, :]).abs() > window // 2, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, j]
    return out


def rotate(x, base):
    half = x.shape[-1] // 2
    turn = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None] * (
        float(np.float32(base)) ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / (2 * half)))
    c, s = turn.cos()[:, None], turn.sin()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def exact_text(name, sequences):
    """Mean-pooled, unnormalised vectors of the texts."""
    w, m = weights(name), MODELS[name]
    d, pl, cut = m["hidden"], m["per_layer_input"], [len(s) for s in sequences]
    x = w.rows("token_embd.weight", sum(sequences, [])) * float(np.float32(math.sqrt(d)))
    if pl:
        per = rms((x @ w["per_layer_model_proj.weight"].T / math.sqrt(d)).reshape(len(x), m["layers"], pl),
                  w["per_layer_proj_norm.weight"])
    for i, sliding in enumerate(m["pattern"]):
        b = "blk.%d." % i
        hd, base = (m["head_dim_swa"], m["rope_base_swa"]) if sliding else (m["head_dim_global"], m["rope_base"])
        h = rms(x, w[b + "attn_norm.weight"])
        q, k, v = ((h @ w[b + "attn_%s.weight" % p].T).reshape(len(x), -1, hd) for p in "qkv")
        q, k, v = rms(q, w[b + "attn_q_norm.weight"]), rms(k, w[b + "attn_k_norm.weight"]), rms(v)
        o = [attend(rotate(a, base), rotate(e, base), f, m["sliding_window"] if sliding else 0)
             for a, e, f in zip(q.split(cut), k.split(cut), v.split(cut))]
        o = torch.cat(o).reshape(len(x), -1) @ w[b + "attn_output.weight"].T
        x = x + rms(o, w[b + "post_attention_norm.weight"])
        f = rms(x, w[b + "ffn_norm.weight"])
        f = gelu(f @ w[b + "ffn_gate.weight"].T) * (f @ w[b + "ffn_up.weight"].T)
        x = x + rms(f @ w[b + "ffn_down.weight"].T, w[b + "post_ffw_norm.weight"])
        if pl:
            p = gelu(x @ w[b + "inp_gate.weight"].T) * per[:, i]
            x = (x + rms(p @ w[b + "proj.weight"].T, w[b + "post_norm.weight"])) * w[b + "layer_output_scale.weight"]
    y = rms(x, w["output_norm.weight"])
    return torch.stack([part.mean(0) for part in y.split(cut)]) @ w["output.weight"].T


def exact_images(s):
    w, m = weights("tower"), MODELS["tower"]
    d, heads, merge = m["hidden"], m["heads"], m["merge"]

    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + m["eps"]) * w[name + ".weight"] + w[name + ".bias"]

    def linear(x, name):
        return x @ w[name + ".weight"].T + w[name + ".bias"]

    out, at = [], 0
    for gx, gy in s["grids"]:
        n = gx * gy
        i = torch.arange(n, device="cuda")
        table = w["v.position_embd.weight"]
        x = linear(torch.from_numpy(s["patches"][at:at + n]).cuda().double(), "v.patch_embd")
        x = x + table[i % gx] + table[m["positions"] + i // gx]
        for layer in range(m["layers"]):
            b = "v.blk.%d." % layer
            h = norm(x, b + "ln1")
            q, k, v = (linear(h, b + "attn_" + p).reshape(n, heads, -1) for p in "qkv")
            x = x + linear(attend(q, k, v, 0, (d // heads) ** -0.5).reshape(n, d), b + "attn_out")
            x = x + linear(gelu(linear(norm(x, b + "ln2"), b + "ffn_up")), b + "ffn_down")
        y = norm(x, "v.post_ln").reshape(gy // merge, merge, gx // merge, merge, d).mean((1, 3)).reshape(-1, d)
        out.append(rms(y, w["mm.soft_emb_norm.weight"]) @ w["mm.input_projection.weight"].T)
        at += n
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("embed", "queries", "pack"):
        y = exact_text(case["model"], texts(case, seed))
        if kind == "pack":
            return y
        y = y[:, :case["dimensions"]]
        y = y / y.norm(dim=1, keepdim=True)
        return list(y) if kind == "queries" else y
    s = prepare(case, seed)
    if kind == "images":
        return exact_images(s)
    if kind in ("gate_up", "projection"):
        rng, x = np.random.default_rng(seed), s["x"].double()
        y = [x @ dequantised(q8_rows(rng, case["features"], case["width"]), case["width"]).T for _ in s["w"]]
        return gelu(y[0]) * y[1] if kind == "gate_up" else y[0]
    if kind == "attention":
        n, heads = lengths(case), zip(*(s[p][:len(s["out"])].double().split(lengths(case)) for p in "qkv"))
        return torch.cat([attend(q, k, v, case["window"]) for q, k, v in heads])
    x = s["x"].double() + rms(s["t"].double(), s["w"].double())
    return [x, rms(x, s["next_w"].double())]
