"""The tile shapes the GEMM launchers choose by the size of a launch, at the edges of each range: every
shape runs the same MFMA over the same k order, so a row's result is the same bits in all of them."""
import numpy as np
import pytest

import gemma_embed as ge

pytestmark = pytest.mark.gpu

# Rows at which a 768-wide projection changes shape on 256 CUs: the skinny kernel up to 320 (10 x 24
# waves), 64 x 64 tiles up to 1344 (21 x 12) and, with shorter stages, up to 2688 (42 x 12), 128 x 128 up
# to 5376 (42 x 6).
EDGES = (1, 320, 321, 1344, 1345, 2688, 2689, 5376, 5377)
# The same for gate/up pairs of 2304 columns: skinny up to 224 (7 x 36), 64 x 128 up to 896 (14 x 18),
# 128 x 128 up to 1792 (14 x 18).
PAIR_EDGES = (224, 225, 896, 897, 1792, 1793)


@pytest.fixture(scope="module")
def ctx():
    c = ge.Context.create(0)
    yield c
    c.close()


def q8(rng, rows, cols):
    blocks = np.zeros((rows * cols // 32, 34), np.uint8)
    d = (np.abs(rng.standard_normal(len(blocks))) * 0.02 / 127 + 1e-4).astype(np.float16)
    blocks[:, :2] = d.view(np.uint8).reshape(-1, 2)
    blocks[:, 2:] = rng.integers(-127, 128, (len(blocks), 32)).astype(np.int8).view(np.uint8)
    return blocks


# K of 1152 takes every shape; 192 and 64 are no multiples of the 128-deep stages, and fill less than a ring
@pytest.mark.parametrize("rows,cols,y_f16", [(768, 1152, False), (768, 768, True), (768, 192, True), (768, 64, False)])
def test_projection_shapes_bitwise(ctx, rows, cols, y_f16):
    rng = np.random.default_rng(rows + cols)
    w = ctx.q8_create(q8(rng, rows, cols), rows, cols)
    x = rng.standard_normal((6400, cols)).astype(np.float16)
    dtype = np.float16 if y_f16 else np.float32
    dx, dy = ctx.alloc(x.nbytes), ctx.alloc(6400 * rows * 4)

    def run(part):
        ctx.upload(dx, part)
        ctx.gemm_q8(w, dx, part.shape[0], dy, y_f16)
        return ctx.download(dy, (part.shape[0], rows), dtype)

    full = run(x)
    for m in EDGES:
        lo = (6400 - m) // 2
        print(f"projection {rows} x {cols}, {m} rows", flush=True)
        assert np.array_equal(run(x[lo:lo + m].copy()), full[lo:lo + m]), m
    ctx.free(dx)
    ctx.free(dy)
    ctx.q8_destroy(w)


# 1120 features: the last 128-column tile of pairs is half outside, with the same changes of shape
@pytest.mark.parametrize("features", [1152, 1120])
def test_gate_up_shapes_bitwise(ctx, features):
    rng = np.random.default_rng(5)
    gate, up = (ctx.q8_create(q8(rng, features, 768), features, 768) for _ in range(2))
    x = rng.standard_normal((2400, 768)).astype(np.float16)
    dx, dy = ctx.alloc(x.nbytes), ctx.alloc(2400 * features * 2)

    def run(part):
        ctx.upload(dx, part)
        ctx.gemm_q8_geglu(gate, up, dx, part.shape[0], dy)
        return ctx.download(dy, (part.shape[0], features), np.float16)

    full = run(x)
    for m in PAIR_EDGES:
        lo = (2400 - m) // 2
        print(f"gate/up, {m} rows", flush=True)
        assert np.array_equal(run(x[lo:lo + m].copy()), full[lo:lo + m]), m
    for p in (dx, dy):
        ctx.free(p)
    for w in (gate, up):
        ctx.q8_destroy(w)


# One head dim per tile width: 256 (one head a tile, 5 slots) and 128 (two heads a tile, 4 slots).
@pytest.mark.parametrize("shape", [dict(hidden=768, heads=3, head_dim_swa=256, head_dim_global=256),
                                   dict(hidden=128, heads=2, head_dim_swa=128, head_dim_global=128)])
def test_qkv_tiles_of_64_and_128_tokens_bitwise(tmp_path, shape):
    """The QKV projection in 64-token tiles (a text alone: from 193 to 3264 tokens at 5 slots of 256), in
    128-token ones (the same text in a pack of 9000 tokens) and on the short batches' kernels."""
    path = ge.synth_write_gguf(str(tmp_path / "qkv.gguf"), **dict(ge.TINY, vocab=512, sliding_window=64, **shape))
    with ge.EmbeddingModel.load(path) as model:
        texts = [ge.synth_tokens(n, 2, 512, n).tolist() for n in (40, 193, 1000, 3264, 3265)]
        rest = [ge.synth_tokens(9, 2, 512, 1500).tolist()]
        pack = model.embed_tokens(texts + rest)
        for i, text in enumerate(texts):
            print(f"text of {len(text)} tokens", flush=True)
            assert np.array_equal(model.embed_tokens([text])[0], pack[i]), len(text)
