"""The per-op entries' temporary buffers, the context's own from call to call: calls of growing and
shrinking sizes, below and above what the context keeps, give what a fresh context gives."""
import numpy as np
import pytest

import gemma_embed as ge

pytestmark = pytest.mark.gpu


def attend(ctx, lengths, seed):
    rng = np.random.default_rng(seed)
    n = sum(lengths)
    q = rng.standard_normal((n + 64, 3, 256)).astype(np.float16)
    k, v = (rng.standard_normal((n + 64, 1, 256)).astype(np.float16) for _ in range(2))
    work = ge.attention_work([(sum(lengths[:i]), x) for i, x in enumerate(lengths)])
    ptrs = [ctx.alloc(a.nbytes) for a in (q, k, v, work)] + [ctx.alloc(n * 3 * 256 * 2)]
    for p, a in zip(ptrs, (q, k, v, work)):
        ctx.upload(p, a)
    ctx.attention(ptrs[0], ptrs[1], ptrs[2], ptrs[4], ptrs[3], len(work), 3, 1, 256, 0)
    out = ctx.download(ptrs[4], (n, 768), np.float16)
    for p in ptrs:
        ctx.free(p)
    return out


def embed(ctx, n, cols, seed):
    """x of n tokens from a 64-row table, with the norm's rows going to a temporary (no h)."""
    rng = np.random.default_rng(seed)
    blocks = np.zeros((64 * cols // 32, 34), np.uint8)
    d = (0.001 + 0.01 * rng.random(len(blocks))).astype(np.float16)
    quants = rng.integers(-127, 128, (len(blocks), 32)).astype(np.int8)
    blocks[:, :2], blocks[:, 2:] = d.view(np.uint8).reshape(-1, 2), quants.view(np.uint8)
    table = ctx.q8_create(blocks, 64, cols)
    ids = rng.integers(0, 64, n).astype(np.int32)
    pt, px = ctx.alloc(ids.nbytes), ctx.alloc(n * cols * 4)
    ctx.upload(pt, ids)
    ctx.embed(ge.C.c_void_p(table), pt, n, 2.0, None, 0, None, 1e-6, px, None)
    x = ctx.download(px, (n, cols), np.float32)
    for p in (pt, px):
        ctx.free(p)
    ctx.q8_destroy(table)
    rows = (d.astype(np.float32)[:, None] * quants.astype(np.float32)).reshape(64, cols) * np.float32(2)
    assert np.array_equal(x, rows[ids])


def test_calls_of_changing_sizes():
    fresh = {}
    calls = [(5, [7]), (6, [300, 41, 1000]), (7, [1, 64, 3])]
    for seed, lengths in calls:
        c = ge.Context.create(0)
        fresh[seed] = attend(c, lengths, seed)
        c.close()
    ctx = ge.Context.create(0)
    for seed, lengths in calls + calls[::-1]:
        print("attention", lengths, flush=True)
        assert np.array_equal(attend(ctx, lengths, seed), fresh[seed])
    for n in (3, 40000, 5):  # 40000 x 1024 halves: more than a context keeps
        print("embed", n, flush=True)
        embed(ctx, n, 1024, n)
    ctx.close()


def test_norm_after_a_refused_attention_call():
    """A call refused after its first launch has waited for it: the ones that the next norm takes for its
    weights are not written over by that kernel."""
    ctx = ge.Context.create(0)
    attend(ctx, [4000], 1)  # sizes the temporaries
    n, heads = 4000, 3
    work = ge.attention_work([(0, n)])
    big = [ctx.alloc((n + 64) * heads * 256 * 2) for _ in range(4)] + [ctx.alloc(work.nbytes)]
    ctx.upload(big[2], np.full((n + 64, 256), 3.0, np.float16))
    ctx.upload(big[4], work)
    x = np.random.default_rng(2).standard_normal((64, 1024)).astype(np.float32)
    px, out = ctx.alloc(x.nbytes), ctx.alloc(x.nbytes)
    ctx.upload(px, x)
    want = x / np.sqrt((x.astype(np.float64) ** 2).mean(axis=1, keepdims=True) + 1e-6)
    for _ in range(5):
        with pytest.raises(ge.GemmaEmbedError) as e:
            ctx.attention(big[0], big[1], big[2], big[3], big[4], len(work), heads, 1, 256, -1)
        assert e.value.code == ge.GE_ERR_INVALID
        ctx.rmsnorm(px, out, None, 64, 1024, 1e-6)
        assert np.abs(ctx.download(out, x.shape, np.float32) - want).max() < 1e-5
    for p in big + [px, out]:
        ctx.free(p)
    ctx.close()
