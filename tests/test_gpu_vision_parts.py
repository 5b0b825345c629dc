"""Image batches of at least 4096 patch rows run as two parts on two streams: every image's vectors are the
bits it has alone, through the one-call entry (whose patches are uploaded part by part) and as a
staged batch, also when the batch before it was larger or ran as one part."""
import numpy as np
import pytest

import gemma_embed as ge

pytestmark = pytest.mark.gpu


def batch(kinds, count, seed):
    grids = [kinds[i % len(kinds)] for i in range(count)]
    return ge.image_patches(seed, grids, 3 * 16 * 16), grids


def test_two_part_batches_bitwise(tiny_vision_gguf):
    ctx = ge.Context.create(0)
    ctx.vision_load(tiny_vision_gguf)
    # 4098 rows with the cut inside, a cut beside one large image, 4095 rows (one part), two parts again
    for kinds, count in (([(12, 12), (12, 9), (3, 3)], 48), ([(12, 12)], 29), ([(3, 3), (12, 12)], 53), ([(9, 12)], 41)):
        patches, grids = batch(kinds, count, count)
        print(f"{count} images, {len(patches)} patch rows", flush=True)
        got, _ = ctx.vision_encode(patches, grids)
        ctx.vision_stage(patches, grids)
        ctx.vision_run()
        ctx.vision_run()
        assert np.array_equal(ctx.vision_read(), got)
        row = tok = 0
        for i, (gx, gy) in enumerate(grids):
            n, t = gx * gy, gx * gy // 9
            if i in (0, 1, 2, count // 2 - 1, count // 2, count // 2 + 1, count - 2, count - 1):
                alone, _ = ctx.vision_encode(patches[row:row + n], [(gx, gy)])
                assert np.array_equal(alone, got[tok:tok + t]), i
            row, tok = row + n, tok + t
    ctx.close()


@pytest.mark.parametrize("count", [1, 30])  # one part; two (4320 patch rows)
def test_too_small_vector_buffer_leaves_the_patches_read(tiny_vision_gguf, count):
    """A call that fails for its vector buffer has read the caller's patches when it returns: overwritten
    after it, the batch still gives their vectors."""
    ctx = ge.Context.create(0)
    ctx.vision_load(tiny_vision_gguf)
    patches, grids = batch([(12, 12)], count, 5)
    want, _ = ctx.vision_encode(patches, grids)
    for _ in range(3):
        given = patches.copy()
        out = np.zeros(want.size - 1, np.float32)
        rc = ge.lib.ge_vision_encode(ctx.handle, ge._ptr(given, ge.C.c_float), len(given), ge._grid_array(grids), count,
                                     ge._ptr(out, ge.C.c_float), out.size, None)
        given[:] = 0.25
        assert rc == ge.GE_ERR_INVALID
        assert np.array_equal(ctx.vision_read(), want)
        ctx.vision_run()
        assert np.array_equal(ctx.vision_read(), want)
        got, _ = ctx.vision_encode(patches, grids)
        assert np.array_equal(got, want)
    ctx.close()
