"""What the library enqueues and leaves behind, on the host HIP runtime (host_hip.cpp): run by
tests/test_host_hip.py in a process of its own, whose GE_LIBRARY is the library's objects over it."""
import ctypes as C

import numpy as np
import pytest

import gemma_embed as ge

P, I = C.c_void_p, C.c_int
LAUNCH = C.CFUNCTYPE(None, C.c_char_p, C.POINTER(P))
lib = ge.lib
lib.host_hip_pending.restype = C.c_uint64
lib.host_hip_pending_copies.restype = C.c_uint64
lib.host_hip_pending_copies.argtypes = [P, C.c_size_t]
lib.host_hip_block.argtypes = [P, C.POINTER(P), C.POINTER(C.c_size_t)]
lib.host_hip_fail.argtypes = [C.c_char_p, I]
lib.host_hip_on_launch.argtypes = [LAUNCH]


class QkvEpilogue(C.Structure):
    """kernels.hpp"""
    _fields_ = [(n, P) for n in ("q_norm", "k_norm", "positions", "rope", "q", "k", "v", "vcol", "vt")] + \
        [("scale", C.c_float), ("eps", C.c_float), ("vt_cols", I), ("heads", I), ("kv_heads", I), ("stage", P)]


def arg(args, i, kind):
    return C.cast(args[i], C.POINTER(kind))[0]


def block_end(p):
    """The end of the allocation p lies in."""
    base, size = P(), C.c_size_t()
    assert lib.host_hip_block(P(p), C.byref(base), C.byref(size)), hex(p)
    return base.value + size.value


def ints(p, n):
    """n int32 of an array in device memory, which must hold them all."""
    assert p + 4 * n <= block_end(p), f"{n} int32 at {p:#x} run past the allocation's end {block_end(p):#x}"
    return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_int32)), (n,)).copy()


class Launches:
    """The launches of a block, read as they are made: (kernel, what `read` returns) of those it knows.
    A failing reader is raised when the block ends (ctypes callbacks swallow exceptions)."""

    def __init__(self, read):
        self.read, self.seen, self.error = read, [], None

    def __enter__(self):
        def on_launch(name, args):
            try:
                got = self.read(name.decode(), args)
                if got is not None:
                    self.seen.append((name.decode(), got))
            except BaseException as e:  # noqa: BLE001
                self.error = self.error or e
        self.callback = LAUNCH(on_launch)
        lib.host_hip_on_launch(self.callback)
        return self.seen

    def __exit__(self, *exc):
        lib.host_hip_on_launch(LAUNCH())
        if self.error and not exc[0]:
            raise self.error


def load(tmp_path, **shape):
    path = ge.synth_write_gguf(str(tmp_path / "m.gguf"), **dict(ge.TINY, **shape))
    return ge.EmbeddingModel.load(path)


def vt_launch(name, args):
    """(tokens, V^T columns of them, vt_cols) of a launch that stores V^T."""
    if "gemm_qkv_kernel" in name or "qkv_rowpass_kernel" in name:
        fused = "gemm_qkv_kernel" in name
        n, e = arg(args, 2 if fused else 1, I), arg(args, 7 if fused else 3, QkvEpilogue)
        vcol, cols, vt = e.vcol, e.vt_cols, e.vt
        if not vt:
            return None
    elif "v_transpose_kernel" in name:
        n, vcol, cols = arg(args, 1, I), arg(args, 3, P), arg(args, 4, I)
    elif "qkv_norm_rope_vt_kernel" in name:
        pytest.fail("a path these checks do not read")
    else:
        return None
    return n, ints(vcol, n), cols


# The QKV epilogue (from 65 rows in tiles, below as a row pass), and the separate V transpose of the
# split-precision layers.
SHAPES = {"fused": dict(heads=3, head_dim_swa=256, head_dim_global=256),
          "transpose": dict(heads=4, head_dim_swa=512, head_dim_global=512)}


@pytest.mark.parametrize("shape", SHAPES)
def test_tokens_of_empty_sequences_have_v_columns(tmp_path, shape):
    """A batch whose sequences are all empty still runs every token through the projections, which store
    its V at vcol[token]: those columns must be there, inside V^T, whatever the batch before left."""
    with load(tmp_path, **SHAPES[shape]) as model:
        h = model.context.handle
        ids = np.full(6000, 500, np.int32)
        pos = (np.arange(6000) % 400).astype(np.int32)
        out = np.zeros((8, model.context.out_dims), np.float32)

        def forward(n, seqs):
            with Launches(vt_launch) as seen:
                model.context._check(lib.ge_forward(h, ge._ptr(ids, C.c_int32), ge._ptr(pos, C.c_int32), n,
                                                    ge._seq_array(seqs), len(seqs), ge._ptr(out, C.c_float), None), "ge_forward")
            assert sum(rows for _, (rows, _, _) in seen) == 2 * n  # two layers, every token
            for name, (_, cols, vt_cols) in seen:
                assert cols.min() >= 0 and cols.max() < vt_cols, (name, cols.min(), cols.max(), vt_cols)

        forward(5000, [(0, 0)])            # a fresh workspace
        forward(40, [(0, 0), (17, 0)])
        forward(5999, [(0, 100), (200, 400)])  # the columns' place then holds other arrays' words
        for n in (3, 64, 1000, 5000):
            forward(n, [(0, 0), (1, 0)])


@pytest.fixture(scope="module")
def tower(tmp_path_factory):
    path = ge.synth_write_vision_gguf(str(tmp_path_factory.mktemp("v") / "tower.gguf"), **ge.TINY_VISION)
    ctx = ge.Context.create(0)
    ctx.vision_load(path)
    yield ctx
    ctx.close()


def vision_call(ctx, patches, grids, room):
    """ge_vision_encode's status and message, with vectors of `room` floats."""
    out = np.zeros(max(room, 1), np.float32)
    rc = lib.ge_vision_encode(ctx.handle, ge._ptr(patches, C.c_float), len(patches), ge._grid_array(grids), len(grids),
                              ge._ptr(out, C.c_float), room, None)
    return rc, lib.ge_last_error(ctx.handle).decode()


@pytest.mark.parametrize("images", [1, 30])  # one part; two (4320 patch rows)
def test_failed_vision_encode_leaves_nothing_in_flight(tower, images):
    """The images are copied from the caller's memory while the tower runs: whichever step fails, the call
    waits for those copies, and a batch whose images did not all arrive is no longer staged."""
    ctx, grids = tower, [(12, 12)] * images
    patches = ge.image_patches(3, grids, ctx.vision_info().patch_area)
    room = images * 16 * ctx.vision_info().proj_dims
    assert vision_call(ctx, patches, grids, room)[0] == ge.GE_OK
    nth_copy = images > 1 and 2 or 1
    for call, n, arrived in ((b"hipMemcpyAsync", 1, False), (b"hipMemcpyAsync", nth_copy, False), (b"hipEventRecord", 2, None),
                             (b"kernel:q8_fragments", 1, None), (b"kernel:gemm_kernel", 2 * images, None),
                             (b"kernel:vit_residual2_ln", 5, None), (b"kernel:vit_pool", 1, True), (b"", 0, True)):
        if call:
            lib.host_hip_fail(call, n)
        rc, message = vision_call(ctx, patches, grids, room if call else room - 1)
        lib.host_hip_fail(call, 1 << 30)
        if rc == ge.GE_OK:
            assert arrived is None  # this batch does not make the call that often
            continue
        assert lib.host_hip_pending_copies(patches.ctypes.data, patches.nbytes) == 0, (call, message)
        assert lib.host_hip_pending() == 0, (call, message)
        if arrived is None:
            arrived = lib.ge_vision_tokens(ctx.handle) >= 0
        if arrived:  # a batch whose images are all there stays staged, and can be read or run again
            if not call:
                assert rc == ge.GE_ERR_INVALID and "vector buffer" in message
                assert ctx.vision_read().size == room
            ctx.vision_run()
            ctx.sync()
        else:
            assert lib.ge_vision_tokens(ctx.handle) == -1
            with pytest.raises(ge.GemmaEmbedError) as e:
                ctx.vision_run()
            assert e.value.code == ge.GE_ERR_STATE
    assert vision_call(ctx, patches, grids, room)[0] == ge.GE_OK


# (failing call, batch staged before, batch whose staging fails): in the workspace as it is, with the staged
# block alone grown (as many tokens, more sequences), with everything grown and past the 1 MiB pinned buffer.
STAGING_FAILURES = [(call, first, second) for call in (b"hipEventSynchronize", b"hipMemcpyAsync", b"hipEventRecord")
                    for first, second in (([[5] * 700, [6] * 300], [[8] * 90]), ([[5] * 1000], [[6]] * 1000))] + \
    [(b"hipHostMalloc", [[5] * 700, [6] * 300], [[7] * 1000] * 140), (b"hipMalloc", [[5] * 1000], [[6]] * 1000)]


@pytest.mark.parametrize("call,first,second", STAGING_FAILURES)
def test_failed_staging_keeps_no_mixed_batch(tmp_path, call, first, second):
    """A staging that fails leaves either the batch before it, its arrays where its launches read them, or none."""
    def read(name, args):
        if "gemm_qkv_kernel" not in name and "qkv_rowpass_kernel" not in name:
            return None
        fused = "gemm_qkv_kernel" in name
        n, e = arg(args, 2 if fused else 1, I), arg(args, 7 if fused else 3, QkvEpilogue)
        return ints(e.positions, n).tolist() + ints(e.vcol, n).tolist()

    with load(tmp_path, **SHAPES["fused"]) as model:
        ctx = model.context
        ctx.batch_stage(first)
        with Launches(read) as before:
            ctx.batch_run()
        lib.host_hip_fail(call, 1)
        with pytest.raises(ge.GemmaEmbedError) as e:
            ctx.batch_stage(second)
        assert e.value.code == ge.GE_ERR_GPU
        with Launches(read) as after:
            try:
                ctx.batch_run()
            except ge.GemmaEmbedError as failed:
                assert failed.code == ge.GE_ERR_STATE
        assert not after or after == before
        ctx.batch_stage(second)
        ctx.batch_run()


@pytest.mark.parametrize("heads,head_dim", [(3, 256), (4, 256)])  # LDS-copy attention; the producer-wave one
def test_refused_attention_call_leaves_nothing_in_flight(heads, head_dim):
    """The per-op entries' temporaries are the context's: a call that is refused after its first kernel was
    launched must have waited, or the next call's constants land in memory that kernel is still writing."""
    ctx = ge.Context.create(0)
    work = ge.attention_work([(0, 100), (100, 30)])
    p = [ctx.alloc(n) for n in (200 * heads * head_dim * 2, 200 * head_dim * 2, 200 * head_dim * 2,
                                200 * heads * head_dim * 2, work.nbytes)]
    ctx.upload(p[4], work)
    ctx.sync()
    for half_window, scale_ok in ((-1, False), (0, True)):
        try:
            ctx.attention(p[0], p[1], p[2], p[3], p[4], len(work), heads, 1, head_dim, half_window)
            assert scale_ok
        except ge.GemmaEmbedError as e:
            assert not scale_ok and e.code == ge.GE_ERR_INVALID
        assert lib.host_hip_pending() == 0, half_window
    ctx.close()


@pytest.mark.parametrize("lengths,parts", [([1000, 1047], 1), ([1000, 1048], 2), ([7, 2041], 1), ([2041, 7], 1),
                                           ([255, 1793], 1), ([256, 1792], 2), ([1792, 256], 2), ([1793, 255], 1),
                                           ([3, 3000, 5], 1), ([600, 3000, 600], 2), ([64] * 40, 2)])
def test_packs_split_only_into_parts_worth_a_stream(tmp_path, lengths, parts):
    """From 2048 tokens, and only where the smaller part has an eighth of them."""
    with load(tmp_path) as model:
        with Launches(lambda name, args: arg(args, 3, I) if "embed_norm_kernel" in name else None) as seen:
            model.context.forward([[5] * n for n in lengths])
    rows = [n for _, n in seen]
    assert len(rows) == parts and sum(rows) == sum(lengths) and min(rows) * 8 >= sum(lengths)


def test_a_context_is_created_beside_a_capture():
    """The search for a second hardware queue waits for its own streams: that must not be refused while another
    part of the program captures a graph, nor end its capture."""
    lib.host_hip_capture(1)
    ctx = ge.Context.create(0)
    assert lib.host_hip_capture(0) == 1
    ctx.close()
