"""A context created while another stream of the program is being captured: it is created, and the capture
goes on."""
import ctypes as C
import threading

import pytest

import gemma_embed as ge

pytestmark = pytest.mark.gpu

GLOBAL, THREAD_LOCAL, RELAXED = 0, 1, 2  # hipStreamCaptureMode


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL, RELAXED])
@pytest.mark.parametrize("same_thread", [True, False])
def test_create_beside_a_capture(mode, same_thread):
    ge.Context.create(0).close()  # the library's code is loaded
    hip = C.CDLL("libamdhip64.so")
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    made = []

    def make():
        try:
            made.append(ge.Context.create(0))
        except ge.GemmaEmbedError as e:
            made.append(e)

    assert hip.hipStreamBeginCapture(stream, mode) == 0
    if same_thread:
        make()
    else:
        t = threading.Thread(target=make)
        t.start()
        t.join()
    ended = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert isinstance(made[0], ge.Context), made
    assert ended == 0
    hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(stream)
    made[0].close()
