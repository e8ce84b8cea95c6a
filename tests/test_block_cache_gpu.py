"""Kept device blocks (mx_malloc / mx_free without a stream) on the GPU; the
rules themselves run on the CPU in test_block_cache.py."""
import ctypes as C
import threading

import pytest

import kokkos_amd as K

pytestmark = pytest.mark.gpu

MiB = 1 << 20


def alloc(rt, size):
    p = C.c_void_p()
    K.check(rt.mx_malloc(C.byref(p), size, None))
    return p


def test_free_leaves_a_capture_elsewhere_alone(paths):
    """Blocks are freed and allocated while another thread records a stream:
    the recording ends well, and its graph runs."""
    rt = K.load("kkmx_rt")
    stream, graph, ex = C.c_void_p(), C.c_void_p(), C.c_void_p()
    K.check(rt.mx_stream_create(C.byref(stream)))
    a, b = alloc(rt, MiB), alloc(rt, 300 * MiB)
    codes = []

    def elsewhere():
        codes.append(rt.mx_free(a, None))
        codes.append(rt.mx_free(b, None))
        p = C.c_void_p()
        codes.append(rt.mx_malloc(C.byref(p), C.c_size_t(2 * MiB), None))
        codes.append(rt.mx_free(p, None))

    K.check(rt.mx_graph_capture_begin(stream))
    t = threading.Thread(target=elsewhere)
    t.start()
    t.join()
    K.check(rt.mx_graph_capture_end(stream, C.byref(graph)))
    assert codes == [0, 0, 0, 0]
    K.check(rt.mx_graph_instantiate(C.byref(ex), graph))
    K.check(rt.mx_graph_launch(ex, stream))
    K.check(rt.mx_stream_sync(stream))
    K.check(rt.mx_graph_exec_destroy(ex))
    K.check(rt.mx_graph_destroy(graph))
    K.check(rt.mx_stream_destroy(stream))
