"""Kept device blocks (mx_malloc / mx_free without a stream) on the GPU; the
rules themselves run on the CPU in test_block_cache.py."""
import ctypes as C
import threading

import numpy as np
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


def test_free_waits_for_queued_work(paths):
    """A block is freed while kernels that write it are still queued on a
    second stream, and taken again: its new content is the new owner's."""
    P, rt = paths, K.load("kkmx_rt")
    n = 16 * MiB  # doubles
    K.check(rt.mx_trim())
    a = alloc(rt, n * 8)
    K.check(P.kkmx_deep_fill_f64(a, n, 1.0), P)
    for _ in range(200):  # about 10 ms of kernels over the block, in place
        K.check(P.kkmx_stream_scale(a, a, n, 1.0), P)
    done = C.c_void_p()
    K.check(rt.mx_event_create(C.byref(done)))
    K.check(rt.mx_event_record(done, C.c_void_p(P.kkmx_stream())))
    assert rt.mx_event_query(done) != 0  # still at work
    K.check(rt.mx_free(a, None))
    assert rt.mx_event_query(done) == 0
    b = alloc(rt, n * 8)
    assert b.value == a.value
    other = C.c_void_p()
    K.check(rt.mx_stream_create(C.byref(other)))
    K.check(rt.mx_memset_async(b, 0, n * 8, other))
    K.check(rt.mx_stream_sync(other))
    K.fence()
    got = np.empty(n)
    K.check(rt.mx_memcpy(got.ctypes.data, b, n * 8))
    assert not got.any()
    K.check(rt.mx_free(b, None))
    K.check(rt.mx_event_destroy(done))
    K.check(rt.mx_stream_destroy(other))


def test_impossible_request_and_second_free(paths):
    rt = K.load("kkmx_rt")
    for n in (2**64 - 1, 2**64 - 43, 2**64 - 65536, 1 << 60):
        p = C.c_void_p(1)
        assert rt.mx_malloc(C.byref(p), C.c_size_t(n), None) != 0
        assert not p.value
        rt.mx_get_last_error()
    a = alloc(rt, 3 * MiB)
    K.check(rt.mx_free(a, None))
    assert rt.mx_free(a, None) != 0
    b = alloc(rt, 3 * MiB)
    assert b.value == a.value
    K.check(rt.mx_free(b, None))
    K.check(rt.mx_trim())
