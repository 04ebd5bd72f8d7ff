"""Which copy of a mapped buffer is current (cldnn_hip_buffer_map / _unmap / _use): every order of host writes and device
uses gives the bytes written last, also where a kernel reads or writes the host copy in place."""
import ctypes as C
import threading

import numpy as np
import pytest

from cldnn_amd import api as cl
from cldnn_amd import hip

pytestmark = pytest.mark.gpu
READ, READ_ONCE, UPDATE, WRITE, WRITE_FOR_HOST = range(5)


def mapped(buf):
    p = hip.lib().cldnn_hip_buffer_map(buf.h, None)
    assert p
    return np.frombuffer((C.c_uint8 * buf.nbytes).from_address(p), np.uint8)


def copy(eng, src, how_src, dst, how_dst):
    L = hip.lib()
    hip.check(L.cldnn_hip_reorder(eng.h, L.cldnn_hip_buffer_use(src.h, how_src), C.byref(src.tensor),
                                  L.cldnn_hip_buffer_use(dst.h, how_dst), C.byref(dst.tensor)))


@pytest.mark.parametrize("features", [1, 33, 16 * 5000], ids=["one_byte", "few", "beyond_the_in_place_limits"])
@pytest.mark.parametrize("how_src", [READ, READ_ONCE])
@pytest.mark.parametrize("how_dst", [WRITE, UPDATE, WRITE_FOR_HOST])
def test_last_write_wins(features, how_src, how_dst):
    eng, L = hip.Engine(0), hip.lib()
    t = hip.Tensor.make(hip.U8, hip.BFYX, 1, features, 1, 61)
    src, dst = hip.Buffer(eng, t), hip.Buffer(eng, t)
    r = np.random.default_rng(features)
    for turn in range(3):
        data = r.integers(0, 256, src.nbytes, dtype=np.uint8)
        mapped(src)[:] = data
        hip.check(L.cldnn_hip_buffer_unmap(src.h))
        for _ in range(2):  # the second read finds the device copy brought up to date
            copy(eng, src, how_src, dst, how_dst)
        m = mapped(dst)
        assert np.array_equal(m, data)
        m[0] ^= 255  # what the host changes in a result is seen by the next reader on the device
        hip.check(L.cldnn_hip_buffer_unmap(dst.h))
        copy(eng, dst, READ, src, WRITE)
        data[0] ^= 255
        assert np.array_equal(src.read_raw(), data)  # the copies of the plain entry points follow too
        assert np.array_equal(dst.read_raw(), data)
    for b in (src, dst):
        b.close()
    eng.close()


def test_input_rewritten_and_reused_between_runs():
    """one input memory: written once and run twice, then rewritten; two networks share it"""
    eng = cl.engine()
    F, DT = cl.format, cl.data_types
    lay = cl.layout(DT.u8, F.bfyx, cl.tensor(2, 3, 9, 7))
    nets = [cl.network(eng, cl.topology(cl.input_layout("x", lay), cl.reorder("y", "x", f, DT.f32))) for f in (F.bfyx, F.yxfb)]
    r = np.random.default_rng(5)
    mem = cl.memory.allocate(eng, lay)
    for _ in range(3):
        x = r.integers(0, 256, (2, 3, 7, 9), dtype=np.uint8)
        mem.write(x)
        for n in nets + nets:
            n.set_input_data("x", mem)
            assert np.array_equal(n.execute()["y"].get_memory().read(), x.astype(np.float32))
        assert np.array_equal(mem.read(), x)


def in_thread(f):
    t = threading.Thread(target=f, daemon=True)
    t.start()
    return t


def test_buffer_can_be_used_while_a_map_waits_for_its_event():
    eng, L = hip.Engine(0), hip.lib()
    buf = hip.Buffer(eng, hip.Tensor.make(hip.U8, hip.BFYX, 1, 64, 1, 1))
    mapped(buf)[:] = 7
    hip.check(L.cldnn_hip_buffer_unmap(buf.h))
    gate, seen = C.c_void_p(), []
    hip.check(L.cldnn_hip_event_create_user(eng.h, 0, C.byref(gate)))
    waiter = in_thread(lambda: seen.append(L.cldnn_hip_buffer_map(buf.h, gate)))
    waiter.join(0.2)
    assert waiter.is_alive() and not seen
    user = in_thread(lambda: L.cldnn_hip_buffer_use(buf.h, READ))  # as the run behind the gate would
    user.join(20)
    assert not user.is_alive()
    hip.check(L.cldnn_hip_event_set(gate))
    waiter.join(20)
    assert not waiter.is_alive() and seen[0]
    hip.check(L.cldnn_hip_buffer_unmap(buf.h))
    hip.check(L.cldnn_hip_event_release(gate))
    buf.close()
    eng.close()


def test_handler_of_an_output_event_may_lock_the_output():
    """whichever thread sees the end of the run first: the one that locks the output or the one that calls the handler"""
    eng = cl.engine()
    F, DT = cl.format, cl.data_types
    lay = cl.layout(DT.u8, F.bfyx, cl.tensor(8, 16, 64, 64))
    net = cl.network(eng, cl.topology(cl.input_layout("x", lay), cl.reorder("y", "x", F.yxfb, DT.f32), cl.reorder("s", "y", F.bfyx, DT.u8)))
    x = np.random.default_rng(3).integers(0, 256, (8, 16, 64, 64), dtype=np.uint8)
    net.set_input_data("x", cl.make_memory(eng, x))
    got, wrong = [], []

    def rounds():
        for _ in range(40):
            out = net.execute()["s"]
            mem, ev, done = out.get_memory(), out.get_event(), threading.Event()

            def handler(_):
                got.append(np.array_equal(mem.read(), x))
                done.set()

            cb = cl.EVENT_HANDLER(handler)
            cl._call("cldnn_add_event_handler", ev.h, cb, None)
            wrong.append(not np.array_equal(mem.read(), x))
            if not done.wait(20):
                return

    t = in_thread(rounds)
    t.join(60)
    assert not t.is_alive() and got == [True] * 40 and not any(wrong)


def test_large_input_is_copied_from_the_unmap_on():
    """beyond the in-place limit: the device has the bytes before any use asks for them, and a map that follows waits for the
    copy whatever event it is given; a result that was only looked at is not copied back"""
    eng, L = hip.Engine(0), hip.lib()
    t = hip.Tensor.make(hip.U8, hip.BFYX, 1, 1 << 15, 1, 1031)
    src, dst = hip.Buffer(eng, t), hip.Buffer(eng, t)
    on_device = L.cldnn_hip_buffer_use(src.h, READ)  # the same pointer for the buffer's life
    r = np.random.default_rng(2)
    old = C.c_void_p()
    hip.check(L.cldnn_hip_event_record(eng.h, C.byref(old)))
    eng.finish()

    def device_bytes():
        hip.check(L.cldnn_hip_reorder(eng.h, on_device, C.byref(t), L.cldnn_hip_buffer_use(dst.h, WRITE), C.byref(t)))
        return dst.read_raw()

    for _ in range(3):
        data = r.integers(0, 256, src.nbytes, dtype=np.uint8)
        mapped(src)[:] = data
        hip.check(L.cldnn_hip_buffer_unmap(src.h))
        p = L.cldnn_hip_buffer_map(src.h, old)  # an event from before the copy
        C.memset(p, 0x5a, src.nbytes)
        assert np.array_equal(device_bytes(), data)
        hip.check(L.cldnn_hip_buffer_unmap(src.h))
        assert (device_bytes() == 0x5a).all() and (src.read_raw() == 0x5a).all()
    L.cldnn_hip_buffer_use(src.h, WRITE)
    mapped(src)[:] = 1
    hip.check(L.cldnn_hip_buffer_unmap(src.h))
    assert (device_bytes() == 0x5a).all() and (src.read_raw() == 1).all()
    copy(eng, src, READ, dst, WRITE)
    assert (dst.read_raw() == 1).all()
    hip.check(L.cldnn_hip_event_release(old))
    src.close(), dst.close(), eng.close()


def test_unmap_while_the_stream_is_captured_records_nothing():
    eng, L = hip.Engine(0), hip.lib()
    t = hip.Tensor.make(hip.U8, hip.BFYX, 1, 1 << 12, 1, 1031)
    src, dst = hip.Buffer(eng, t), hip.Buffer(eng, t)
    stream = C.c_void_p(L.cldnn_hip_engine_stream(eng.h))
    eng.finish()
    mapped(src)[:] = 0x33
    graph, nodes = C.c_void_p(), C.c_size_t(99)
    assert L.hipStreamBeginCapture(stream, 2) == 0  # relaxed
    status = L.cldnn_hip_buffer_unmap(src.h)
    assert L.hipStreamEndCapture(stream, C.byref(graph)) == 0
    hip.check(status)
    assert L.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 0
    assert L.hipGraphDestroy(graph) == 0
    copy(eng, src, READ, dst, WRITE)
    assert (dst.read_raw() == 0x33).all()
    src.close(), dst.close(), eng.close()


def test_a_failure_of_the_runtime_is_reported_once():
    """by the entry it happened in, not again by the launch behind it: an allocation beyond the device's memory, and a recording that is
    broken off by an allocation, whose launches then go out one by one"""
    eng, L = hip.Engine(0), hip.lib()
    src, dst = (hip.Buffer(eng, hip.Tensor.make(hip.U8, hip.BFYX, 1, 3, 5, 7)) for _ in range(2))
    best, us = C.c_int32(), C.c_float()
    huge = hip.Tensor.make(hip.S8, hip.FS_B_YX_FSV16, 1 << 22, 64, 256, 256)  # 16 TiB
    w = np.ones((64, 64, 1, 1), np.int8)
    desc = hip.conv_desc(huge, w.shape, "s8")
    assert L.cldnn_hip_conv_tune(eng.h, C.byref(desc), w.ctypes.data_as(C.c_void_p), None, None, None, None, 1, C.byref(best), C.byref(us), None, None) != 0
    assert b"hipMalloc" in L.cldnn_hip_last_error()
    hip.check(L.cldnn_hip_buffer_fill(src.h, 1))
    copy(eng, src, READ, dst, WRITE)
    assert (dst.read_raw() == 1).all()

    recording, refused = C.c_void_p(), C.c_void_p()
    hip.check(L.cldnn_hip_engine_record_begin(eng.h))
    copy(eng, src, READ, dst, WRITE)
    assert L.cldnn_hip_buffer_alloc(eng.h, 64, C.byref(refused)) != 0
    assert L.cldnn_hip_engine_record_end(eng.h, C.byref(recording)) != 0 and not recording.value
    hip.check(L.cldnn_hip_buffer_fill(src.h, 2))
    copy(eng, src, READ, dst, WRITE)
    assert (dst.read_raw() == 2).all()
    src.close(), dst.close(), eng.close()
