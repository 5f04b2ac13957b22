"""Vectors small enough to travel in a launch's arguments and to come back through a window of pinned memory: the bytes, the
order with the launches round them, and what else may read a device block."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# out[i] = 2 v[i] + 1
KERNEL = ("(kernel sarek_kern (params (param (var v 1 (vec f32))) (param (var out 2 (vec f32))) (param (var n 3 i32))) (locals) "
          "(body (let (var tid 4 i32) (intr (Std) global_thread_id) (if (lt (var tid 4 i32) (var n 3 i32)) "
          "(assign (lelem out (var tid 4 i32)) (add (mul (read v (var tid 4 i32)) (f32 2.0)) (f32 1.0)))))) (native_fn true))")


@pytest.fixture()
def sarek(hip, torch_cuda):
    from spoc_amd import sarek as s
    s.Device.init()
    return s


def launch(s, v, out):
    n = v.length
    s.Execute.run_vectors(ir=KERNEL, args=[s.Execute.Vec(v), s.Execute.Vec(out), s.Execute.Int(n)],
                          block=s.Execute.dims1d(256), grid=s.Execute.dims1d((n + 255) // 256))


@pytest.mark.parametrize("small", [1, 0])
@pytest.mark.parametrize("size,count", [(1, 1), (1, 3), (3, 341), (1, 1023), (1, 1024), (1, 1025), (3, 1023), (4, 256), (4, 257),
                                        (4, 767), (4, 768), (4, 769), (1, 3071), (8, 384), (16, 192)])
def test_bytes_of_every_length(hip, sarek, small, size, count):
    """Up and down again, elements of 1 to 16 bytes, lengths round the two payloads and past them, small path on and off."""
    rng = np.random.default_rng(size * 10000 + count)
    hip.set_tunable("transfer.small", small)
    try:
        v = sarek.Vector.create_custom(size, count)
        for _ in range(3):
            data = rng.integers(0, 256, size * count, dtype=np.uint8)
            v.host.view(np.uint8).reshape(-1)[:] = data
            hip.check(hip.lib.sarek_hip_vector_write(v._h, C.c_void_p(data.ctypes.data), 0, count))
            sarek.Transfer.to_device(v)
            v.host.view(np.uint8).reshape(-1)[:] = 0
            sarek.Transfer.to_cpu(v, force=True)
            assert np.array_equal(v.host.view(np.uint8).reshape(-1), data)
    finally:
        hip.set_tunable("transfer.small", 1)


@pytest.mark.parametrize("n", [1, 255, 256, 300, 768, 769])
def test_each_launch_sees_the_host_data_of_its_time(sarek, n):
    """Host blocks are written again right behind their launches, many in a row without a wait: every result is of the data
    that was there when its launch was asked for."""
    outs = [sarek.Vector.create(sarek.Vector.float32, n) for _ in range(50)]
    ins = [sarek.Vector.create(sarek.Vector.float32, n) for _ in outs]
    for i, (v, out) in enumerate(zip(ins, outs)):
        v.fill_from(np.arange(n, dtype=np.float32) + i)
        launch(sarek, v, out)
        v.host[:] = -1
    for i, out in enumerate(outs):
        assert np.array_equal(out.to_array(), 2 * (np.arange(n, dtype=np.float32) + i) + 1)


def test_a_block_whose_address_is_known_is_complete(hip, torch_cuda, sarek):
    """Another stream reads a vector's block right after the address was handed out, and right after an upload from then on."""
    torch = torch_cuda
    side = torch.cuda.Stream()
    x = torch.randn(4096, 4096, device="cuda")
    for _ in range(5):
        v = sarek.Vector.create(sarek.Vector.float32, 256)
        v.fill_from(np.full(256, 3.0, np.float32))
        hip.gemm_f32(x, x)                       # the default stream is busy while the upload is queued behind it
        sarek.Transfer.to_device(v)
        got = torch.empty(256, device="cuda")
        for want in (3.0, 4.0):
            ptr = v.device_ptr
            with torch.cuda.stream(side):
                got.copy_(torch.as_tensor(_Block(ptr, 256), device="cuda"))
            side.synchronize()
            assert bool((got == want).all())
            v.fill_from(np.full(256, 4.0, np.float32))
            hip.gemm_f32(x, x)
            sarek.Transfer.to_device(v)


class _Block:
    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=(n,), typestr="<f4", strides=None, version=2)


def test_a_download_behind_long_work(hip, torch_cuda, sarek):
    """Work that outlasts the look for the mark: the download waits for the stream."""
    torch = torch_cuda
    x = torch.randn(4096, 4096, device="cuda")
    for i in range(3):
        v, out = sarek.Vector.create(sarek.Vector.float32, 256), sarek.Vector.create(sarek.Vector.float32, 256)
        v.fill_from(np.full(256, i, np.float32))
        for _ in range(10):
            hip.gemm_f32(x, x)                   # some 9 ms
        launch(sarek, v, out)
        assert np.array_equal(out.to_array(), np.full(256, 2 * i + 1, np.float32))


def test_threads_with_vectors_of_their_own(sarek):
    """Four threads upload, launch and read small vectors at once; one of them at a time has the window."""
    wrong = []

    def work(t):
        v, out = (sarek.Vector.create(sarek.Vector.float32, 200 + t) for _ in range(2))
        for i in range(100):
            v.to_array()
            v.fill_from(np.full(200 + t, 1000 * t + i, np.float32))
            launch(sarek, v, out)
            if not np.array_equal(out.to_array(), np.full(200 + t, 2 * (1000 * t + i) + 1, np.float32)):
                wrong.append((t, i))
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("mode", [0, 1, 2])              # hipStreamCaptureModeGlobal, ThreadLocal, Relaxed
@pytest.mark.parametrize("small", [1, 0])
def test_refused_while_a_stream_is_captured(hip, sarek, small, mode):
    """A copy is an error while a stream is captured, and spoils the capture; a small one by whatever way it travels, up as
    down, on device blocks that are there already.  Afterwards both work."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    runtime = C.CDLL(path)
    hip.set_tunable("transfer.small", small)
    try:
        up, down, fresh = (sarek.Vector.create(sarek.Vector.float32, 256) for _ in range(3))
        for v in (up, down, fresh):
            v.fill_from(np.full(256, 2.0, np.float32))
            sarek.Transfer.to_device(v)
        sarek.Transfer.to_cpu(fresh, force=True)          # the window for downloads is there
        up.fill_from(np.full(256, 3.0, np.float32))
        for blocking in (True, False):
            for copy in (lambda: sarek.Transfer.to_device(up), lambda: sarek.Transfer.to_cpu(down, force=True)):
                stream, graph = C.c_void_p(), C.c_void_p()
                assert runtime.hipStreamCreateWithFlags(C.byref(stream), 0 if blocking else 1) == 0
                assert runtime.hipStreamBeginCapture(stream, mode) == 0
                try:
                    with pytest.raises(hip.SarekHipError, match="Capture"):
                        copy()
                finally:
                    ended = runtime.hipStreamEndCapture(stream, C.byref(graph))
                    runtime.hipGetLastError()
                    assert runtime.hipStreamDestroy(stream) == 0
                assert ended == 901 and not graph.value   # hipErrorStreamCaptureInvalidated
        sarek.Transfer.to_device(up)
        up.host[:] = 0
        sarek.Transfer.to_cpu(up, force=True)
        assert np.array_equal(up.host, np.full(256, 3.0, np.float32))
    finally:
        hip.set_tunable("transfer.small", 1)
