"""Graph replays around the length where a chain of kernels stops being replayed as its launches:
every replay against the eager result with eager work between, and destroy waiting for the last
replay."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernels", [1, 2, 6, 7, 10, 11, 12, 13, 40])
def test_chain_lengths(gpu, kernels):
    print(f"graph chain of {kernels} kernels", flush=True)
    st = gpu.Stream()
    n = 4096
    x = gpu.DeviceBuffer.from_array(np.linspace(-8, 8, n, dtype=np.float32))
    outs = [gpu.DeviceBuffer.empty((n,), np.int8) for _ in range(kernels)]

    def record():
        for i, o in enumerate(outs):
            gpu.srq_quantize(x, o, n, 0.05 * (i + 1), stream=st.handle)

    g = gpu.Graph(st, record)
    for rep in range(3):
        xs = np.linspace(-8 - rep, 8 + rep, n, dtype=np.float32)
        x.upload(xs)
        for o in outs:
            o.fill(0x7B, st.handle)  # eager work between replays
        g.launch()
        st.synchronize()
        for i, o in enumerate(outs):
            s = np.float32(0.05 * (i + 1))
            want = np.clip(np.rint(xs / s), -128, 127).astype(np.int8)
            assert np.array_equal(o.download(), want), (rep, i)
    g.close()
    st.close()


@pytest.mark.parametrize("kernels", [4, 20])
def test_destroy_waits_for_the_last_replay(gpu, kernels):
    print(f"graph of {kernels} fills destroyed right after its launch", flush=True)
    st, other = gpu.Stream(), gpu.Stream()
    n = 64 << 20
    b = gpu.DeviceBuffer.empty((n,), np.uint8)
    b.fill(0)
    gpu.synchronize()
    g = gpu.Graph(st, lambda: [b.fill(i + 1, st.handle) for i in range(kernels)])
    g.launch()
    g.close()
    got = b.download(other.handle)  # another stream: only the destroy's wait orders this read
    assert np.all(got == kernels)
    st.close()
    other.close()


@pytest.mark.parametrize("kernels", [1, 6, 20])
def test_destroy_orders_host_memory(gpu, kernels):
    # the graph writes pinned host memory; after the destroy the host reads it with no other wait
    print(f"graph of {kernels} fills of host memory destroyed right after its launch", flush=True)
    st = gpu.Stream()
    n = 8 << 20
    host = ctypes.c_void_p()
    gpu._check(gpu.lib().g4_host_alloc(ctypes.byref(host), n))
    seen = np.ctypeslib.as_array(ctypes.cast(host, ctypes.POINTER(ctypes.c_uint8)), (n,))
    try:
        for rep in range(3):
            seen[:] = 0
            g = gpu.Graph(st, lambda: [gpu._check(gpu.lib().g4_fill_u8(host, i + 1, n, st.handle))
                                       for i in range(kernels)])
            g.launch()
            g.close()
            assert np.all(seen == kernels), rep
    finally:
        st.synchronize()
        gpu.lib().g4_host_free(host)
        st.close()


@pytest.mark.parametrize("kernels", [6, 7, 10, 11])
def test_replay_behind_its_own_running_replay(gpu, kernels):
    # launched again while it runs (as kernel launches), and after it was waited for (as a graph launch)
    print(f"graph chain of {kernels} kernels, replays in flight", flush=True)
    st = gpu.Stream()
    n = 16 << 20
    b = gpu.DeviceBuffer.empty((n,), np.uint8)
    outs = [gpu.DeviceBuffer.empty((4096,), np.int8) for _ in range(kernels - 1)]
    x = gpu.DeviceBuffer.from_array(np.linspace(-8, 8, 4096, dtype=np.float32))

    def record():
        b.fill(kernels, st.handle)  # long enough that the next launch finds it running
        for i, o in enumerate(outs):
            gpu.srq_quantize(x, o, 4096, 0.05 * (i + 1), stream=st.handle)

    g = gpu.Graph(st, record)
    want = [np.clip(np.rint(np.linspace(-8, 8, 4096, dtype=np.float32) / np.float32(0.05 * (i + 1))), -128, 127)
            for i in range(kernels - 1)]
    for rep in range(4):
        for o in outs + [b]:
            o.fill(0x7B, st.handle)
        for _ in range(1 + 3 * (rep % 2)):
            g.launch()
        st.synchronize()
        assert np.all(b.download() == kernels), rep
        for o, w in zip(outs, want):
            assert np.array_equal(o.download(), w.astype(np.int8)), rep
    g.close()
    st.close()


@pytest.mark.parametrize("kernels", [3, 8, 20])
def test_replay_leaves_a_capture_of_the_thread_alone(gpu, kernels):
    # a graph launched on another stream while this thread captures: the capture ends as usual
    print(f"graph of {kernels} kernels launched during a capture", flush=True)
    st, cap = gpu.Stream(), gpu.Stream()
    x = gpu.DeviceBuffer.from_array(np.linspace(-8, 8, 4096, dtype=np.float32))
    outs = [gpu.DeviceBuffer.empty((4096,), np.int8) for _ in range(kernels)]
    mine = gpu.DeviceBuffer.empty((4096,), np.int8)
    g = gpu.Graph(st, lambda: [gpu.srq_quantize(x, o, 4096, 0.05, stream=st.handle) for o in outs])
    g.launch()

    def record():
        gpu.srq_quantize(x, mine, 4096, 0.1, stream=cap.handle)
        for _ in range(3):
            g.launch()

    h = gpu.Graph(cap, record)
    h.launch()
    cap.synchronize()
    st.synchronize()
    xs = np.linspace(-8, 8, 4096, dtype=np.float32)
    assert np.array_equal(mine.download(), np.clip(np.rint(xs / np.float32(0.1)), -128, 127).astype(np.int8))
    for o in outs:
        assert np.array_equal(o.download(), np.clip(np.rint(xs / np.float32(0.05)), -128, 127).astype(np.int8))
    for s in (h, g, st, cap):
        s.close()
