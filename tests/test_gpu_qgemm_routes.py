"""The kernels of M > 2 and the rules between them, at their edges: the small-M kernel's block rows and
column tiles, the strips, the tile kernel's 32- and 64-row forms, rings and K split, and the tall tiles.
Ragged rows and columns, K of odd and even stage counts, both weight widths, every input and output kind,
against the oracle; each test asserts the kernel it is about."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,m,n,k", [
    (4, 33, 256, 512), (4, 63, 257, 1536), (4, 64, 2048, 1536), (4, 64, 2049, 1536),   # 256 / 258 blocks
    (4, 96, 1365, 2048), (4, 97, 1365, 2048), (4, 500, 250, 1536), (4, 64, 40, 2304),
    (4, 130, 1000, 768), (4, 100, 1500, 1024), (4, 256, 1530, 1280), (4, 40, 6100, 1536),  # tile, 6..12 stages
    (8, 33, 17, 512), (8, 64, 256, 1536), (8, 128, 999, 896), (8, 300, 700, 1152), (8, 1030, 70, 640),
    (8, 512, 1024, 1536), (8, 513, 1024, 768),  # 32 and 34 blocks on one XCD
])
def test_routes(gpu, oracle, bits, m, n, k):
    check_every_kind(gpu, oracle, bits, m, n, k)


def check_every_kind(gpu, oracle, bits, m, n, k):
    print(f"routes bits={bits} m={m} n={n} k={k} {gpu.kernel_for_shape(bits, m, n, k)}", flush=True)
    g = np.random.default_rng(m + n + k)
    x = g.standard_normal((m, k)).astype(np.float16)
    w = g.integers(0, 256, (n, k * bits // 8), dtype=np.uint8)
    s = (g.uniform(0.5, 1.5, n) / (np.sqrt(k) * (4.6 if bits == 4 else 73.6))).astype(np.float32)
    want, acc, codes = oracle.qgemm(bits, w, s, x.astype(np.float32), n, k, m, 0.05, 0.1)
    xq = np.clip(np.rint(x.astype(np.float32) / np.float32(0.05)), -128, 127).astype(np.int8)
    dw, ds = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(s)
    for xin in (x, x.astype(np.float32), xq):
        dx = gpu.DeviceBuffer.from_array(xin)
        for dt, ref in ((np.int32, acc), (np.int8, codes), (np.float32, want)):
            out = gpu.DeviceBuffer.empty((m, n), dt)
            out.fill(0x7B)
            gpu.qgemm(bits, dw, ds, dx, out, k, n, m, 0.05, 0.1)
            got = out.download()
            assert np.array_equal(got.view(np.uint8), np.asarray(ref, dt).reshape(m, n).view(np.uint8)), (xin.dtype, dt)


@pytest.mark.parametrize("bits,m,n,k", [
    (4, 16, 4096, 256), (4, 16, 4097, 512), (4, 5, 8193, 512), (4, 16, 12289, 256), (4, 9, 9001, 3328),
    (4, 17, 4099, 1536), (4, 32, 8200, 1536), (4, 31, 16500, 256), (8, 32, 4100, 384), (8, 12, 8300, 3200),
    # 23 column tiles by 22 block rows: two tiles per block would be 264 blocks
    (8, 697, 366, 128), (4, 700, 360, 2048), (8, 697, 361, 2176), (4, 1640, 140, 2048), (8, 1700, 140, 2048),
    (8, 20, 16729, 256), (8, 29, 18921, 384), (8, 513, 2048, 128), (8, 52, 3697, 3200), (8, 52, 3697, 3072),
    (8, 20, 17000, 128), (8, 512, 1537, 128), (8, 513, 1600, 128), (8, 31, 16385, 128), (4, 64, 3071, 768), (4, 40, 4096, 2304), (4, 100, 1500, 2048),
])
def test_column_tiles(gpu, oracle, bits, m, n, k):
    # 16-wave blocks of one, two and four column tiles and the 4-wave blocks, either side of each line
    check_every_kind(gpu, oracle, bits, m, n, k)


@pytest.mark.parametrize("m,n,k", [(2048, 6144, 512), (2047, 6137, 768), (1793, 5953, 512), (4096, 6144, 512)])
@pytest.mark.parametrize("xdt", [np.float16, np.int8])
def test_tall_tiles(gpu, m, n, k, xdt):
    kind = gpu.KIND_F16 if xdt == np.float16 else gpu.KIND_I8
    assert gpu.kernel_for_shape(4, m, n, k, kind) == "qgemm-4bit-mfma-tall"
    # whole rounds of 256 x 192 tiles: full tiles, ragged last rows and columns (odd N: the stores fall
    # back to single outputs), two rounds; 4 and 6 K stages
    print(f"tall m={m} n={n} k={k} x={np.dtype(xdt)}", flush=True)
    g = np.random.default_rng(m + n)
    w = g.integers(0, 256, (n, k // 2), dtype=np.uint8)
    s = g.uniform(0.005, 0.02, n).astype(np.float32)
    x = g.standard_normal((m, k)).astype(np.float16)
    xq = np.clip(np.rint(x.astype(np.float32) / np.float32(0.05)), -128, 127)
    wc = np.empty((n, k), np.float32)
    wc[:, 0::2], wc[:, 1::2] = w & 15, w >> 4
    # |sum| <= 512 x 8 x 128 x 1.5 < 2^24: float32 products and sums are exact in any order
    acc = xq.astype(np.float32) @ (wc - 8).T
    y = (np.float32(0.05) * s)[None, :] * acc
    q = np.clip(np.rint(y / np.float32(0.1)), -128, 127)
    dw, ds = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(s)
    dx = gpu.DeviceBuffer.from_array(x if xdt == np.float16 else xq.astype(np.int8))
    for dt, ref in ((np.int32, acc), (np.int8, q), (np.float32, q * np.float32(0.1))):
        out = gpu.DeviceBuffer.empty((m, n), dt)
        out.fill(0x7B)
        gpu.qgemm(4, dw, ds, dx, out, k, n, m, 0.05, 0.1)
        assert np.array_equal(out.download(), ref.astype(dt)), dt


@pytest.mark.parametrize("bits,m,n,k", [
    # strips of 64 rows x 32, 48 and 64 columns, either side of one per CU; ragged row tiles (M % 16 of 1,
    # 15 and 0), ragged columns, fewer stages than waves, and 1 .. 6 stages per wave with a remainder
    (4, 33, 8192, 512), (4, 64, 8193, 256), (4, 65, 6145, 768), (4, 129, 4097, 1280), (4, 513, 1363, 2304),
    (4, 1023, 31, 256), (4, 1040, 257, 1024), (4, 177, 1535, 5120), (4, 191, 2700, 6144),
    (8, 1025, 130, 1024), (8, 65, 6145, 1152), (8, 2000, 257, 1024), (8, 143, 1801, 2176),
    # row groups on every second and fourth XCD, and strips in turn
    (4, 281, 2048, 256), (4, 513, 1024, 512), (4, 1132, 884, 512), (8, 1100, 850, 1024),
])
def test_strips(gpu, oracle, bits, m, n, k):
    for kind in (gpu.KIND_F32, gpu.KIND_F16):
        assert gpu.kernel_for_shape(bits, m, n, k, kind).endswith("mfma-strip")
    check_every_kind(gpu, oracle, bits, m, n, k)


@pytest.mark.parametrize("bits,m,n,k", [
    # 64-row tiles on rings of 4 and 3 stages (K of 4 and more stages, and 2), 4-bit codes interleaved by the
    # snap (f16 / f32) and in natural order (int8), 8-bit; ragged last rows and columns
    (4, 200, 6145, 512), (4, 200, 6145, 256), (4, 512, 4001, 768), (8, 512, 6143, 640), (8, 2048, 1537, 256),
    # 32-row tiles that are no strips: one more column than 256 strips of 64
    (4, 512, 2049, 256), (4, 512, 2049, 1280), (8, 513, 1024, 256), (8, 500, 2100, 1152),
])
def test_tiles(gpu, oracle, bits, m, n, k):
    for kind in (gpu.KIND_F32, gpu.KIND_F16, gpu.KIND_I8):
        assert gpu.kernel_for_shape(bits, m, n, k, kind).endswith("mfma-tile")
    check_every_kind(gpu, oracle, bits, m, n, k)


@pytest.mark.parametrize("bits,m,n,k", [
    # 16-row blocks past 16 rows, either side of one block per CU; ragged last rows and columns; f32 that is
    # snapped in a pass of its own (1024 x 1536)
    (4, 17, 2048, 512), (4, 17, 2049, 256), (4, 31, 1536, 6400), (4, 33, 1361, 1536), (4, 49, 1024, 768),
    (4, 250, 255, 1536), (4, 257, 240, 2304), (4, 1024, 121, 1536), (8, 18, 1536, 128), (8, 32, 257, 1536), (8, 100, 500, 6400),
])
def test_sixteen_row_blocks(gpu, oracle, bits, m, n, k):
    assert "small" in gpu.kernel_for_shape(bits, m, n, k, gpu.KIND_F16)
    check_every_kind(gpu, oracle, bits, m, n, k)


@pytest.mark.parametrize("bits,m,n,k,xdt", [
    # fewer than 48 Ki snaps on a CU: one launch with no codes buffer
    (4, 32, 2048, 1536, np.float16), (4, 17, 1536, 2048, np.float16), (4, 28, 2048, 2048, np.float32),
    # calls that snap in a pass of their own once a buffer is there
    (4, 1024, 256, 2048, np.float32), (8, 1024, 121, 1536, np.float32), (4, 697, 361, 2048, np.float16),
    (8, 697, 361, 2048, np.float32),
])
def test_first_call_inside_a_capture(gpu, bits, m, n, k, xdt):
    print(f"captured first call bits={bits} m={m} n={n} k={k}", flush=True)
    g = np.random.default_rng(m)
    x = gpu.DeviceBuffer.from_array(g.standard_normal((m, k)).astype(xdt))
    w = gpu.DeviceBuffer.from_array(g.integers(0, 256, (n, k * bits // 8), dtype=np.uint8))
    s = gpu.DeviceBuffer.from_array(g.uniform(0.005, 0.02, n).astype(np.float32))
    out, want = (gpu.DeviceBuffer.empty((m, n), np.int32) for _ in range(2))
    st = gpu.Stream()
    graph = gpu.Graph(st, lambda: gpu.qgemm(bits, w, s, x, out, k, n, m, 0.05, 0.1, stream=st.handle))
    gpu.qgemm(bits, w, s, x, want, k, n, m, 0.05, 0.1)
    for _ in range(3):
        out.fill(0x7B, st.handle)
        graph.launch()
        st.synchronize()
        assert np.array_equal(out.download(), want.download())
    graph.close()
    st.close()


def test_noalloc_past_its_scratch(gpu):
    # 12 Mi activation codes: more than the static array holds, served in one launch that needs none
    m, n, k = 8192, 16, 1536
    assert m * k > gpu.lib().g4_qgemm_noalloc_max_codes()
    print(f"noalloc m={m} n={n} k={k} f32", flush=True)
    g = np.random.default_rng(5)
    x = gpu.DeviceBuffer.from_array(g.standard_normal((m, k)).astype(np.float32))
    w = gpu.DeviceBuffer.from_array(g.integers(0, 256, (n, k // 2), dtype=np.uint8))
    s = gpu.DeviceBuffer.from_array(g.uniform(0.005, 0.02, n).astype(np.float32))
    outs = [gpu.DeviceBuffer.empty((m, n), np.int32) for _ in range(2)]
    for fn, o in zip((gpu.qgemm_noalloc, gpu.qgemm), outs):
        o.fill(0x7B)
        fn(4, w, s, x, o, k, n, m, 0.05, 0.1)
    assert np.array_equal(outs[0].download(), outs[1].download())
