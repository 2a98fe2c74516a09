"""The activation snap's quotient on every kind of scale, through the kernels that snap in bulk (the
small-M kernel at M = 5, the snap pass of the tile kernel at M = 40): scales inside the range of the
residual steps, at its ends and past them (the dividing path), a negative one, and inputs at and
around every half integer, beyond the clamps, infinite and NaN. Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.05, 0.1, 0.6181102395057678, 2.0 ** -100, 2.0 ** -101, 1e-35, 2.0 ** 100,
                                   3e30, 1e36, -0.05])
@pytest.mark.parametrize("bits,m", [(4, 5), (8, 5), (4, 40), (8, 40)])
def test_snap_scales(gpu, oracle, scale, bits, m):
    print(f"snap scale={scale} bits={bits} m={m}", flush=True)
    g = np.random.default_rng(11)
    k, n = 512, 19
    s = np.float32(scale)
    h = (np.arange(m * k) % 263 - 131).astype(np.float64) + 0.5
    with np.errstate(over="ignore"):
        x = (h * float(s)).astype(np.float32)
    ulps = (np.arange(m * k) // 263 % 7 - 3).astype(np.int32)
    x = (x.view(np.int32) + np.where(np.isfinite(x), ulps, 0)).view(np.float32).reshape(m, k)
    x[0, :6] = [np.inf, -np.inf, np.nan, 0.0, -0.0, np.float32(1e-45)]
    x[1, :3] = [np.float32(3e38), np.float32(-3e38), s]
    w = g.integers(0, 256, (n, k * bits // 8), dtype=np.uint8)
    ws = g.uniform(0.005, 0.02, n).astype(np.float32)
    _, acc, _ = oracle.qgemm(bits, w, ws, x, n, k, m, float(s), 0.1)
    out = gpu.DeviceBuffer.empty((m, n), np.int32)
    out.fill(0x7B)
    gpu.qgemm(bits, gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(ws),
              gpu.DeviceBuffer.from_array(x), out, k, n, m, float(s), 0.1)
    assert np.array_equal(out.download(), acc)


@pytest.mark.parametrize("m,n,k", [(3, 16, 256), (17, 6144, 256), (32, 256, 6144), (31, 40, 1536), (16, 6144, 1536),
                                   (12, 1536, 6144), (24, 4097, 1280)])
@pytest.mark.parametrize("xdt", [np.float32, np.float16])
def test_small_m_fused_and_passed_snap(gpu, oracle, m, n, k, xdt):
    # both sides of the rule that moves the snap into a pass of its own, ragged rows and columns
    print(f"small m={m} n={n} k={k} {np.dtype(xdt)}", flush=True)
    g = np.random.default_rng(m * n + k)
    x = g.standard_normal((m, k)).astype(xdt)
    w = g.integers(0, 256, (n, k // 2), dtype=np.uint8)
    ws = g.uniform(0.005, 0.02, n).astype(np.float32)
    _, acc, _ = oracle.qgemm(4, w, ws, x.astype(np.float32), n, k, m, 0.05, 0.1)
    out = gpu.DeviceBuffer.empty((m, n), np.int32)
    out.fill(0x7B)
    gpu.qgemm(4, gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(ws),
              gpu.DeviceBuffer.from_array(x), out, k, n, m, 0.05, 0.1)
    assert np.array_equal(out.download(), acc)
