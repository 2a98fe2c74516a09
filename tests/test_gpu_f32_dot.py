"""The uncalibrated f32 code dot (inScale 0) at the edges of its kernel: K around whole slabs and
chunks per lane, rows around the 4-row groups and the 16-group runs, one and two columns, f32 and
f16 activations. The result is held to 64-bit sums, and a column's bits must not depend on how many
columns share the launch."""
import numpy as np
import pytest

import npref

pytestmark = pytest.mark.gpu


def dev(g4, a):
    return g4.DeviceBuffer.from_array(np.ascontiguousarray(a))


def out_buf(g4, shape):
    b = g4.DeviceBuffer.empty(shape, np.float32)
    b.fill(0x7B)
    return b


@pytest.mark.parametrize("bits,k,n", [
    (4, 256, 1), (4, 512, 3), (4, 768, 67), (4, 1536, 5), (4, 1792, 64), (4, 16384, 21),
    (8, 128, 2), (8, 1024, 66), (8, 1152, 9), (8, 1536, 130), (8, 16384, 7),
    (4, 256, 12288), (8, 128, 12289),  # the last that runs its columns apart, the first together (256 CUs)
    (4, 1536, 13000),   # two groups per wave
    (4, 256, 200003),   # more than one 16-group run per wave
])
@pytest.mark.parametrize("xdt", [np.float32, np.float16])
def test_f32_code_dot(gpu, bits, k, n, xdt):
    print(f"f32 dot bits={bits} k={k} n={n} x={np.dtype(xdt)}", flush=True)
    g = np.random.default_rng(k + n)
    w = g.integers(0, 256, (n, k * bits // 8), dtype=np.uint8)
    s = g.uniform(0.005, 0.02, n).astype(np.float32)
    x = g.standard_normal((2, k)).astype(xdt)
    dw, ds = dev(gpu, w), dev(gpu, s)
    o2 = out_buf(gpu, (2, n))
    gpu.qgemv(bits, dw, ds, dev(gpu, x), o2, k, n, 2, 0.0, 0.0)
    got = o2.download()
    codes = npref.codes(bits, w).astype(np.float64)
    xd = x.astype(np.float64)
    # K products of one rounding each and K additions, in any order, then the scale's rounding
    tol = (2.0 * k + 2) * 2.0 ** -24 * (np.abs(xd) @ np.abs(codes).T) * s
    assert np.all(np.abs(got - (xd @ codes.T) * s) <= tol)
    for c in range(2):
        o1 = out_buf(gpu, (n,))
        gpu.qgemv(bits, dw, ds, dev(gpu, x[c]), o1, k, n, 1, 0.0, 0.0)
        assert np.array_equal(o1.download().view(np.uint32), got[c].view(np.uint32))


@pytest.mark.parametrize("bits", [4, 8])
def test_f32_code_dot_infinities(gpu, bits):
    # K past a whole slab: the padded lanes must not turn an infinity's row into NaN
    k, n = 2048 + 256, 10
    g = np.random.default_rng(7)
    w = g.integers(0, 256, (n, k * bits // 8), dtype=np.uint8)
    s = np.full(n, 0.01, np.float32)
    x = g.standard_normal((1, k)).astype(np.float32)
    x[0, -1] = np.inf
    o = out_buf(gpu, (n,))
    gpu.qgemv(bits, dev(gpu, w), dev(gpu, s), dev(gpu, x[0]), o, k, n, 1, 0.0, 0.0)
    last = npref.codes(bits, w)[:, -1].astype(np.float32)
    with np.errstate(invalid="ignore"):
        want = last * np.float32(np.inf)
    got = o.download()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(want)], want[~np.isnan(want)])
