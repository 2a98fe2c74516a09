"""Decode attention at the edges of its matrix-core products, bit for bit against the restatement:
fewer than eight heads, a last chunk of 1, 31 or 32 positions, one and two halves per block (grids
up to and past the CU count), values whose products are subnormal, and cache rows past the position
that hold NaN and infinities (read as stand-ins, never used)."""
import numpy as np
import pytest

import decode_oracle as d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("rows,pos", [(2, 0), (2, 62), (2, 63), (2, 64), (9, 990), (9, 1023)])
@pytest.mark.parametrize("tiny", [False, True])
def test_attention_heads_and_tails(gpu, heads, rows, pos, tiny):
    print(f"attention heads={heads} rows={rows} pos={pos} tiny={tiny}", flush=True)
    L = gpu.lib()
    rng = np.random.default_rng(1000 * heads + pos + rows)
    hd, cap, ins = 256, 1024 + 40, 0.05
    scale = np.float32(2.0 ** -70) if tiny else np.float32(1.0)
    q = (rng.standard_normal((rows, heads, hd)) * 0.25).astype(np.float32) * scale
    kv = rng.uniform(-1.7, 1.7, (rows, 2, cap, hd)).astype(np.float32)
    kv[:, 0] *= scale
    if tiny:
        kv[:, 1, ::2] *= np.float32(2.0 ** -126)
    kv[:, :, pos + 1:] = np.array([np.nan, np.inf], np.float32)[rng.integers(0, 2, (rows, 2, cap - pos - 1, hd))]
    dq = gpu.DeviceBuffer.from_array(q)
    dkv = gpu.DeviceBuffer.from_array(kv)
    ws_bytes = L.g4_attention_workspace_bytes(rows, heads, pos, 0)
    ws = gpu.DeviceBuffer(ws_bytes, np.uint8)
    f = gpu.DeviceBuffer.empty((rows, heads, hd), np.float32)
    f.fill(0x7B)
    gpu._check(L.g4_attention_decode(dq.ptr, dkv.ptr, dkv.ptr + cap * hd * 4, 2 * cap * hd, rows, heads,
                                     hd, pos, None, 0, ws.ptr, ws_bytes, ins, None, f.ptr, None))
    got = f.download()
    for r in range(rows):
        want = np.asarray(d.attention_decode(q[r], kv[r, 0], kv[r, 1], pos, 0), np.float32)
        assert np.array_equal(got[r].view(np.uint32), want.view(np.uint32)), r
