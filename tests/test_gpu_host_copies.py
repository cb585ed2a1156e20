"""Host-pointer calls on both sides of the size up to which x and y go through
pinned memory (256 KB each), with odd byte counts, repeated calls with other
inputs, and several calls sharing the pinned memory: the same bits as the
device-pointer call."""
import numpy as np
import pytest

import oracle as O
import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,o,k", [(1, 1, 128), (1, 7, 256), (3, 129, 128), (32, 300, 4096), (33, 300, 4096),
                                   (64, 2048, 128), (65, 2048, 128), (65, 2048, 2048), (5, 33, 77)])
def test_matches_device_call(ghip, m, o, k):
    rng = np.random.default_rng(m * 7919 + o)
    for _ in range(3):
        codes = rng.integers(0, 254, (o, k), dtype=np.uint8)
        codes[codes >= 0x7F] += 1
        scales = np.exp2(rng.uniform(-13, -7, ((o + 127) // 128, (k + 127) // 128))).astype(np.float32)
        x = O.f32_to_bf16(rng.standard_normal((m, k)).astype(np.float32))
        y = np.empty(m * o + 8, np.uint16)
        y[m * o:] = 0xABCD
        assert ghip.apus_ghip_fp8blk_linear(O.ptr(codes), O.ptr(scales), O.ptr(x), O.ptr(y), m, o, k) == 0
        dc, ds, dx, dy = G.dev(codes), G.dev(scales), G.dev(x), G.empty(m * o * 2)
        assert ghip.apus_ghip_fp8blk_linear_dev(G.vp(dc), G.vp(ds), G.vp(dx), G.vp(dy), m, o, k, 0,
                                                G.stream()) == 0
        assert np.array_equal(y[:m * o].reshape(m, o), G.host(dy, np.uint16, (m, o)))
        assert (y[m * o:] == 0xABCD).all()
