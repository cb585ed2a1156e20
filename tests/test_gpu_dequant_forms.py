"""The dequant's chunk forms against the oracle, bit for bit: widths that are
and are not whole chunks of 8, chunks that meet a scale block's end, a row's
end or both, partial last chunks, more than one workgroup, addresses that
only the element form takes, and scales that are not finite (whose NaN
products keep their bits)."""
import ctypes

import numpy as np
import pytest

import oracle as O
import gpu_util as G

pytestmark = pytest.mark.gpu


def run(ghip, codes, scales, exact, shift=0):
    o, k = codes.shape
    dc, ds = G.dev(np.concatenate([np.zeros(shift, np.uint8), codes.ravel()])), G.dev(scales)
    out = G.empty(o * k * 2 + 64)
    rc = ghip.apus_ghip_fp8blk_dequant_dev(ctypes.c_void_p(G.vp(dc).value + shift), G.vp(ds),
                                           G.vp(out), o, k, exact, G.stream())
    assert rc == 0
    return G.host(out, np.uint16, (o * k + 32,))[:o * k].reshape(o, k)


def case(o, k, seed):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 256, (o, k), dtype=np.uint8)
    scales = np.exp2(rng.uniform(-14, -4, ((o + 127) // 128, (k + 127) // 128))).astype(np.float32)
    return codes, scales


@pytest.mark.parametrize("o,k", [(1, 1), (3, 7), (5, 8), (1, 9), (300, 9), (129, 15), (7, 24), (131, 127),
                                 (257, 128), (130, 129), (129, 130), (260, 133), (33, 136), (129, 255),
                                 (128, 1999), (4, 2048), (3, 4104), (385, 1536), (1, 4095), (1, 4097)])
@pytest.mark.parametrize("shift", [0, 8, 1])
def test_forms(ghip, o, k, shift):
    codes, scales = case(o, k, o * 10007 + k)
    assert np.array_equal(run(ghip, codes, scales, 1, shift), O.dequant(codes, scales))
    if k % 16 or shift:         # these forms know the NaN codes whatever the flag says
        assert np.array_equal(run(ghip, codes, scales, 0, shift), O.dequant(codes, scales))


@pytest.mark.parametrize("k", [256, 250])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, -np.nan])
def test_scales_not_finite(ghip, k, value):
    codes, scales = case(300, k, 3)
    scales[1, 0] = scales[2, 1] = value
    with np.errstate(invalid="ignore"):
        want = O.dequant(codes, scales)
    got = run(ghip, codes, scales, 1)
    # the sign of a NaN that the product itself makes (inf x 0) is the machine's choice
    made = np.isinf(np.repeat(np.repeat(scales, 128, 0)[:300], 128, 1)[:, :k]) & ((codes & 127) == 0)
    assert np.array_equal(got[~made], want[~made])
    assert ((got[made] & 0x7FFF) > 0x7F80).all()
