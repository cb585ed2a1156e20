"""The SwiGLU clamps (c/gmoe.h:217-222: gate clamped above, up clamped on
both sides, before the silu) at limits tight enough that most g and u
values clamp, through the decode launch (K3) and each form of the prefill
(K4: the weight streams, the queued tiles and the full ones), against the
oracle's per-token loop at the same limit. Each case also checks, with the
oracle's own g and u, that the clamps fire on both sides, and that the
output differs from the one at the default limit, so the store's limit is
the one the kernels use.

Floor: at such limits every h_i sits near +-limit * silu(limit), and each
expert's down GEMM cancels deeply (an output of -0.39 from terms whose
|sum| is 19.8), so a one-ulp step of one h_i -- a legitimate difference of
the GPU's own gate/up GEMM -- moves the combined output by up to
w_e * 2^-8 * sum_i |h_i * wd_i|, which the combine's floor sum_e |contrib_e|
does not see. The floor here is therefore sum_e w_e * sum_i |h_i * wd_i|
(the expert-output floor of tests/tolerance.py, carried through the
combine) where that is larger. A wrong clamp moves h_i by O(limit) on
about half the elements and the outputs by O(floor)."""
import ctypes

import numpy as np
import pytest

import oracle as O
from test_gpu_moe import open_store, random_slabs, moe_floor
from test_gpu_prefill import prefill, floor_of, skewed_routing
from test_gpu_prefill_forms import FULL, QUEUED, ROWS
from tolerance import assert_close_combined, record

pytestmark = pytest.mark.gpu

E, DIM, INTER = 6, 256, 256


def split_slab(sl, dim=DIM, inter=INTER):
    """(wg, wu, wd) dequantized to bf16 from one expert slab."""
    out, off = [], 0
    for (o, k) in [(inter, dim), (inter, dim), (dim, inter)]:
        c = sl[off:off + o * k].reshape(o, k)
        off += o * k
        ns = O.nblocks(o) * O.nblocks(k)
        s = sl[off:off + 4 * ns].view(np.float32).reshape(O.nblocks(o), O.nblocks(k))
        off += 4 * ns
        out.append(O.dequant(c, s))
    return out


@pytest.fixture(scope="module")
def slabs():
    return random_slabs(E, DIM, INTER, np.random.default_rng(91))


@pytest.fixture(scope="module", params=[0.5, 4.0])
def store(ghip, slabs, request):
    limit = request.param
    stores = {}
    for lim in (limit, 10.0):
        s = open_store(ghip, E, DIM, INTER, limit=lim)
        for e, sl in enumerate(slabs):
            assert ghip.apus_ghip_store_put(s, e, O.ptr(sl), sl.nbytes) == 0
        stores[lim] = s
    yield ghip, stores, limit
    for s in stores.values():
        ghip.apus_ghip_store_close(s)


def oracle_inner(slabs, x, idx, w, limit, inter=INTER):
    """(floor [T, dim] = sum_j w_tj * sum_i |h_i * wd_ci| over the token's
    experts, and the fractions of their g above limit, u above limit and u
    below -limit), from the oracle's g, u and h (before the clamps for g
    and u)."""
    W = [split_slab(sl, x.shape[1], inter) for sl in slabs]
    wd_abs = [np.abs(O.bf16_to_f32(wd).astype(np.float64)) for _, _, wd in W]
    T, k = idx.shape
    floor = np.zeros(x.shape)
    gs, us = [], []
    for t in range(T):
        for j in range(k):
            wg, wu, wd = W[idx[t, j]]
            _, g, u, h = O.swiglu_expert(wg, wu, wd, x[t], limit)
            gs.append(O.bf16_to_f32(g))
            us.append(O.bf16_to_f32(u))
            hd = np.abs(O.bf16_to_f32(h).astype(np.float64))
            floor[t] += w[t, j] * (wd_abs[idx[t, j]] @ hd)
    g, u = np.concatenate(gs), np.concatenate(us)
    return floor, ((g > limit).mean(), (u > limit).mean(), (u < -limit).mean())


def test_decode_clamps(store, slabs):
    ghip, stores, limit = store
    rng = np.random.default_rng(int(limit * 8))
    for trial in range(3):
        x = O.f32_to_bf16(rng.standard_normal(DIM).astype(np.float32))
        idx = rng.permutation(E)[:4].astype(np.int32)
        w = rng.uniform(0.05, 1.0, 4).astype(np.float32)
        inner, frac = oracle_inner(slabs, x[None], idx[None], w[None], limit)
        assert min(frac) > 0.05, frac
        outs = {}
        for lim, s in stores.items():
            out = np.empty(DIM, np.uint16)
            rc = ghip.apus_ghip_moe_decode(s, O.ptr(x), O.ptr(idx), O.ptr(w), 4,
                                           O.ptr(out))
            assert rc == 0, ghip.apus_ghip_last_error()
            outs[lim] = out
        want, eo = O.moe_forward(slabs, DIM, INTER, x, idx[None], w[None], limit=limit,
                                 want_expert_out=True)
        st = assert_close_combined(outs[limit], want[0],
                                   np.maximum(moe_floor(eo, w[None], idx[None])[0], inner[0]),
                                   "decode limit=%g trial %d" % (limit, trial))
        record("swiglu_limit%g_decode_trial%d" % (limit, trial), st, clamp_fracs=[round(float(v), 4) for v in frac])
        assert not np.array_equal(outs[limit], outs[10.0])


@pytest.mark.parametrize("T,k,form", [(40, 3, ROWS), (600, 4, FULL)])
def test_prefill_clamps(store, slabs, T, k, form):
    ghip, stores, limit = store
    assert ghip.ghip_moe_prefill_form(DIM, INTER, E, k, ctypes.c_size_t(T)) == form
    rng = np.random.default_rng(T * 7 + k)
    x = O.f32_to_bf16(rng.standard_normal((T, DIM)).astype(np.float32))
    idx, w = skewed_routing(rng, T, E, k, hot=2)
    inner, frac = oracle_inner(slabs, x, idx, w, limit)
    assert min(frac) > 0.05, frac
    outs = {lim: prefill(ghip, s, x, idx, w, host=(T < 100))
            for lim, s in stores.items()}
    want, eo = O.moe_forward(slabs, DIM, INTER, x, idx, w, limit=limit,
                             want_expert_out=True, threads=8)
    st = assert_close_combined(outs[limit], want, np.maximum(floor_of(eo, w, idx), inner),
                               "prefill limit=%g T=%d k=%d" % (limit, T, k))
    record("swiglu_limit%g_prefill_T%d_k%d" % (limit, T, k), st, clamp_fracs=[round(float(v), 4) for v in frac])
    assert not np.array_equal(outs[limit], outs[10.0])


@pytest.mark.parametrize("limit", [0.5, 4.0])
def test_prefill_queued_clamps(ghip, limit):
    """The queued form's three bodies: an expert in every token (a tile of
    more than 128 rows), tiles of 17 to 128 rows, tiles of at most 16."""
    E, dim, inter, T, k = 16, 1024, 1024, 160, 4
    rng = np.random.default_rng(17)
    assert ghip.ghip_moe_prefill_form(dim, inter, E, k, ctypes.c_size_t(T)) == QUEUED
    slabs = random_slabs(E, dim, inter, rng)
    x = O.f32_to_bf16((0.5 * rng.standard_normal((T, dim))).astype(np.float32))
    p = 1.0 / np.arange(1, E) ** 1.5
    idx = np.array([rng.permutation(np.append(1 + rng.choice(E - 1, k - 1, False, p / p.sum()), 0))
                    for _ in range(T)], np.int32)
    rows = np.bincount(idx.ravel(), minlength=E)
    assert rows.max() > 128 and any(16 < r <= 128 for r in rows) and any(0 < r <= 16 for r in rows)
    w = rng.uniform(0.02, 0.6, (T, k)).astype(np.float32)
    inner, frac = oracle_inner(slabs, x, idx, w, limit, inter)
    assert min(frac) > 0.05, frac
    outs = []
    for lim in (limit, 10.0):
        s = open_store(ghip, E, dim, inter, limit=lim)
        try:
            for e, sl in enumerate(slabs):
                assert ghip.apus_ghip_store_put(s, e, O.ptr(sl), sl.nbytes) == 0
            outs.append(prefill(ghip, s, x, idx, w, host=False))
        finally:
            ghip.apus_ghip_store_close(s)
    want, eo = O.moe_forward(slabs, dim, inter, x, idx, w, limit=limit, want_expert_out=True,
                             threads=8)
    assert_close_combined(outs[0], want, np.maximum(floor_of(eo, w, idx), inner),
                          "queued prefill limit=%g" % limit)
    assert not np.array_equal(outs[0], outs[1])
