"""The forms a routed-MoE prefill launch takes (csrc/k_moe_prefill.hip,
csrc/k_moe_rows.hip) at the row counts where each can go wrong, every output
against the oracle's per-token loop (tests/tolerance.py): the weight streams
of few rows, the queued tile form's bodies (streams up to 16 rows, k split
between the wave halves up to 128, row halves above), the one-launch
permutation and its limits, and experts with NaN codes in each. The form is
asked of the library's own rule, so that a case that no longer reaches what it
is for fails."""
import ctypes

import numpy as np
import pytest

import oracle as O
import gpu_util as G
from tolerance import assert_close_combined
from test_gpu_moe import open_store, random_slabs
from test_gpu_prefill import floor_of, prefill

pytestmark = pytest.mark.gpu


QUEUED, FULL, ROWS = range(3)


def form(ghip, dim, inter, E, k, T):
    return ghip.ghip_moe_prefill_form(dim, inter, E, k, ctypes.c_size_t(T))


def routing_of(rows, rng):
    """[T, k] ids that give expert e rows[e] rows (the rest repeats, dropped).
    Experts past 16 spread their rows over the tokens with the fewest."""
    if len([r for r in rows if r]) > 16:
        T = max(max(rows), sum(rows) // 12)
        mine = [[] for _ in range(T)]
        for e in sorted(range(len(rows)), key=lambda e: -rows[e]):
            for t in sorted(range(T), key=lambda t: len(mine[t]))[:rows[e]]:
                mine[t].append(e)
        k = max(len(m) for m in mine)
        return np.array([list(rng.permutation(m)) + [m[0]] * (k - len(m)) for m in mine], np.int32)
    T, k = max(rows), max(1, max(sum(r > t for r in rows) for t in range(max(rows))))
    idx = np.empty((T, k), np.int32)
    for t in range(T):
        mine = list(rng.permutation([e for e, r in enumerate(rows) if r > t]))
        idx[t] = mine + [mine[0]] * (k - len(mine))
    return idx


def floor(slabs, dim, inter, x, idx, w, eo):
    """Every row is checked, with as few as one expert a token, so the floor is
    the one of the full-size checks: the combine's sum of |terms|, or, where
    an expert's down products cancel, its own terms carried through the
    weights -- a one-ulp step of one h_i (2^-8 |h_i| at most) moves that
    output by up to 2^-8 |h_i wd_i|, however small the sum."""
    return np.maximum(floor_of(eo, w, idx),
                      O.moe_expert_floor(slabs, dim, inter, x, idx, w, threads=16))


def check(ghip, dim, inter, rows, nan, want_form):
    """One store and routing; k <= 16 slots a token."""
    E = len(rows)
    rng = np.random.default_rng(sum(rows) + dim)
    slabs = random_slabs(E, dim, inter, rng, nan_codes_in=nan)
    s = open_store(ghip, E, dim, inter)
    try:
        for e, sl in enumerate(slabs):
            assert ghip.apus_ghip_store_put(s, e, O.ptr(sl), sl.nbytes) == 0
        idx = routing_of(rows, rng)
        T, k = idx.shape
        assert k <= 16 and form(ghip, dim, inter, E, k, T) == want_form
        w = rng.uniform(0.02, 0.6, (T, k)).astype(np.float32)
        x = O.f32_to_bf16((rng.standard_normal((T, dim)) *
                           rng.uniform(0.5, 4.0, (T, 1))).astype(np.float32))
        out = prefill(ghip, s, x, idx, w, host=False)
        want, eo = O.moe_forward(slabs, dim, inter, x, idx, w, want_expert_out=True, threads=16)
        assert_close_combined(out, want, floor(slabs, dim, inter, x, idx, w, eo), "%s" % (rows,))
        assert np.array_equal(out, prefill(ghip, s, x, idx, w, host=False))
    finally:
        ghip.apus_ghip_store_close(s)


@pytest.mark.parametrize("dim,inter,rows", [
    (256, 128, [1]), (512, 384, [1, 15, 16, 17, 0, 31, 32, 33, 48]),
    # parts of 32 rows: tiles of up to 256 rows and two tiles of an expert
    (256, 256, [260, 3, 0, 16] + [0] * 8), (256, 128, [256, 64, 65, 255, 33, 32, 1, 95, 96, 97, 0, 300] + [0] * 16),
    # every tile longer than one part, and longer ones past the 512th tile
    (256, 128, [33] * 16), (256, 128, [1] * 600 + [70, 0, 2, 40]),
    (1024, 128, [5] * 16)])
def test_prefill_streams(ghip, dim, inter, rows):
    """Little work: the weight streams, in passes of 16 rows."""
    check(ghip, dim, inter, rows, nan=(len(rows) - 1,), want_form=ROWS)


@pytest.mark.parametrize("rows", [
    [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128],
    [129, 159, 160, 161, 191, 192, 193, 223, 0, 8, 9, 40, 41, 70, 0, 100],
    [224, 225, 255, 256, 257, 20, 0, 0, 0, 4, 7, 300, 50, 10, 16, 80]])
def test_prefill_queued_bodies(ghip, rows):
    """Sparse tiles with enough work for the queued form (more than 3 GFLOP,
    under 128 rows an expert): each body's row remainders; the experts with
    NaN codes take the exact one."""
    dim, inter = 1024, 1024
    assert 6.0 * sum(rows) * dim * inter > 3e9 and sum(rows) > len(rows)
    T, k = routing_of(rows, np.random.default_rng(0)).shape
    assert T * k < 128 * len(rows) * 16
    check(ghip, dim, inter, rows + [0] * max(0, (T * k) // 127 + 1 - len(rows)), nan=(1, 4, 13),
          want_form=QUEUED)


@pytest.mark.parametrize("rows", [[256, 255, 225, 224], [257, 130, 300, 129, 31], [193, 192, 160, 128]])
def test_prefill_full_tiles(ghip, rows):
    """Tiles mostly full: each body of the static form."""
    check(ghip, 512, 256, rows, nan=(3,), want_form=FULL)


def test_prefill_permutation_limit(ghip):
    """1024 pairs are sorted in one launch, 1025 in four: the same results for
    the tokens both have. Up to 1024 experts."""
    dim, inter, E = 256, 128, 1000
    rng = np.random.default_rng(6)
    slab = random_slabs(1, dim, inter, rng)[0]
    s = open_store(ghip, E, dim, inter)
    try:
        for e in range(E):
            assert ghip.apus_ghip_store_put(s, e, O.ptr(slab), slab.nbytes) == 0
        x = O.f32_to_bf16(rng.standard_normal((1025, dim)).astype(np.float32))
        idx = rng.integers(0, E, (1025, 1)).astype(np.int32)
        w = rng.uniform(0.02, 0.6, (1025, 1)).astype(np.float32)
        a = prefill(ghip, s, x[:1024], idx[:1024], w[:1024], host=False)
        b = prefill(ghip, s, x, idx, w, host=False)
        assert np.array_equal(a, b[:1024])
        want, eo = O.moe_forward([slab] * E, dim, inter, x, idx, w, want_expert_out=True,
                                 threads=16)
        assert_close_combined(b, want, floor([slab] * E, dim, inter, x, idx, w, eo), "1025 pairs")
    finally:
        ghip.apus_ghip_store_close(s)


def test_prefill_activations_past_4_gib(ghip):
    """h of more than 4 GiB: the tokens go in slices, and each reads its own
    rows of x and h."""
    dim, inter, E, T, period = 256, 16384, 2, 131272, 1009
    assert T * inter * 2 > 1 << 32
    rng = np.random.default_rng(9)
    slabs = random_slabs(E, dim, inter, rng)
    s = open_store(ghip, E, dim, inter)
    try:
        for e, sl in enumerate(slabs):
            assert ghip.apus_ghip_store_put(s, e, O.ptr(sl), sl.nbytes) == 0
        x = O.f32_to_bf16(rng.standard_normal((period, dim)).astype(np.float32))
        idx = rng.integers(0, E, (period, 1)).astype(np.int32)
        w = rng.uniform(0.02, 0.6, (period, 1)).astype(np.float32)
        out = prefill(ghip, s, np.resize(x, (T, dim)), np.resize(idx, (T, 1)), np.resize(w, (T, 1)),
                      host=False)
        want, eo = O.moe_forward(slabs, dim, inter, x, idx, w, want_expert_out=True, threads=16)
        assert_close_combined(out[:period], want, floor(slabs, dim, inter, x, idx, w, eo), "first tokens")
        whole = T // period * period
        assert (out[:whole].reshape(-1, period, dim) == out[:period]).all()
        assert np.array_equal(out[whole:], out[:T - whole])
    finally:
        ghip.apus_ghip_store_close(s)
