"""The work the performance figures are about: calls of the public entry points (include/backend_hip.h) as an engine
makes them, over the sizes it makes them with.

Three families, at the shapes of this repository's configurations and tests:

  linear   the FP8-block projections of the attention layers (q_a 1536x4096, q_b 16384x1536, kv_a 512x4096, o_proj
           4096x16384) and the BF16 ones (square projections, expert-sized matrices, the LM head 154880x4096), from one
           decode row over the 2..4 rows of a speculative verify and short prompts to prefill; device pointers, and the
           host-pointer form behind the hook table;
  dequant  FP8 blocks to BF16 weights;
  MoE      288 experts of 4096/2048 with 8 of them a token, with and without the shared expert: one decode token
           (given routing, logits, or the router in the launch), the router alone, and prefill from a few tokens to 8192;
           and smaller banks.

draw() takes one of these families with sizes spread over the same ranges, ragged ones among them.
"""
import ctypes
import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DSA = {"q_a": (1536, 4096), "q_b": (16384, 1536), "kv_a": (512, 4096), "o_proj": (4096, 16384)}
LM_HEAD = (154880, 4096)
BANK = {"experts": 288, "dim": 4096, "inter": 2048, "topk": 8}
# scales of the synthetic banks: uniform codes have an rms of ~100, so weights come out near 0.02
SCALES = (1e-4, 4e-4)
LIMIT = 10.0


def listed():
    def dense(name, op, shape, rows, **more):
        return {"name": name, "op": op, "M": rows, "N": shape[0], "K": shape[1], **more}

    return [
        # one decode token through the smallest projection: launch and latency
        dense("fp8 kv_a decode M1", "fp8_linear", DSA["kv_a"], 1, exact=0),
        # a speculative verify (1 token + 3 drafts) through the largest one
        dense("fp8 o_proj verify M4", "fp8_linear", DSA["o_proj"], 4, exact=0),
        # a short prompt, or a small batch of requests: a row count between decode and prefill
        dense("fp8 q_a short M11", "fp8_linear", DSA["q_a"], 11, exact=0),
        # prefill of a prompt of no particular length
        dense("fp8 q_b prefill M1111", "fp8_linear", DSA["q_b"], 1111, exact=0),
        # the engine's own call: host activations and result through the hook's entry point, weights registered
        dense("fp8 q_a host M1", "fp8_host", DSA["q_a"], 1),
        # BF16 weights made once from FP8 blocks (any code, NaN codes too: the exact decode)
        {"name": "dequant 16384x4096", "op": "dequant", "N": 16384, "K": 4096, "exact": 1},
        # the LM head of a decode step
        dense("bf16 lm_head decode M1", "bf16_linear", LM_HEAD, 1),
        # a BF16 projection of a prompt
        dense("bf16 proj prefill M600", "bf16_linear", (4096, 4096), 600),
        # the MoE layer of one decode token: router, 8 routed experts and the shared one in one call
        dict(BANK, name="moe decode router shared", op="decode", routing="router", shared=True),
        # the MoE layer of a short prompt, a verify of a few sequences, or a small batch
        dict(BANK, name="moe prefill T12", op="prefill", T=12, zipf=0.0, shared=False),
        # a prompt with skewed routing: from experts with no token to experts with over a thousand
        dict(BANK, name="moe prefill T2048 zipf", op="prefill", T=2048, zipf=1.1, shared=False),
        # the longest prompt, the whole layer
        dict(BANK, name="moe prefill T8192 shared", op="prefill", T=8192, zipf=0.0, shared=True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["fp8_linear", "fp8_linear", "bf16_linear", "bf16_linear", "fp8_host", "dequant", "decode", "prefill",
                     "prefill", "router"])
    if op in ("fp8_linear", "fp8_host"):
        case = {"op": op, "M": _log(rng, 1, 2048)}
        if rng.random() < 0.6:
            case["N"], case["K"] = rng.choice(sorted(DSA.values()) + [(2048, 4096), (16384, 4096)])
        else:  # generic shapes: any row count, whole scale blocks along K or (small ones) not
            case["N"] = _log(rng, 64, 8192)
            case["K"] = 128 * _log(rng, 1, 64)
            case["M"] = min(case["M"], 256)
            if rng.random() < 0.25:
                case.update(N=min(case["N"], 2000), K=case["K"] // 4 + rng.randrange(1, 128), M=min(case["M"], 64))
        if op == "fp8_host":
            case["M"] = min(case["M"], 256)
        else:
            case["exact"] = rng.choice([0, 0, 0, -1])
        return case
    if op == "bf16_linear":
        case = {"op": op, "M": _log(rng, 1, 2048)}
        pick = rng.random()
        if pick < 0.6:
            case["N"], case["K"] = rng.choice([(4096, 4096), (2048, 4096), (4096, 2048), (288, 4096), (8192, 4096)])
        elif pick < 0.75:
            case["N"], case["K"] = LM_HEAD
            case["M"] = min(case["M"], rng.choice([4, 16]))
        else:
            case["N"], case["K"] = _log(rng, 64, 8192), 64 * _log(rng, 1, 96)
            case["M"] = min(case["M"], 512)
            if rng.random() < 0.25:
                case.update(N=min(case["N"], 2000), K=case["K"] // 4 + rng.randrange(1, 64), M=min(case["M"], 64))
        return case
    if op == "dequant":
        return {"op": op, "N": _log(rng, 128, 16384), "K": rng.choice([1536, 2048, 4096, 127 + rng.randrange(2000)]),
                "exact": rng.choice([0, 1])}
    bank = dict(rng.choice([BANK, BANK, {"experts": 64, "dim": 2048, "inter": 1024, "topk": 6},
                            {"experts": 16, "dim": 1024, "inter": 512, "topk": 4}]))
    if op == "router":
        return {"op": op, "experts": rng.choice([bank["experts"], rng.randrange(16, 512)]), "dim": bank["dim"], "topk": bank["topk"]}
    case = dict(bank, op=op, shared=rng.random() < 0.5)
    if op == "decode":
        case["routing"] = rng.choice(["given", "logits", "router"])
        case["topk"] = rng.choice([bank["topk"], rng.randrange(1, 17)])
    else:
        case["T"] = _log(rng, 2, 8192 if case["experts"] > 16 else 2048)
        case["zipf"] = rng.choice([0.0, 1.1])
    return case


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------

_pkg = None


def _lib():
    """The package (its directory is no Python name) and its library. torch is imported first, so the library's HIP
    runtime (by its soname) is the one torch has loaded."""
    global _pkg
    if _pkg is None:
        path = os.path.join(ROOT, "apus-glm5.3-flash_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("apus_ghip", path, submodule_search_locations=[os.path.dirname(path)])
        _pkg = importlib.util.module_from_spec(spec)
        sys.modules["apus_ghip"] = _pkg
        spec.loader.exec_module(_pkg)
        err = ctypes.create_string_buffer(256)
        if _pkg.load().apus_ghip_enable(err, 256) != 0:
            raise RuntimeError(err.value.decode())
    return _pkg.load()


def _gen(seed, tag):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + tag) & 0x7FFFFFFFFFFFFFFF)


def _nb(n):
    return (n + 127) // 128


def _fp8(case, seed):
    """Codes and block scales of a quantized normal weight: each 128x128 block's largest value at code 448."""
    N, K, g = case["N"], case["K"], _gen(seed, 1)
    n, k = _nb(N) * 128, _nb(K) * 128
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02)
    scales = (w.view(n // 128, 128, k // 128, 128).abs().amax(dim=(1, 3)) / 448.0).contiguous()
    w.view(n // 128, 128, k // 128, 128).div_(scales[:, None, :, None])
    codes = w.to(torch.float8_e4m3fn).view(torch.uint8)[:N, :K].contiguous()
    return codes, scales


def _bf16(shape, seed, tag, scale=1.0):
    return torch.randn(shape, generator=_gen(seed, tag), device="cuda").mul_(scale).to(torch.bfloat16)


def _route(T, E, k, zipf, seed):
    """[T, k] distinct experts a token, uniform or Zipf over seeded ranks, and softmax weights."""
    p = torch.arange(1, E + 1, dtype=torch.float64, device="cuda") ** -zipf
    p = p[torch.randperm(E, generator=_gen(seed, 21), device="cuda")]
    # the k largest of log p + Gumbel noise: k draws without replacement
    u = torch.rand((T, E), generator=_gen(seed, 22), device="cuda", dtype=torch.float64).clamp_(1e-300)
    idx = (p.log() - (-u.log()).log()).topk(k, dim=1).indices.to(torch.int32)
    w = torch.softmax(torch.randn((T, k), generator=_gen(seed, 23), device="cuda"), dim=1)
    return idx.contiguous(), w.contiguous()


def _shared_slab(case, seed):
    """The shared expert's three matrices: [(codes, scales)] in slab order."""
    dim, inter = case["dim"], case["inter"]
    parts = []
    for j, (n, k) in enumerate([(inter, dim), (inter, dim), (dim, inter)]):
        g = _gen(seed, 30 + j)
        codes = torch.randint(0, 254, (n, k), generator=g, device="cuda", dtype=torch.int16)
        codes = (codes + (codes >= 127)).to(torch.uint8)
        scales = torch.empty((_nb(n), _nb(k)), device="cuda").uniform_(*SCALES, generator=g)
        parts.append((codes, scales))
    return parts


class _State:
    """What a program holds between calls: the buffers, the store, and the call itself."""

    store = None
    regions = ()

    def __del__(self):
        if self.store is not None:
            self.lib.apus_ghip_store_close(self.store)
        for p in self.regions:
            self.lib.apus_ghip_unregister_region(p)


def prepare(case, seed):
    lib = _lib()
    s = _State()
    s.lib = lib
    op = case["op"]
    stream = torch.cuda.current_stream().cuda_stream
    if op in ("fp8_linear", "fp8_host", "bf16_linear"):
        M, N, K = case["M"], case["N"], case["K"]
        x = _bf16((M, K), seed, 2)
        if op == "bf16_linear":
            w = _bf16((N, K), seed, 1, 0.02)
            y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
            s.keep = (w, x, y)
            s.call = lib.apus_ghip_bf16_gemm_dev
            s.args = (w.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, stream)
        else:
            codes, scales = _fp8(case, seed)
            y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda" if op == "fp8_linear" else "cpu")
            if op == "fp8_host":
                codes, scales, x = codes.cpu(), scales.cpu(), x.cpu()
                s.regions = (codes.data_ptr(), scales.data_ptr())
                for p, n in zip(s.regions, (codes.numel(), scales.numel() * 4)):
                    _pkg.check(lib.apus_ghip_register_region(p, n), "register_region")
            s.keep = (codes, scales, x, y)
            s.call = lib.apus_ghip_fp8blk_linear_dev if op == "fp8_linear" else lib.apus_ghip_fp8blk_linear
            s.args = tuple(t.data_ptr() for t in s.keep) + (M, N, K)
            if op == "fp8_linear":
                s.args += (case["exact"], stream)
        s.out = y
        return s
    if op == "dequant":
        codes, scales = _fp8(case, seed)
        s.out = torch.empty((case["N"], case["K"]), dtype=torch.bfloat16, device="cuda")
        s.keep = (codes, scales)
        s.call = lib.apus_ghip_fp8blk_dequant_dev
        s.args = (codes.data_ptr(), scales.data_ptr(), s.out.data_ptr(), case["N"], case["K"], case["exact"], stream)
        return s
    E, dim, k = case["experts"], case["dim"], case["topk"]
    gate = bias = None
    if op == "router" or case.get("routing") == "router":
        gate = _bf16((E, dim), seed, 3, dim ** -0.5)
        bias = torch.randn(E, generator=_gen(seed, 4), device="cuda").mul_(0.05)
    if op == "router":
        x = _bf16((dim,), seed, 2)
        scores = torch.empty(E, device="cuda")
        idx, w = torch.empty(k, dtype=torch.int32, device="cuda"), torch.empty(k, device="cuda")
        s.keep, s.out = (x, gate, bias), {"scores": scores, "idx": idx, "w": w}
        s.call = lib.apus_ghip_moe_router_dev
        s.args = (x.data_ptr(), gate.data_ptr(), None, bias.data_ptr(), E, dim, k, 2.5, scores.data_ptr(), idx.data_ptr(),
                  w.data_ptr(), stream)
        return s
    err = ctypes.create_string_buffer(256)
    store = ctypes.c_void_p()
    _pkg.check(lib.apus_ghip_store_open(ctypes.byref(store), E, dim, case["inter"], LIMIT, err, 256), "store_open")
    s.store = store
    _pkg.check(lib.apus_ghip_store_synth(store, seed, 0, *SCALES), "store_synth")
    if case["shared"]:
        slab = torch.cat([t.reshape(-1).view(torch.uint8) for p in _shared_slab(case, seed) for t in p]).cpu()
        _pkg.check(lib.apus_ghip_store_put_shared(store, slab.data_ptr(), slab.numel()), "put_shared")
    T = case.get("T", 1)
    x = _bf16((T, dim), seed, 2)
    out = torch.empty((T, dim), dtype=torch.bfloat16, device="cuda")
    if op == "prefill":
        idx, w = _route(T, E, k, case["zipf"], seed)
        _pkg.check(lib.apus_ghip_moe_prefill_reserve(store, T, k), "prefill_reserve")
        s.keep, s.out = (x, idx, w), out
        s.call = lib.apus_ghip_moe_prefill_dev
        s.args = (store, x.data_ptr(), T, idx.data_ptr(), w.data_ptr(), k, out.data_ptr(), stream)
    elif case["routing"] == "router":
        idx, w = torch.empty(k, dtype=torch.int32, device="cuda"), torch.empty(k, device="cuda")
        s.keep, s.out = (x, gate, bias), {"out": out, "idx": idx, "w": w}
        s.call = lib.apus_ghip_moe_decode_router_dev
        s.args = (store, x.data_ptr(), gate.data_ptr(), bias.data_ptr(), 2.5, k, out.data_ptr(), idx.data_ptr(), w.data_ptr(),
                  stream)
    else:
        logits = idx = w = None
        if case["routing"] == "logits":
            logits = torch.randn(E, generator=_gen(seed, 5), device="cuda")
        else:
            idx, w = _route(1, E, k, 0.0, seed)
        s.keep, s.out = (x, logits, idx, w), out
        s.call = lib.apus_ghip_moe_decode_dev
        s.args = (store, x.data_ptr()) + tuple(None if t is None else t.data_ptr() for t in (logits, idx, w)) + (
            k, out.data_ptr(), stream)
    return s


def run(state):
    if state.call(*state.args) != 0:
        raise RuntimeError(_pkg.last_error())
    return state.out


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, what it may be off by, what it should be
# ---------------------------------------------------------------------------------------------------------------------


def _touched(case):
    """Expected number of experts with a token."""
    E, k, T = case["experts"], case["topk"], case.get("T", 1)
    p = [(r + 1) ** -case.get("zipf", 0.0) for r in range(E)]
    z = sum(p)
    return sum(1.0 - (1.0 - min(1.0, k * q / z)) ** T for q in p)


def work(case):
    op = case["op"]
    if op in ("fp8_linear", "fp8_host", "bf16_linear"):
        M, N, K = case["M"], case["N"], case["K"]
        w = 2 * N * K if op == "bf16_linear" else N * K + 4 * _nb(N) * _nb(K)
        return {"bytes": w + 2 * M * (N + K), "flops": 2 * M * N * K}
    if op == "dequant":
        N, K = case["N"], case["K"]
        return {"bytes": 3 * N * K + 4 * _nb(N) * _nb(K), "flops": N * K}
    E, dim, k = case["experts"], case["dim"], case["topk"]
    if op == "router":
        return {"bytes": 2 * E * dim + 2 * dim + 8 * E + 8 * k, "flops": 2 * E * dim}
    inter, T, shared = case["inter"], case.get("T", 1), int(case["shared"])
    slab = 3 * dim * inter + 12 * _nb(dim) * _nb(inter)
    touched = (k if op == "decode" else _touched(case)) + shared
    gate = 2 * E * dim + 4 * E if case.get("routing") == "router" else 0
    return {"bytes": touched * slab + 4 * T * dim + 8 * T * k + gate, "flops": 6 * T * (k + shared) * dim * inter}


def tolerance(case):
    op = case["op"]
    if op == "dequant":
        return "exact"
    if op == "router":
        return {"rel": 1e-5, "max": 1e-4}
    if op in ("decode", "prefill"):
        return {"rel": 1e-2, "max": 0.08}
    return {"rel": 7e-3, "max": 0.03}


def _deq(codes, scales):
    """bf16(e4m3(code) * scale), in 64 bits: the weights as the format defines them (the two NaN codes are +-480)."""
    c = torch.arange(256, device=codes.device)
    e, m = (c >> 3) & 15, c & 7
    table = torch.where(e > 0, (8 + m) * torch.exp2((e - 10).double()), m * 2.0 ** -9)
    table = torch.where(c > 127, -table, table).float()
    n, k = codes.shape
    s = scales.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    return (table[codes.long()] * s).to(torch.bfloat16).double()


def _mix64(z):
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * (0x94D049BB133111EB - (1 << 64))
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _draws(seed, stream, n):
    """The first n 64-bit draws of a stream of the banks' generator (include/apus_synth.h), as signed numbers."""
    wrap = lambda v: (v + (1 << 63)) % (1 << 64) - (1 << 63)  # noqa: E731
    key = _mix64(torch.tensor(wrap(seed + (stream + 1) * 0x632BE59BD9B4E019), device="cuda"))
    return _mix64(torch.arange(1, n + 1, device="cuda") * (0x9E3779B97F4A7C15 - (1 << 64)) + key)


def _expert(case, seed, e):
    """Expert e's three matrices in 64 bits, from the definition of the synthetic banks."""
    dim, inter = case["dim"], case["inter"]
    if e == case["experts"]:
        return [_deq(c, s) for c, s in _shared_slab(case, seed)]
    a, b = (math.log(torch.tensor(v, dtype=torch.float32).item()) for v in SCALES)
    got = []
    for j, (n, k) in enumerate([(inter, dim), (inter, dim), (dim, inter)]):
        u = _draws(seed, e * 8 + 2 * j + 1024, n * k)
        r = (u % 254 + (u < 0) * ((1 << 64) % 254)) % 254
        codes = (r + (r >= 127)).to(torch.uint8).view(n, k)
        u = _draws(seed, e * 8 + 2 * j + 1 + 1024, _nb(n) * _nb(k))
        unit = ((u >> 11) & ((1 << 53) - 1)).double() * 2.0 ** -53
        got.append(_deq(codes, torch.exp(a + unit * (b - a)).float().view(_nb(n), _nb(k))))
    return got


def _experts_out(case, seed, x, idx, w):
    """sum over a token's experts of weight * down(silu(min(gate, limit)) * clamp(up)), in 64 bits."""
    y = torch.zeros_like(x)
    E = case["experts"]
    for e in range(E + int(case["shared"])):
        if e < E:
            t, j = (idx == e).nonzero(as_tuple=True)
            if not len(t):
                continue
            we = w[t, j].double()[:, None]
        else:
            t, we = torch.arange(len(x), device="cuda"), 1.0
        wg, wu, wd = _expert(case, seed, e)
        g, u = x[t] @ wg.T, x[t] @ wu.T
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        y.index_add_(0, t, we * ((g * torch.sigmoid(g) * u) @ wd.T))
    return y


def exact(case, seed):
    op = case["op"]
    if op == "dequant":
        return _deq(*_fp8(case, seed))
    if op in ("fp8_linear", "fp8_host", "bf16_linear"):
        x = _bf16((case["M"], case["K"]), seed, 2).double()
        w = _bf16((case["N"], case["K"]), seed, 1, 0.02).double() if op == "bf16_linear" else _deq(*_fp8(case, seed))
        y = x @ w.T
        return y.cpu() if op == "fp8_host" else y
    E, dim, k = case["experts"], case["dim"], case["topk"]
    idx = w = scores = None
    x = _bf16((dim,) if op == "router" else (case.get("T", 1), dim), seed, 2).double()
    if op == "router" or case.get("routing") == "router":
        gate = _bf16((E, dim), seed, 3, dim ** -0.5).double()
        bias = torch.randn(E, generator=_gen(seed, 4), device="cuda").mul_(0.05).double()
        scores = torch.sigmoid(gate @ x.reshape(-1))
        idx = (scores + bias).topk(k).indices
        w = scores[idx] / scores[idx].sum() * 2.5
        if op == "router":
            return {"scores": scores, "idx": idx.to(torch.int32), "w": w}
        y = _experts_out(case, seed, x, idx[None], w[None])
        return {"out": y, "idx": idx.to(torch.int32), "w": w}
    if case.get("routing") == "logits":
        logits = torch.randn(E, generator=_gen(seed, 5), device="cuda").double()
        top = logits.topk(k)
        idx, w = top.indices[None], torch.softmax(top.values, 0)[None]
    else:
        idx, w = _route(case.get("T", 1), E, k, case.get("zipf", 0.0), seed)
    return _experts_out(case, seed, x, idx, w)
