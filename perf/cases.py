"""The work that a program using this library has it do, as cases that can be timed.

A case is one kind of call with its sizes and options, made once for each of `layers`
weight matrices (or caches): a serving loop goes through all layers of a model before it
meets a matrix again, so decode cases hold enough layers that the matrices come from
memory and not from a cache.  Calls go through the public Python entry points
(`capi`), on the default stream, one after the other, as a program makes them.

Kinds
  gemm   c = x W^T with packed weights (`fmt` "w4": groups of `gs` with FP16 scales and,
         when not `sym`, 4-bit zero-points; "mx": MXFP4), through the dispatcher
  act    FP16 activations quantized (`fmt` "a8": MXFP8, "a4": MXFP4) and multiplied with
         MXFP4 weights on the scaled matrix cores
  attn   one query token per sequence against a cache of S positions (`fmt` "w4", "f8",
         "f16"); `page` > 0: pooled pages with one block table per sequence
  kv     FP16 keys and values quantized into a cache (`fmt` "w4", "f8")
"""
import importlib
import math

import torch

_pkg = importlib.import_module("w4a16-dequant-gemm_amd")
capi = _pkg.capi

DEV = "cuda"
FP8_MAX = 448.0


def listed():
    return [
        # the smallest call: one token through square projections, layer after layer; launch
        # and memory latency count as much as bandwidth
        _gemm("w4_m1_square", "w4", 1, 4096, 4096, 128, True, 32),
        # a batch of sixteen sequences through an up projection with zero-points
        _gemm("w4_m16_up", "w4", 16, 11008, 4096, 128, False, 6),
        # small groups and a row length that is no multiple of 32, nine sequences
        _gemm("w4_m9_ragged_k", "w4", 9, 11008, 4104, 8, False, 4),
        # MXFP4 down projection, a larger decode batch (not a multiple of the tile)
        _gemm("mx_m50_down", "mx", 50, 4096, 14336, 32, True, 5),
        # a chunk of a prompt mixed with decode tokens: between decode and prefill
        _gemm("w4_m333_chunk", "w4", 333, 4096, 4096, 64, False, 4),
        # prefill of a 2048-token prompt
        _gemm("w4_m2048_prefill", "w4", 2048, 4096, 4096, 128, True, 1),
        # the largest: several prompts at once through a wide projection, ragged in M
        _gemm("w4_m4000_wide", "w4", 4000, 11008, 4096, 32, False, 1),
        # 8-bit activations against MXFP4 weights, a large serving batch
        _act("a8_m192_up", "a8", 192, 14336, 4096, 4),
        # long-context decode, grouped queries, 4-bit cache: 8 sequences of 32768 tokens
        _attn("attn_w4_long", "w4", 8, 8, 4, 32768, 128, 32, True, 0, False, 1),
        # everyday decode from a paged pool: 16 sequences of 1500 tokens that share a prefix
        _attn("attn_w4_paged", "w4", 16, 8, 4, 1500, 128, 32, True, 16, True, 8),
        # FP8 cache with one scale per row, medium context, ragged length
        _attn("attn_f8_medium", "f8", 4, 8, 4, 6007, 128, 128, True, 0, False, 4),
        # prefill writes its keys and values: one 4096-token sequence, 8 cache heads, 4 layers
        _kv("kv_w4_prefill", "w4", 8, 4096, 128, 32, True, 4),
    ]


def _gemm(name, fmt, M, N, K, gs, sym, layers):
    return {"name": name, "kind": "gemm", "fmt": fmt, "M": M, "N": N, "K": K, "gs": gs,
            "sym": sym, "layers": layers}


def _act(name, fmt, M, N, K, layers):
    return {"name": name, "kind": "act", "fmt": fmt, "M": M, "N": N, "K": K, "layers": layers}


def _attn(name, fmt, nseq, hkv, group, S, D, gs, sym, page, shared, layers):
    return {"name": name, "kind": "attn", "fmt": fmt, "nseq": nseq, "hkv": hkv, "group": group,
            "S": S, "D": D, "gs": gs, "sym": sym, "page": page, "shared": shared, "slab_scale": False,
            "layers": layers}


def _kv(name, fmt, H, S, D, gs, sym, layers):
    return {"name": name, "kind": "kv", "fmt": fmt, "H": H, "S": S, "D": D, "gs": gs, "sym": sym,
            "layers": layers}


# ---- draws ---------------------------------------------------------------------------------

# (N, K) of projections this repository's tests and benchmark name
_SHAPES = [(4096, 4096), (11008, 4096), (14336, 4096), (4096, 11008), (4096, 14336), (5120, 5120),
           (13824, 5120), (5120, 13824), (8192, 8192), (6144, 4096), (22016, 4096), (28672, 4096)]
_MAX_COST = 2.0 * 4000 * 11008 * 4096 * 0.8  # flops; a byte counts as 150 of them


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))


def _shape(rng):
    if rng.random() < 0.5:
        return rng.choice(_SHAPES)
    step_n, step_k = rng.choice([(16, 128), (128, 128), (64, 256), (8, 32), (1, 128), (16, 8)])
    return (max(1, int(_log(rng, 1024, 16384)) // step_n) * step_n,
            max(1, int(_log(rng, 1024, 14336)) // step_k) * step_k)


def _cost(case):
    w = work(case)
    return w["flops"] + 150 * w["bytes"]


def _draw_once(rng):
    pick = rng.random()
    if pick < 0.62:
        N, K = _shape(rng)
        fmt = "w4" if rng.random() < 0.75 else "mx"
        M = int(_log(rng, 1, 64) if rng.random() < 0.6 else _log(rng, 65, 4096))
        if rng.random() < 0.3:
            M = max(1, M // 8 * 8)
        gs = 32 if fmt == "mx" else rng.choice([32, 64, 128, 128, 128, 128, 48, 8])
        sym = True if fmt == "mx" else rng.random() < 0.5
        layers = max(1, min(32, round(1.3e8 / (N * K / 2)))) if M <= 64 else 1
        case = _gemm("", fmt, M, N, K, gs, sym, layers)
    elif pick < 0.70:
        N, K = rng.choice(_SHAPES[:5])
        M = int(_log(rng, 1, 2048))
        layers = max(1, min(32, round(1.3e8 / (N * K / 2)))) if M <= 256 else 1
        case = _act("", rng.choice(["a8", "a4"]), M, N, K, layers)
    elif pick < 0.93:
        fmt = rng.choice(["w4", "w4", "f8", "f16"])
        nseq, hkv = int(_log(rng, 1, 32)), rng.choice([2, 4, 8, 8])
        D = 128 if rng.random() < 0.8 else 64
        page = rng.choice([0, 16, 16, 64]) if fmt == "w4" else 0
        gs = rng.choice([32, 32, 64, 128 if D == 128 else 32])
        case = _attn("", fmt, nseq, hkv, rng.choice([1, 4, 4, 8]), int(_log(rng, 200, 32768)), D, gs,
                     fmt != "w4" or rng.random() < 0.6, page, page > 0 and rng.random() < 0.5, 1)
        case["slab_scale"] = fmt == "f8" and rng.random() < 0.4
        case["layers"] = max(1, min(16, round(1.3e8 / work(case)["bytes"])))
    else:
        D = rng.choice([128, 128, 64])
        case = _kv("", rng.choice(["w4", "w4", "f8"]), rng.choice([4, 8, 8, 32]),
                   int(_log(rng, 1, 8192)), D, rng.choice([32, 64]), rng.random() < 0.6, 4)
    del case["name"]
    return case


def draw(rng):
    while True:
        case = _draw_once(rng)
        if _cost(case) <= _MAX_COST:
            return case


# ---- inputs --------------------------------------------------------------------------------


def _words(k):
    return (k + 7) // 8


def _half(gen, *shape):
    return torch.randn(*shape, dtype=torch.float16, device=DEV, generator=gen)


def _ints(*shape):
    return torch.empty(*shape, dtype=torch.int32, device=DEV)


def _halves(*shape):
    return torch.empty(*shape, dtype=torch.float16, device=DEV)


def _bytes(*shape):
    return torch.empty(*shape, dtype=torch.uint8, device=DEV)


def _weights_w4(gen, N, K, gs, sym, status):
    """One quantized matrix: N(0, 0.02), and with zero-points a tenth of the groups one-sided."""
    w = torch.randn(N, K, dtype=torch.float64, device=DEV, generator=gen).mul_(0.02)
    G = (K + gs - 1) // gs
    if not sym:
        one_sided = torch.rand(N, G, device=DEV, generator=gen) < 0.1
        one_sided = one_sided.repeat_interleave(gs, dim=1)[:, :K]
        w = torch.where(one_sided, w.abs(), w)
    q, s = _ints(N, _words(K)), _halves(N, G)
    z = None if sym else _ints(N, _words(G))
    view = capi.packed_view(N, K, gs, G, sym, q.data_ptr(), s.data_ptr(), 0 if sym else z.data_ptr())
    capi.quantize(view, w.data_ptr(), status.data_ptr())
    return view, (q, s, z)


def _weights_mx(gen, N, K, status):
    """One MXFP4 matrix: N(0, 0.02) with one per cent of the elements at 20 sigma."""
    w = torch.randn(N, K, dtype=torch.float64, device=DEV, generator=gen).mul_(0.02)
    far = torch.rand(N, K, device=DEV, generator=gen) < 0.01
    w = torch.where(far, w.sign() * 0.4, w)
    B = (K + 31) // 32
    q, s = _ints(N, _words(K)), _bytes(N, B)
    view = capi.packed_mx_view(N, K, B, q.data_ptr(), s.data_ptr())
    capi.quantize_mx(view, w.data_ptr(), status.data_ptr())
    return view, (q, s)


def _prepare_gemm(case, gen):
    M, N, K, L = case["M"], case["N"], case["K"], case["layers"]
    status = _ints(1)
    mats = [_weights_mx(gen, N, K, status) if case["fmt"] == "mx" else
            _weights_w4(gen, N, K, case["gs"], case["sym"], status) for _ in range(L)]
    x, c = _half(gen, L, M, K), _halves(L, M, N)
    call = capi.gemm_mx if case["fmt"] == "mx" else capi.gemm
    return {"run": _run_gemm, "call": call, "M": M, "out": c, "keep": (mats, x),
            "layers": [(v, x[i].data_ptr(), c[i].data_ptr()) for i, (v, _) in enumerate(mats)]}


def _run_gemm(s):
    call, M = s["call"], s["M"]
    for view, x, c in s["layers"]:
        call(view, x, c, M)
    return s["out"]


def _prepare_act(case, gen):
    M, N, K, L = case["M"], case["N"], case["K"], case["layers"]
    B = (K + 31) // 32
    status = _ints(1)
    mats = [_weights_mx(gen, N, K, status) for _ in range(L)]
    x, c = _half(gen, L, M, K), _halves(L, M, N)
    xs = _bytes(M, B)
    if case["fmt"] == "a8":
        xq = _bytes(M, K)
        xv = capi.act_mx8_view(M, K, B, xq.data_ptr(), xs.data_ptr())
        quant, mul = capi.quantize_mx8_f16, capi.gemm_mx_w4a8
    else:
        xq = _ints(M, _words(K))
        xv = capi.packed_mx_view(M, K, B, xq.data_ptr(), xs.data_ptr())
        quant, mul = capi.quantize_mx_f16, capi.gemm_mx_w4a4
    return {"run": _run_act, "quant": quant, "mul": mul, "xv": xv, "status": status.data_ptr(),
            "out": c, "keep": (mats, x, xq, xs, status),
            "layers": [(v, x[i].data_ptr(), c[i].data_ptr()) for i, (v, _) in enumerate(mats)]}


def _run_act(s):
    quant, mul, xv, status = s["quant"], s["mul"], s["xv"], s["status"]
    for view, x, c in s["layers"]:
        quant(xv, x, status)
        mul(view, xv, c)
    return s["out"]


def _cache_w4(gen, H, S, D, gs, sym, status):
    G = (D + gs - 1) // gs
    t = [_ints(H, S, _words(D)), _halves(H, S, G), None if sym else _ints(H, S, _words(G)),
         _ints(H, S, _words(D)), _halves(H, S, G), None if sym else _ints(H, S, _words(G))]
    view = capi.kv_view(H, S, D, gs, G, sym, *[0 if a is None else a.data_ptr() for a in t])
    k, v = _half(gen, H, S, D), _half(gen, H, S, D)
    capi.quantize_cache(view, k.data_ptr(), v.data_ptr(), status.data_ptr(), src_f16=True)
    return view, t


def _cache_f8(gen, H, S, D, gs, slab_scale, status):
    k, v = _half(gen, H, S, D), _half(gen, H, S, D)
    G = (D + gs - 1) // gs
    if slab_scale:  # one scale per head, as a model's calibration gives it
        sides = []
        for a in (k, v):
            s = (a.abs().amax(dim=(1, 2)).float() / FP8_MAX).half()
            sides += [(a.float() / s.float()[:, None, None]).to(torch.float8_e4m3fn).view(torch.uint8), s]
        view = capi.kv_f8_view(H, S, D, gs, G, *[a.data_ptr() for a in sides])
        return view, sides
    t = [_bytes(H, S, D), _halves(H, S, G), _bytes(H, S, D), _halves(H, S, G)]
    view = capi.kv_f8_view(H, S, D, gs, G, *[a.data_ptr() for a in t])
    capi.quantize_cache_f8(view, k.data_ptr(), v.data_ptr(), status.data_ptr(), src_f16=True)
    return view, t


def _tables(gen, nseq, S, page, shared):
    """One block table per sequence over pages handed out in arbitrary order; with `shared`
    every four sequences have the pages of their first quarter in common."""
    n = (S + page - 1) // page
    prefix = n // 4 if shared else 0
    lots = (nseq + 3) // 4
    npages = lots * prefix + nseq * (n - prefix)
    free = torch.randperm(npages, device=DEV, generator=gen).to(torch.int32)
    head = free[: lots * prefix].view(lots, prefix).repeat_interleave(4, dim=0)[:nseq]
    tail = free[lots * prefix:].view(nseq, n - prefix)
    return torch.cat([head, tail], dim=1).contiguous(), npages


def _prepare_attn(case, gen):
    nseq, hkv, group, S, D, L = (case[k] for k in ("nseq", "hkv", "group", "S", "D", "layers"))
    fmt, page = case["fmt"], case["page"]
    H = nseq * hkv
    status = _ints(1)
    q, out = _half(gen, L, H * group, D), _halves(L, H * group, D)
    keep, calls = [q, status], []
    for i in range(L):
        qp, op = q[i].data_ptr(), out[i].data_ptr()
        if fmt == "f16":
            k, v = _half(gen, H, S, D), _half(gen, H, S, D)
            keep += [k, v]
            calls.append((capi.attention_fp16_flash, (qp, k.data_ptr(), v.data_ptr(), op, H, S, D),
                          {"group": group}))
        elif fmt == "f8":
            view, t = _cache_f8(gen, H, S, D, case["gs"], case["slab_scale"], status)
            keep.append(t)
            calls.append((capi.attention_f8_flash, (view, qp, op),
                          {"group": group, "scale_mode": int(case["slab_scale"])}))
        elif page:
            bt, npages = _tables(gen, nseq, S, page, case["shared"])
            pool, t = _cache_w4(gen, hkv, npages * page, D, case["gs"], case["sym"], status)
            pool.S = S  # the view's S is the logical length of a sequence
            keep += [bt, t]
            calls.append((capi.attention_w4_flash_paged_batched,
                          (pool, bt.data_ptr(), nseq, bt.shape[1], page, npages, group, qp, op), {}))
        else:
            view, t = _cache_w4(gen, H, S, D, case["gs"], case["sym"], status)
            keep.append(t)
            calls.append((capi.attention_w4_flash, (view, qp, op), {"group": group}))
    return {"run": _run_attn, "calls": calls, "out": out, "keep": keep}


def _run_attn(s):
    for call, args, options in s["calls"]:
        call(*args, **options)
    return s["out"]


def _prepare_kv(case, gen):
    H, S, D, gs, sym, L = (case[k] for k in ("H", "S", "D", "gs", "sym", "layers"))
    status = _ints(1)
    make = _cache_w4 if case["fmt"] == "w4" else _cache_f8
    caches = [make(gen, H, S, D, gs, sym if case["fmt"] == "w4" else False, status) for _ in range(L)]
    k, v = _half(gen, L, H, S, D), _half(gen, L, H, S, D)
    call = capi.quantize_cache if case["fmt"] == "w4" else capi.quantize_cache_f8
    return {"run": _run_kv, "call": call, "status": status, "keep": (k, v),
            "out": [a for _, t in caches for a in t if a is not None] + [status],
            "layers": [(view, k[i].data_ptr(), v[i].data_ptr()) for i, (view, _) in enumerate(caches)]}


def _run_kv(s):
    call, status = s["call"], s["status"].data_ptr()
    for view, k, v in s["layers"]:
        call(view, k, v, status, src_f16=True)
    return s["out"]


_PREPARE = {"gemm": _prepare_gemm, "act": _prepare_act, "attn": _prepare_attn, "kv": _prepare_kv}


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return _PREPARE[case["kind"]](case, gen)


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without -----------------------------------------------------------


def _cache_bytes(fmt, rows, D, gs, sym, slabs_with_one_scale=0):
    """Both sides of a cache of `rows` rows."""
    if fmt == "f16":
        return rows * D * 2 * 2
    G = (D + gs - 1) // gs
    if fmt == "f8":
        return 2 * (rows * D + 2 * (slabs_with_one_scale or rows * G))
    return 2 * rows * (_words(D) * 4 + 2 * G + (0 if sym else 4 * _words(G)))


def _weight_bytes(case):
    N, K = case["N"], case["K"]
    if case["kind"] == "act" or case["fmt"] == "mx":
        return N * _words(K) * 4 + N * ((K + 31) // 32)
    G = (K + case["gs"] - 1) // case["gs"]
    return N * (_words(K) * 4 + 2 * G + (0 if case["sym"] else 4 * _words(G)))


def work(case):
    L, kind = case["layers"], case["kind"]
    if kind in ("gemm", "act"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": L * (_weight_bytes(case) + 2 * M * (N + K)), "flops": L * 2 * M * N * K}
    if kind == "attn":
        nseq, hkv, group, S, D = (case[k] for k in ("nseq", "hkv", "group", "S", "D"))
        rows, tables = nseq * hkv * S, 0
        if case["page"]:
            n = (S + case["page"] - 1) // case["page"]
            again = (nseq - (nseq + 3) // 4) * (n // 4) if case["shared"] else 0
            rows -= again * case["page"] * hkv
            tables = 4 * nseq * n
        cache = _cache_bytes(case["fmt"], rows, D, case["gs"], case["sym"],
                             nseq * hkv if case["slab_scale"] else 0)
        heads = nseq * hkv * group
        return {"bytes": L * (cache + tables + 2 * 2 * heads * D), "flops": L * 4 * heads * S * D}
    rows, D = case["H"] * case["S"], case["D"]
    return {"bytes": L * (2 * 2 * rows * D + _cache_bytes(case["fmt"], rows, D, case["gs"], case["sym"])),
            "flops": L * 2 * 2 * rows * D}


def tolerance(case):
    # Caches are bytes that are fixed by the formats.  Products and attention round FP32 sums to
    # FP16 and may round a weight or a probability to FP16 on the way: against the same product in
    # FP64 the listed cases measured 2.1e-4 to 2.7e-4 of the result's norm and at most 1.05e-3 of
    # a value (or of the root mean square, for smaller values); four times that is allowed.
    if case["kind"] == "kv":
        return "exact"
    return {"rel": 1e-3, "max": 4e-3}
