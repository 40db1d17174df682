"""The cases by which the speed of the KV cache is judged.

A case is a dict of plain values. What an inference engine does with the cache
is a handful of calls, and each case is one of them (`kind`):

  fetch      KVCache.update_and_fetch(k, v, fetch=True): store new positions,
             return the visible dequantized K and V (the reference's own call)
  step       KVCache.decode_step: one new token of one sequence, one layer
  projected  KVCache.decode_step_projected: the same from raw projections
             through k_norm, RoPE and v_norm, K == V
  stack      one token through the 30 layers of a Gemma-4-26B-A4B-shaped model
             (every layer's decode_step), the whole of a decode step's cache work
  batch      PagedPool.decode_step: one new token of many ragged sequences
  prefill    KVCache.prefill_step: a prompt chunk on a sliding layer
  chunks     PagedPool.prefill_step: prompt chunks of one or several sequences,
             each after a prefix of its own

over the affine (4, 8 bits), TurboQuant codebook (2, 3, 4 bits; 3 is the
reference's default) and plain bf16 caches.

A pass leaves the cache ready for the next one of the same cost: rings
overwrite their oldest slots, a paged sequence's positions are the caller's
and stay where they are, and a linear cache is trimmed to the length it had
(`trim`), so that its visible length is the same on every pass.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..",
                                "gemma4-moe-flash-mlx-turbo_amd"))
import fmkv  # noqa: E402

MODES = {"affine": fmkv.MODE_AFFINE, "codebook": fmkv.MODE_CODEBOOK, "plain": fmkv.MODE_PLAIN}

# (KV heads, query heads, head_dim): the sliding and the global layers of
# Gemma-4-26B-A4B, and a smaller model's layer
SLIDING = {"Hkv": 8, "Hq": 16, "D": 256}
GLOBAL = {"Hkv": 2, "Hq": 16, "D": 512}
SMALL = {"Hkv": 4, "Hq": 8, "D": 128}

# positions that a linear cache holds beyond its first length: a pass appends
# one, and no program here makes as many passes on one cache
HEADROOM = 65536
# different tokens that the passes over one state go through in turn
STEPS = 64


def listed():
    return [
        # the store half and the fetch half of the reference's
        # update_and_fetch on a sliding layer, one token: the smallest call
        {"name": "fetch_ring_a4", "kind": "fetch", **SLIDING, "mode": "affine", "bits": 4,
         "window": 1024, "T": 3000, "n": 1, "f32": False},
        # one decoded token, sliding layer of a 4-bit model: launch latency
        {"name": "step_ring_a4", "kind": "step", **SLIDING, "mode": "affine", "bits": 4,
         "window": 1024, "T": 5000, "tau": 0.0, "f32": False},
        # one decoded token, global layer, 32K context, 8 bits
        {"name": "step_global_a8_32k", "kind": "step", **GLOBAL, "mode": "affine", "bits": 8,
         "window": 0, "T": 32768, "tau": 0.0, "f32": False},
        # the same layer from raw projections on the reference's default
        # cache (3-bit codebook), an odd context length
        {"name": "step_global_cb3_projected", "kind": "projected", **GLOBAL, "mode": "codebook",
         "bits": 3, "window": 0, "T": 20011, "tau": 0.0, "f32": False},
        # unquantized cache (--no-kv-quant), a middling context, f32 output
        {"name": "step_global_plain", "kind": "step", **GLOBAL, "mode": "plain", "bits": 16,
         "window": 0, "T": 9001, "tau": 0.0, "f32": True},
        # a whole decoded token: 25 sliding layers of 4 bits and 5 global
        # layers of 8 bits at 131072 positions
        {"name": "stack_a4_a8_128k", "kind": "stack", "mode": "affine", "bits": 4, "bits_global": 8,
         "window": 1024, "T": 131072, "f32": False},
        # a server's decode step: 32 ragged sequences, sliding-layer shape
        {"name": "batch32_a4", "kind": "batch", **SLIDING, "mode": "affine", "bits": 4,
         "n_seqs": 32, "T_min": 512, "T": 16384, "tau": 0.0, "f32": False},
        # a small server on default caches, global layers
        {"name": "batch8_cb3", "kind": "batch", **GLOBAL, "mode": "codebook", "bits": 3,
         "n_seqs": 8, "T_min": 300, "T": 9000, "tau": 0.0, "f32": False},
        # sparse-V decoding (--sparse-v-threshold) of two long conversations
        {"name": "batch2_a8_sparse", "kind": "batch", **GLOBAL, "mode": "affine", "bits": 8,
         "n_seqs": 2, "T_min": 20000, "T": 32768, "tau": 1e-3, "f32": False},
        # a prompt chunk on a global layer late in a long prompt
        {"name": "chunk_global_a8_32k", "kind": "chunks", **GLOBAL, "mode": "affine", "bits": 8,
         "n_seqs": 1, "T_min": 32768, "T": 32768, "n": 2048, "f32": False},
        # a prompt chunk on a sliding layer
        {"name": "prefill_ring_a4", "kind": "prefill", **SLIDING, "mode": "affine", "bits": 4,
         "window": 1024, "T": 6000, "n": 2048, "f32": False},
        # short follow-up messages of several conversations on default caches
        {"name": "chunks4_cb3", "kind": "chunks", **GLOBAL, "mode": "codebook", "bits": 3,
         "n_seqs": 4, "T_min": 700, "T": 8000, "n": 77, "f32": False},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    mode, bits = rng.choice([("affine", 4), ("affine", 8), ("codebook", 3), ("codebook", 3),
                             ("codebook", 2), ("codebook", 4), ("plain", 16)])
    f32 = rng.random() < 0.25
    tau = rng.choice([0.0, 0.0, 0.0, 1e-3, 1e-4])
    shape = rng.choice([SLIDING, GLOBAL, GLOBAL, SMALL])
    kind = rng.choice(["fetch", "step", "step", "projected", "batch", "batch", "prefill", "chunks",
                       "chunks", "stack"])
    base = {"kind": kind, **shape, "mode": mode, "bits": bits, "f32": f32}
    if kind == "fetch":
        window = rng.choice([0, _log(rng, 64, 4096)])
        return {**base, "window": window, "T": _log(rng, 64, 16384),
                "n": _log(rng, 1, 64) if window else 1}
    if kind in ("step", "projected"):
        window = rng.choice([0, 0, _log(rng, 64, 4096)])
        return {**base, "window": window, "T": _log(rng, 128, 65536), "tau": tau}
    if kind == "stack":
        return {"kind": kind, "mode": mode, "bits": bits, "bits_global": bits,
                "window": _log(rng, 512, 1024), "T": _log(rng, 1024, 65536), "f32": f32}
    if kind == "batch":
        n = rng.randint(2, 32)
        top = _log(rng, 512, 16384)
        return {**base, "n_seqs": n, "T_min": max(1, top // rng.randint(2, 16)), "T": top, "tau": tau}
    if kind == "prefill":
        return {**base, "window": _log(rng, 128, 2048), "T": _log(rng, 64, 8192),
                "n": _log(rng, 2, 2048)}
    n_seqs = rng.choice([1, 1, 2, 4, 8])
    n = _log(rng, 2, 2048 // n_seqs)
    top = _log(rng, 64, 32768 // max(1, n_seqs // 2))
    return {**base, "n_seqs": n_seqs, "T_min": max(1, top // rng.randint(1, 8)), "T": top, "n": n}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)


def _outliers(g, heads, D):
    """[heads, D] gains: four channels of a head are 20 times the others, as
    K and V of trained layers have them."""
    gain = torch.ones(heads, D, device="cuda")
    at = torch.rand(heads, D, generator=g, device="cuda").argsort(dim=1)[:, :4]
    return gain.scatter_(1, at, 20.0)


def _rows(g, shape, gain=None):
    """bf16 N(0, 1) rows [..., heads, D], times the heads' channel gains."""
    out = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    flat = out.view(-1, *shape[-2:])
    for i in range(0, flat.shape[0], 16384):
        x = torch.randn((min(16384, flat.shape[0] - i), *shape[-2:]), generator=g, device="cuda")
        flat[i:i + 16384] = x if gain is None else x * gain
    return out


def _scale(case, D):
    """The softmax scale: scores of a standard deviation of about 2.5, so that
    some dozens or hundreds of positions share the weight."""
    k_norm = 1.0 if case["kind"] == "projected" else math.sqrt((D + 4 * 399) / D)
    return 2.5 / (math.sqrt(D) * k_norm)


def _dtype(case):
    return torch.float32 if case["f32"] else torch.bfloat16


def _lengths(case, seed):
    """Positions that each sequence holds before the call, on the host."""
    g = torch.Generator().manual_seed(seed * 31 + 5)
    n, lo, hi = case["n_seqs"], case["T_min"], case["T"]
    lens = torch.randint(lo, hi + 1, (n,), generator=g)
    # the same total for every seed, so that passes on other inputs cost alike
    want = n * (lo + hi) // 2
    if hi > lo:
        lens = lens + (want - int(lens.sum())) // n
        lens = lens.clamp(lo, hi)
    return [int(x) for x in lens]


PROLOGUE = {"eps": 1e-6, "theta": 1e6}


def _rope_dims(D):
    return max(D // 4, 32)


def _inputs(case, seed):
    """The tensors of a single-sequence case: prefix K/V, then the calls' own."""
    g = _gen(seed)
    Hkv, Hq, D, T = case["Hkv"], case["Hq"], case["D"], case["T"]
    n = case.get("n", 1)
    calls = 1 if case["kind"] == "prefill" else STEPS
    gain = None if case["kind"] == "projected" else _outliers(g, Hkv, D)
    x = {"k0": _rows(g, (T, Hkv, D), gain), "k": _rows(g, (calls, n, Hkv, D), gain)}
    if case["kind"] == "projected":
        x["v0"], x["v"] = None, [None] * calls
        x["w"] = (1.0 + 0.1 * torch.randn(D, generator=g, device="cuda")).bfloat16()
    else:
        x["v0"], x["v"] = _rows(g, (T, Hkv, D), gain), _rows(g, (calls, n, Hkv, D), gain)
    if case["kind"] != "fetch":
        x["q"] = _rows(g, (calls, n, Hq, D))
    return x


def _new_cache(case, D, Hkv, window, bits, T):
    if case["mode"] == "plain":
        return fmkv.KVCache.new_with_window(D, window or None, Hkv, 0 if window else T + HEADROOM)
    return fmkv.KVCache.new_quantized_with_window(D, bits, window or None, Hkv,
                                                  0 if window else T + HEADROOM,
                                                  mode=MODES[case["mode"]])


def _layers(case):
    """(full attention?, Hkv, D, window, bits) of the stack's 30 layers."""
    types = (["sliding_attention"] * 5 + ["full_attention"]) * 5
    specs = fmkv.layer_cache_specs(types, 256, 8, global_head_dim=512, n_global_kv_heads=2,
                                   sliding_window=case["window"], attention_k_eq_v=True,
                                   kv_quant_bits=case["bits"],
                                   global_kv_quant_bits=case["bits_global"])
    return [(s.is_full, s.n_kv_heads, s.head_dim, s.window, s.bits) for s in specs]


def _stack_inputs(case, seed):
    """Prefixes (one for each kind of layer: its layers hold the same) and each
    layer's own token."""
    g = _gen(seed)
    x = {"layers": []}
    for full, (Hkv, D), T in ((False, (8, 256), min(case["T"], case["window"] + 40)),
                              (True, (2, 512), case["T"])):
        gain = _outliers(g, Hkv, D)
        x[full] = (gain, _rows(g, (T, Hkv, D), gain), _rows(g, (T, Hkv, D), gain))
    for full, Hkv, D, _, _ in _layers(case):
        gain = x[full][0]
        x["layers"].append((_rows(g, (1, Hkv, D), gain), _rows(g, (1, Hkv, D), gain),
                            _rows(g, (16, D))))
    return x


def _paged_inputs(case, seed):
    g = _gen(seed)
    Hkv, Hq, D = case["Hkv"], case["Hq"], case["D"]
    n = case.get("n", 1)
    gain = _outliers(g, Hkv, D)
    lens = _lengths(case, seed)
    prefix = [(_rows(g, (T, Hkv, D), gain), _rows(g, (T, Hkv, D), gain)) for T in lens]
    k = _rows(g, (len(lens), n, Hkv, D), gain)
    v = _rows(g, (len(lens), n, Hkv, D), gain)
    q = _rows(g, (len(lens), n, Hq, D))
    return lens, prefix, k, v, q


def prepare(case, seed):
    if case["kind"] == "stack":
        x = _stack_inputs(case, seed)
        caches = []
        for full, Hkv, D, window, bits in _layers(case):
            cache = _new_cache(case, D, Hkv, window, bits, case["T"])
            _, k, v = x[full]
            for i in range(0, k.shape[0], 8192):
                cache.append(k[i:i + 8192], v[i:i + 8192])
            caches.append(cache)
        return {"case": case, "caches": caches, "calls": x["layers"], "dtype": _dtype(case),
                "scales": [_scale(case, layer[2]) for layer in _layers(case)]}
    D, Hkv = case["D"], case["Hkv"]
    state = {"case": case, "scale": _scale(case, D), "dtype": _dtype(case), "i": 0}
    if case["kind"] in ("batch", "chunks"):
        lens, prefix, k, v, q = _paged_inputs(case, seed)
        n = k.shape[1]
        need = [(T + n + 15) // 16 for T in lens]
        width = max(need)
        order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).int()
        table = torch.zeros(len(lens), width, dtype=torch.int32)
        at = 0
        for s, nb in enumerate(need):
            table[s, :nb] = order[at:at + nb]
            at += nb
        table = table.cuda()
        pool = fmkv.PagedPool(fmkv.make_desc(Hkv, D, case["bits"], mode=MODES[case["mode"]]), sum(need))
        for s, (k0, v0) in enumerate(prefix):
            for i in range(0, k0.shape[0], 8192):
                pool.append(k0[None, i:i + 8192], v0[None, i:i + 8192], table[s:s + 1],
                            torch.tensor([i], dtype=torch.int32, device="cuda"))
        start = torch.tensor(lens, dtype=torch.int32, device="cuda")
        state.update(pool=pool, table=table, start=start, lens=start + n, longest=max(lens) + n,
                     k=k, v=v, q=q[:, 0].contiguous() if case["kind"] == "batch" else q)
        return state
    x = _inputs(case, seed)
    cache = _new_cache(case, D, Hkv, case["window"], case["bits"], case["T"])
    if case["kind"] == "projected":
        state["prologue"] = fmkv.make_prologue(x["w"], PROLOGUE["eps"], _rope_dims(D),
                                               PROLOGUE["theta"], v_from_k=True)
    for i in range(0, case["T"], 8192):
        if case["kind"] == "projected":
            cache.append_projected(x["k0"][i:i + 8192], None, state["prologue"])
        else:
            cache.append(x["k0"][i:i + 8192], x["v0"][i:i + 8192])
    # what each pass is given, cut before: a program has its own rows at hand
    q = x.get("q")
    if q is not None and case["kind"] != "prefill":
        q = q[:, 0]
    calls = x["k"].shape[0]
    state["calls"] = [(x["k"][i], x["v"][i], None if q is None else q[i]) for i in range(calls)]
    state["cache"] = cache
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "stack":
        outs = []
        for cache, (k, v, q), scale in zip(state["caches"], state["calls"], state["scales"]):
            if cache.desc.window == 0:
                cache.trim(case["T"])
            outs.append(cache.decode_step(k, v, q, scale, dtype=state["dtype"]))
        return outs
    if kind == "batch":
        return state["pool"].decode_step(state["k"], state["v"], state["table"], state["start"],
                                         state["lens"], state["longest"], state["q"], state["scale"],
                                         case["tau"], dtype=state["dtype"])
    if kind == "chunks":
        return state["pool"].prefill_step(state["k"], state["v"], state["table"], state["start"],
                                          state["q"], state["scale"], dtype=state["dtype"])
    cache = state["cache"]
    k, v, q = state["calls"][state["i"] % len(state["calls"])]
    state["i"] += 1
    if kind == "prefill":
        return cache.prefill_step(k, v, q, state["scale"], dtype=state["dtype"])
    if case["window"] == 0:
        cache.trim(case["T"])
    if kind == "step":
        return cache.decode_step(k, v, q, state["scale"], case["tau"], dtype=state["dtype"])
    if kind == "projected":
        return cache.decode_step_projected(k, None, state["prologue"], q, state["scale"],
                                           case["tau"], dtype=state["dtype"])
    # fetch: the caller's dtype goes through peek_kv where it is not the default
    if not case["f32"]:
        return cache.update_and_fetch(k, v, fetch=True)
    cache.update_and_fetch(k, v)
    return cache.peek_kv(dtype=torch.float32)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _token_bytes(mode, bits, D):
    """Stored bytes of one position of one KV head, K and V."""
    if mode == "plain":
        return 4 * D
    if mode == "codebook":
        return 2 * (D * bits // 8 + 2)
    return 2 * (D * bits // 8 + D // 64 * 4)


def work(case):
    out = 4 if case["f32"] else 2
    if case["kind"] == "stack":
        w = {"bytes": 0, "flops": 0}
        for full, Hkv, D, window, bits in _layers(case):
            seen = min(case["T"] + 1, window) if window else case["T"] + 1
            w["bytes"] += seen * Hkv * _token_bytes(case["mode"], bits, D)
            w["bytes"] += Hkv * D * 4 + 16 * D * (2 + out)
            w["flops"] += 4 * 16 * D * seen
        return w
    Hkv, D = case["Hkv"], case["D"]
    per = Hkv * _token_bytes(case["mode"], case["bits"], D)
    n = case.get("n", 1)
    if case["kind"] == "fetch":
        seen = min(case["T"] + n, case["window"] or case["T"] + n)
        return {"bytes": n * Hkv * D * 4 + n * per + seen * (per + Hkv * D * 2 * out), "flops": 0}
    Hq = case["Hq"]
    if case["kind"] in ("batch", "chunks"):
        mean = (case["T_min"] + case["T"]) / 2 if case["T"] > case["T_min"] else case["T"]
        seqs = [mean] * case["n_seqs"]
    else:
        seqs = [case["T"]]
    total = {"bytes": 0, "flops": 0}
    for T in seqs:
        window = case.get("window", 0)
        if window and T + n > window:
            pairs = sum(min(T + i + 1, window) for i in range(n))
            seen = min(T + n, window + n - 1)
        else:
            pairs = n * T + n * (n + 1) // 2
            seen = T + n
        total["bytes"] += seen * per + n * (Hkv * D * 4 + Hq * D * (2 + out))
        total["flops"] += 4 * Hq * D * pairs
    return total


def tolerance(case):
    if case.get("tau", 0.0) > 0.0:
        # a weight within rounding of the threshold may fall on either side
        return {"rel": 1e-2, "max": 0.2}
    if case["f32"]:
        # f32 sums in another order (other splits of the same positions): 2e-6
        # on plain caches, 2e-5 on affine and 9e-5 on codebook ones, whose
        # weights times value scales go through pairs of f16
        return {"rel": {"plain": 1e-5, "affine": 1e-4, "codebook": 4e-4}[case["mode"]]}
    # bf16 results: values that round to the other neighbour
    return {"rel": 2e-3, "max": 0.05}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

CENTROIDS = {
    2: ([0.453, 1.510], [0.0, 0.982]),
    3: ([0.245, 0.756, 1.344, 2.152], [0.0, 0.501, 1.050, 1.748]),
    4: ([0.128, 0.388, 0.657, 0.942, 1.256, 1.618, 2.069, 2.733],
        [0.0, 0.258, 0.522, 0.800, 1.099, 1.437, 1.844, 2.401]),
}


def _signs(D):
    s, state = [], 42
    for _ in range(D):
        state = (state * 6364136223846793005 + 1442695040888963407) % (1 << 64)
        s.append(-1.0 if state >> 63 else 1.0)
    return torch.tensor(s, dtype=torch.float64, device="cuda")


def _hadamard(x):
    """x . H / sqrt(D) over the last dimension."""
    D = x.shape[-1]
    shape, h = x.shape, 1
    x = x.reshape(-1, D)
    while h < D:
        a = x.view(-1, D // (2 * h), 2, h)
        x = torch.stack((a[:, :, 0] + a[:, :, 1], a[:, :, 0] - a[:, :, 1]), dim=2).reshape(-1, D)
        h *= 2
    return (x / math.sqrt(D)).view(shape)


def _half(x):
    return x.float().half().double()


def _stored(x, mode, bits):
    """What a cache holds of rows x [..., D] (f64): in the rotated basis
    unless plain."""
    if mode == "plain":
        return x.bfloat16().double()
    D = x.shape[-1]
    s = _signs(D)
    if mode == "codebook":
        # z = (x / |x|) R sqrt(D), the bin whose bounds hold it
        norm = x.float().double().square().sum(-1, keepdim=True).sqrt()
        z = _hadamard(x / (norm + 1e-8)) * s * math.sqrt(D)
        cent, bound = CENTROIDS[bits]
        cent = torch.tensor([-c for c in reversed(cent)] + cent, dtype=torch.float64, device="cuda")
        bound = torch.tensor([-b for b in reversed(bound[1:])] + bound, dtype=torch.float32,
                             device="cuda").double()
        at = torch.bucketize(z, bound, right=True)
        return cent.float().double()[at] * _half(norm) / math.sqrt(D)
    y = (_hadamard(x) * s).view(*x.shape[:-1], D // 64, 64)
    top, low = y.amax(-1, keepdim=True), y.amin(-1, keepdim=True)
    scale = ((top - low) / ((1 << bits) - 1)).clamp_min(1e-7)
    side = low.abs() > top.abs()
    scale = torch.where(side, scale, -scale)
    edge = torch.where(side, low, top)
    q0 = torch.round(edge / scale)
    scale = torch.where(q0 != 0, edge / torch.where(q0 != 0, q0, 1.0), scale)
    bias = torch.where(q0 != 0, edge, 0.0)
    code = torch.round((y - bias) / scale).clamp(0, (1 << bits) - 1)
    return (code * _half(scale) + _half(bias)).view(x.shape)


def _many(f, x, *more):
    """f over slices of the rows, to bound the memory of its steps."""
    return torch.cat([f(x[i:i + 8192], *[m[i:i + 8192] for m in more])
                      for i in range(0, x.shape[0], 8192)])


def _attend(case, mode, q, k, v, first, start, window, scale):
    """q [n, Hq, D] at positions start .. over stored k, v [T, Hkv, D] of
    positions first ..: [n, Hq, D] in f64."""
    n, Hq, D = q.shape
    rep = Hq // k.shape[1]
    q = q.double()
    if mode != "plain":
        s = _signs(D)
        q = _hadamard(q) * s
    pos = torch.arange(first, first + k.shape[0], device="cuda")
    at = torch.arange(start, start + n, device="cuda")[:, None]
    hidden = pos[None] > at
    if window:
        hidden |= pos[None] <= at - window
    out = torch.empty(n, Hq, D, dtype=torch.float64, device="cuda")
    for h in range(k.shape[1]):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for g in range(h * rep, (h + 1) * rep):
            w = torch.mm(q[:, g].contiguous(), kt).mul_(scale).masked_fill_(hidden, -math.inf)
            w = torch.softmax(w, dim=1)
            tau = case.get("tau", 0.0)
            if tau > 0.0:
                w = torch.where(w < tau, 0.0, w)
            out[:, g] = torch.mm(w, vh)
    if mode != "plain":
        out = _hadamard(out * s)
    return out


def _projected(case, x, w, first):
    """K and V rows that the prologue makes of raw rows x [n, Hkv, D]."""
    D = case["D"]
    y = x.double()
    r = 1.0 / (y.square().mean(-1, keepdim=True) + PROLOGUE["eps"]).sqrt()
    k = (y * r * w.double()).bfloat16().double()
    half = _rope_dims(D) // 2
    # the angle is formed in 32 bits, as the model's rope does
    freq = (PROLOGUE["theta"] ** (-torch.arange(half, dtype=torch.float64, device="cuda") / half)).float()
    pos = torch.arange(first, first + x.shape[0], dtype=torch.float32, device="cuda")
    angle = (pos[:, None] * freq).double()[:, None]
    a, b = k[..., :half].clone(), k[..., half:2 * half].clone()
    k[..., :half] = a * angle.cos() - b * angle.sin()
    k[..., half:2 * half] = a * angle.sin() + b * angle.cos()
    k = k.bfloat16().double()
    square = x.float().square().bfloat16().double()
    mean = square.mean(-1, keepdim=True).bfloat16().double()
    return k, y / (mean + PROLOGUE["eps"]).sqrt()


def exact(case, seed):
    mode = case["mode"]
    if case["kind"] == "stack":
        x = _stack_inputs(case, seed)
        held = {}
        outs = []
        for (full, Hkv, D, window, bits), (k, v, q) in zip(_layers(case), x["layers"]):
            if full not in held:
                held = {full: [_many(lambda r: _stored(r.double(), mode, bits), y) for y in x[full][1:]]}
            kv = [torch.cat((old, _stored(new.double(), mode, bits))) for old, new in zip(held[full], (k, v))]
            T = kv[0].shape[0]
            outs.append(_attend(case, mode, q[None], *kv, 0, T - 1, window, _scale(case, D))[0])
        return outs
    D, bits = case["D"], case["bits"]
    scale = _scale(case, D)
    if case["kind"] in ("batch", "chunks"):
        lens, prefix, k, v, q = _paged_inputs(case, seed)
        outs = []
        for s, T in enumerate(lens):
            kv = [_many(lambda r: _stored(r.double(), mode, bits), torch.cat((old, new[s])))
                  for old, new in zip(prefix[s], (k, v))]
            outs.append(_attend(case, mode, q[s], *kv, 0, T, 0, scale))
        outs = torch.stack(outs)
        return outs[:, 0] if case["kind"] == "batch" else outs
    x = _inputs(case, seed)
    T, n, window = case["T"], x["k"].shape[1], case["window"]
    first = max(0, T - window) if window else 0
    k = torch.cat((x["k0"][first:], x["k"][0]))
    if case["kind"] == "projected":
        k, v = _projected(case, k, x["w"], first)
    else:
        k, v = k.double(), torch.cat((x["v0"][first:], x["v"][0])).double()
    k, v = (_many(lambda r: _stored(r, mode, bits), y) for y in (k, v))
    if case["kind"] == "fetch":
        if window:
            k, v = k[-window:], v[-window:]
        if mode != "plain":
            s = _signs(D)
            k, v = (_many(lambda r: _hadamard(r * s), y) for y in (k, v))
        return k, v
    out = _attend(case, mode, x["q"][0], k, v, first, T, window, scale)
    return out if case["kind"] == "prefill" else out[0]
