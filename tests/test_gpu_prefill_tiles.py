"""Prefill attention at the edges of its tiles: 64 query rows of a work-group
(64 / G positions), steps of 32 keys in two 16-key blocks, and the 16-key
block that a chunk's first position cuts. Every mode and head_dim, a chunk
shorter than, as long as and one longer than a row tile after prefixes that
end inside, at and past a block and a step; and soft softmax (many positions
share the weight, so a dropped or doubled key shows) over a few hundred keys.
f32 outputs against the oracle's exact attention, both of the same stored rows:
each value is a weighted mean of stored rows. A score is below 2^6 in
magnitude and a sum of f32 terms good to a few units in the last place,
2^-22, so a weight is good to 2^-16 relative (the bf16 pairs of plain caches:
2^-17), and a value, at most 2^8 (N(0, 1) times 20 times 3.05), to 2^-8 = 4e-3
at worst. On average a value is 2^3 (the rows' scale of up to 3 and the
outliers together) and the same 2^-16 bounds its error to 2^-13 = 1.2e-4; a
lost residual part (2^-12 of every weight at least) or a key missed or taken
twice among the few hundred is at 2e-3 there."""
import numpy as np
import pytest

from gpu_util import dev_bf16, kv_batch

pytestmark = pytest.mark.gpu

SHAPES = [  # mode, D, bits, Hkv, Hq
    (0, 512, 8, 1, 8), (0, 512, 4, 1, 4), (0, 256, 4, 2, 4), (0, 256, 8, 1, 1),
    (0, 128, 8, 1, 8), (0, 128, 4, 2, 2), (1, 512, 3, 1, 8), (1, 512, 4, 1, 2),
    (1, 256, 2, 2, 4), (1, 256, 3, 1, 3), (1, 128, 3, 1, 4), (1, 128, 4, 1, 2),
    (2, 512, 16, 1, 8), (2, 256, 16, 2, 4), (2, 128, 16, 1, 5),
]


def soft_q(seed, n, Hq, D):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, Hq, D)).astype(np.float32)
    return (x.view(np.uint32) >> 16).astype(np.uint16)


@pytest.mark.parametrize("mode,D,bits,Hkv,Hq", SHAPES)
@pytest.mark.parametrize("window", [0, 48])
def test_prefill_tile_edges(gpu, ora, mode, D, bits, Hkv, Hq, window):
    import torch

    tile = 64 // (Hq // Hkv)
    for prefix, n in ((0, 1), (0, tile + 1), (15, tile), (16, tile - 1 or 1), (31, 17), (33, tile + 1),
                      (300, 2 * tile + 1), (640, tile), (655, tile + 1), (672, 1), (687, 17)):
        cap = 0 if window else prefix + n
        if mode == 2:
            cache = gpu.KVCache.new_with_window(D, window or None, Hkv, cap)
        else:
            cache = gpu.KVCache.new_quantized_with_window(D, bits, window or None, Hkv, cap, mode=mode)
        oc = ora.OracleCache(Hkv, D, bits, window, cap, mode=mode)
        if prefix:
            k, v = kv_batch(prefix, prefix, Hkv, D), kv_batch(prefix + 1, prefix, Hkv, D)
            cache.append(dev_bf16(k), dev_bf16(v))
            oc.append(k, v)
        k, v = kv_batch(n + 2, n, Hkv, D), kv_batch(n + 3, n, Hkv, D)
        q = soft_q(n, n, Hq, D)
        scale = 0.3 / np.sqrt(D)
        out = cache.prefill_step(dev_bf16(k), dev_bf16(v), dev_bf16(q), scale, dtype=torch.float32)
        torch.cuda.synchronize()
        err = np.abs(out.cpu().numpy().astype(np.float64) - oc.prefill(k, v, q, scale))
        assert err.max() < 4e-3 and err.mean() < 1.2e-4, f"prefix {prefix} n {n}: {err.max():.2e} {err.mean():.2e}"


@pytest.mark.parametrize("mode,D,bits,Hq", [(0, 512, 8, 8), (1, 256, 3, 4), (2, 128, 16, 8)])
def test_prefill_split_ragged_and_captured(gpu, ora, mode, D, bits, Hq):
    """A few rows of ragged sequences (one too short for a second key range,
    one long, one that starts at its chunk), split over the keys; twice in a
    row, then on a second stream right after the first, then captured (there
    unsplit) and replayed: the oracle's result each time; the same bits from every split call."""
    import torch

    starts, n, Hkv = [20, 1500, 0, 333], 5, 1
    need = [(p + n + 15) // 16 for p in starts]
    table = np.zeros((len(starts), max(need)), np.int32)
    at = 0
    for s, nb in enumerate(need):
        table[s, :nb] = np.arange(at, at + nb)[::-1]
        at += nb
    pool = gpu.PagedPool(gpu.make_desc(Hkv, D, bits, mode=mode), at)
    dtab = torch.from_numpy(table).cuda()
    dstart = torch.tensor(starts, dtype=torch.int32, device="cuda")
    k, v = kv_batch(1, len(starts) * n, Hkv, D), kv_batch(2, len(starts) * n, Hkv, D)
    q = soft_q(3, len(starts) * n, Hq, D)
    shape = (len(starts), n, -1, D)
    k, v, q = k.reshape(shape), v.reshape(shape), q.reshape(shape)
    scale = 0.3 / np.sqrt(D)
    want = []
    for s, p in enumerate(starts):
        oc = ora.OracleCache(Hkv, D, bits, 0, p + n, mode=mode)
        if p:
            k0, v0 = kv_batch(10 + s, p, Hkv, D), kv_batch(20 + s, p, Hkv, D)
            oc.append(k0, v0)
            pool.append(dev_bf16(k0)[None], dev_bf16(v0)[None], dtab[s:s + 1],
                        torch.zeros(1, dtype=torch.int32, device="cuda"))
        want.append(oc.prefill(k[s], v[s], q[s], scale))
    want = np.stack(want)
    dk, dv, dq = dev_bf16(k), dev_bf16(v), dev_bf16(q)

    def call():
        return pool.prefill_step(dk, dv, dtab, dstart, dq, scale, dtype=torch.float32)

    def check(out, what):
        err = np.abs(out.cpu().numpy().astype(np.float64) - want)
        # (a codebook row's reconstruction is not bounded by its largest value,
        # as the bound above takes it: the path's own 2e-2 for the worst value,
        # the mean bound as above)
        assert err.max() < 2e-2 and err.mean() < 1.2e-4, f"{what}: {err.max():.2e} {err.mean():.2e}"

    first, second = call(), call()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    third = call()
    with torch.cuda.stream(side):
        fourth = call()
    torch.cuda.synchronize()
    check(first, "split")
    for o in (second, third, fourth):
        assert torch.equal(first, o)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        captured = call()
    for i in range(3):
        captured.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(captured, f"replay {i}")
        assert torch.equal(first, call())


@pytest.mark.parametrize("mode,D,bits,Hq,amp", [
    (0, 512, 4, 8, 3700.0), (0, 256, 4, 4, 3700.0), (0, 128, 4, 2, 3700.0), (0, 512, 8, 8, 62000.0),
    (0, 128, 8, 4, 62000.0), (1, 512, 4, 8, 450.0), (1, 256, 4, 2, 450.0), (1, 128, 4, 4, 450.0),
    (0, 512, 4, 8, 7500.0), (0, 256, 4, 4, 7500.0), (0, 128, 4, 1, 7500.0), (1, 512, 4, 4, 900.0),
    (1, 128, 4, 1, 900.0)])
@pytest.mark.parametrize("n,rise", [(5, 7.75), (5, 6.9), (600, 7.75), (600, 6.9)])
def test_prefill_weights_beyond_f16(gpu, ora, mode, D, bits, Hq, amp, n, rise):
    """V scales of up to 483 (affine; valid below 511) and, past that, 950, and
    norms / sqrt(D) of 450 and 900 (4-bit codebook), behind scores that rise
    (base 2) after the first keys by less and by more than what moves the
    reference maximum: weights p * scale of up to 1.1e5 where that is past
    f16's 65504. There the pair is 65504 and a residual r <= 65504 rounded or
    cut to 2^-10 of itself, hence good to 2^-11 of the weight, and the value
    to 2^-11 of the longest row that it averages."""
    import torch

    prefix, Hkv = 700, 1
    cap = prefix + n
    rng = np.random.default_rng(n + D)

    def bf16(x):
        return (np.ascontiguousarray(x, np.float32).view(np.uint32) >> 16).astype(np.uint16)

    u = rng.standard_normal(D).astype(np.float32)
    k = np.tile(u, (cap, Hkv, 1))
    k[:48] = 0.0
    oc = ora.OracleCache(Hkv, D, bits, 0, cap, mode=mode)
    if mode == 0:  # uniform in the stored basis: scale = range / codes, biases within f16
        y = rng.uniform(-1.0, 1.0, (cap, Hkv, D)) * rng.uniform(0.65 * amp, amp, (cap, 1, 1))
        v = ora.unrotate_rows_f64(y, oc.sgn)
    else:  # rows of one norm
        v = rng.standard_normal((cap, Hkv, D))
        v *= amp * np.sqrt(D) / np.linalg.norm(v, axis=-1, keepdims=True)
    k, v, q = bf16(k), bf16(v), np.tile(bf16(u), (n, Hq, 1))
    oc.append(k[:prefix], v[:prefix])
    ks, vs = oc.dequant_kv()
    score = float(ks[-1, 0] @ (q[0, 0].astype(np.uint32) << 16).view(np.float32))
    scale = float(np.float32(rise * np.log(2.0) / score))
    held = oc.meta[:prefix, 1, 0].view(np.float16).astype(np.float64)
    held = np.abs(held[:, 0::2]) if mode == 0 else held / np.sqrt(D)
    assert 450 <= 1.01 * held.max() and 2.0 ** 6.9 * held.max() < 131008
    cache = gpu.KVCache(gpu.make_desc(Hkv, D, bits, 0, cap, mode))
    cache.append(dev_bf16(k[:prefix]), dev_bf16(v[:prefix]))
    out = cache.prefill_step(dev_bf16(k[prefix:]), dev_bf16(v[prefix:]), dev_bf16(q), scale,
                             dtype=torch.float32)
    torch.cuda.synchronize()
    err = np.abs(out.cpu().numpy().astype(np.float64) - oc.prefill(k[prefix:], v[prefix:], q, scale))
    bound = 2.0 ** -11 * np.sqrt((vs ** 2).sum(-1).max())
    assert np.isfinite(err).all() and err.max() < bound, f"{err.max():.3e} of {bound:.3e}"


@pytest.mark.parametrize("mode,D,bits,Hq", [
    (0, 512, 8, 8), (0, 256, 4, 4), (0, 128, 8, 2), (1, 512, 4, 8), (1, 256, 3, 4), (1, 128, 2, 1),
    (2, 512, 16, 8), (2, 256, 16, 4), (2, 128, 16, 1)])
@pytest.mark.parametrize("window,bad", [(0, 707), (0, 723), (600, 113), (600, 701)])
@pytest.mark.parametrize("n", [60, 2100])
def test_prefill_hides_infinite_rows(gpu, ora, mode, D, bits, Hq, window, bad, n):
    """A position whose V is infinite or past what a scale or norm holds: the queries before it and those whose window has left it are the
    finite results of the other rows (n = 2100: on grids of their own, not
    split over the keys); those that see it are not finite. bad: inside and at
    the edge of the chunk's first key blocks, or in the prefix."""
    import torch

    prefix, Hkv = 693, 1
    cap = prefix + n

    def caches():
        return (gpu.KVCache(gpu.make_desc(Hkv, D, bits, window, 0 if window else cap, mode)),
                ora.OracleCache(Hkv, D, bits, window, 0 if window else cap, mode=mode))

    cache, oc = caches()
    k, v = kv_batch(n, cap, Hkv, D), kv_batch(n + 1, cap, Hkv, D)
    vx = v.copy()
    vx[bad, 0, 3] = 0xff80 if mode == 2 else 0x7f00  # -inf (else 1.7e38)
    q = soft_q(n, n, Hq, D)
    scale = 0.3 / np.sqrt(D)
    cache.append(dev_bf16(k[:prefix]), dev_bf16(vx[:prefix]))
    oc.append(k[:prefix], v[:prefix])
    out = cache.prefill_step(dev_bf16(k[prefix:]), dev_bf16(vx[prefix:]), dev_bf16(q), scale,
                             dtype=torch.float32).cpu().numpy().astype(np.float64)
    pos = np.arange(prefix, cap)
    sees = (pos >= bad) & ((pos < bad + window) if window else True)
    rows = np.nonzero(~sees)[0]
    rows = rows[(np.abs(pos[rows] - bad) < 80) | (np.abs(pos[rows] - bad - window) < 80)]
    assert rows.size and sees.any() and not np.isfinite(out[sees]).all(axis=(1, 2)).any()
    err = np.abs(out[rows] - oc.prefill(k[prefix:], v[prefix:], q, scale, rows=rows))
    assert np.isfinite(out[~sees]).all()
    assert err.max() < 2e-2 and err.mean() < 1.2e-4, f"{err.max():.2e} {err.mean():.2e}"


# every kernel instance: mode, bits, D
INSTANCES = [(m, b, D) for m, bits in ((0, (4, 8)), (1, (2, 3, 4)), (2, (16,))) for b in bits for D in (128, 256, 512)]


@pytest.mark.parametrize("mode,bits,D", INSTANCES)
@pytest.mark.parametrize("prefix,n,wide", [(70, 3, 0), (70, 3, 3000), (1200, 3, 3000), (1, 97, 0), (1201, 97, 3000),
                                           (1200, 800, 0), (30, 2100, 0)])
def test_prefill_grids(gpu, ora, mode, bits, D, prefix, n, wide):
    """Grids of 1, 13, 100 and 263 work-groups over short and long contexts,
    on tables as wide as the sequence and far wider: rows shared by eight
    waves or not, one key range or several, a merge that finds nothing to
    merge. Every row finite, the first and last tiles' rows against the
    oracle's exact attention. (A codebook row's reconstruction is not bounded
    by its largest value: the path's own 2e-2 for the worst value there.)"""
    import torch

    Hkv, Hq, cap = 1, 8, prefix + n
    oc = ora.OracleCache(Hkv, D, bits, 0, cap, mode=mode)
    nb = (cap + 15) // 16
    pool = gpu.PagedPool(gpu.make_desc(Hkv, D, bits, mode=mode), nb)
    table = torch.zeros((1, max(nb, wide)), dtype=torch.int32, device="cuda")
    table[0, :nb] = torch.arange(nb - 1, -1, -1, dtype=torch.int32, device="cuda")
    k, v = kv_batch(prefix, cap, Hkv, D), kv_batch(prefix + 1, cap, Hkv, D)
    q = soft_q(n, n, Hq, D)
    scale = 0.3 / np.sqrt(D)
    oc.append(k[:prefix], v[:prefix])
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    pool.append(dev_bf16(k[:prefix])[None], dev_bf16(v[:prefix])[None], table, zero)
    args = [dev_bf16(x)[None] for x in (k[prefix:], v[prefix:], q)]
    out = pool.prefill_step(args[0], args[1], table, zero + prefix, args[2], scale, dtype=torch.float32)
    torch.cuda.synchronize()
    out = out.cpu().numpy().astype(np.float64)[0]
    assert np.isfinite(out).all()
    rows = sorted({*range(min(n, 9)), *range(max(0, n - 9), n), n // 2})
    err = np.abs(out[rows] - oc.prefill(k[prefix:], v[prefix:], q, scale, rows=rows))
    assert err.max() < (2e-2 if mode == 1 else 4e-3) and err.mean() < 1.2e-4, f"{err.max():.2e} {err.mean():.2e}"


@pytest.mark.parametrize("mode,bits,D", [(0, 4, 128), (1, 3, 256), (2, 16, 128), (0, 8, 512)])
@pytest.mark.parametrize("n", [3, 100])
def test_prefill_longest_length_given(gpu, ora, mode, bits, D, n):
    """max_seq_len on a wide table: the bits of the call on a table of that
    width; far too small or too large ones: the oracle's result all the same."""
    import torch

    starts, Hkv, Hq = [600, 40, 0, 1500], 1, 4
    need = [(p + n + 15) // 16 for p in starts]
    wide = torch.zeros((4, 2000), dtype=torch.int32, device="cuda")
    pool = gpu.PagedPool(gpu.make_desc(Hkv, D, bits, mode=mode), sum(need))
    start = torch.tensor(starts, dtype=torch.int32, device="cuda")
    k, v = kv_batch(n, 4 * n, Hkv, D).reshape(4, n, Hkv, D), kv_batch(n + 1, 4 * n, Hkv, D).reshape(4, n, Hkv, D)
    q = soft_q(n, 4 * n, Hq, D).reshape(4, n, Hq, D)
    scale, want, at = 0.3 / np.sqrt(D), [], 0
    for s, p in enumerate(starts):
        wide[s, :need[s]] = torch.arange(at, at + need[s], dtype=torch.int32, device="cuda")
        at += need[s]
        oc = ora.OracleCache(Hkv, D, bits, 0, p + n, mode=mode)
        if p:
            k0, v0 = kv_batch(50 + s, p, Hkv, D), kv_batch(60 + s, p, Hkv, D)
            oc.append(k0, v0)
            pool.append(dev_bf16(k0)[None], dev_bf16(v0)[None], wide[s:s + 1], start[2:3])
        want.append(oc.prefill(k[s], v[s], q[s], scale))
    want, args = np.stack(want), [dev_bf16(x) for x in (k, v, q)]

    def call(table, longest):
        return pool.prefill_step(args[0], args[1], table, start, args[2], scale, dtype=torch.float32,
                                 max_seq_len=longest)

    exact = call(wide[:, :max(need)].contiguous(), 0)
    assert torch.equal(exact, call(wide, max(starts) + n))
    for longest in (0, 1, 300, 32000, 1 << 30):
        err = np.abs(call(wide, longest).cpu().numpy().astype(np.float64) - want)
        assert err.max() < (2e-2 if mode == 1 else 4e-3) and err.mean() < 1.2e-4, f"{longest}: {err.max():.2e}"
    with pytest.raises(gpu.Exception_):
        call(wide, -1)
