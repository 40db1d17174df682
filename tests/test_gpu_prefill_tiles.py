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
                      (300, 2 * tile + 1)):
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
