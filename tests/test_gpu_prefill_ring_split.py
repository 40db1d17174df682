"""Key-split prefill on a ring: short chunks on layers of some hundreds of
positions' window, past a wrap. The key ranges cut across the two stores (the
ring, then the staged chunk), the block that the chunk's start cuts is visited
once per store, and a range may hold nothing that a row sees. Windows that are
and are not whole head-blocks, chunks that start at a block and inside one.
f32 outputs against the oracle's exact attention with soft weights, whose mean
a key missed or taken twice would move (bounds as in test_gpu_prefill_tiles);
stored slots bit-exact afterwards."""
import numpy as np
import pytest

from gpu_util import check_codes, dev_bf16, kv_batch
from test_gpu_prefill_tiles import INSTANCES, soft_q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,bits,D", INSTANCES)
@pytest.mark.parametrize("W", [300, 1000, 1024])
def test_ring_split_chunks(gpu, ora, mode, bits, D, W):
    import torch

    Hkv, Hq = 2, 8
    cache = gpu.KVCache(gpu.make_desc(Hkv, D, bits, W, 0, mode))
    oc = ora.OracleCache(Hkv, D, bits, W, mode=mode)
    # 16-aligned and unaligned starts past the first wrap; 400: two and four waves a work-group
    for i, n in enumerate((W + 16 - W % 16 + 64, 1, 17, 77, 16, 5, 400, 77)):
        k, v = kv_batch(100 * i + W, n, Hkv, D), kv_batch(100 * i + W + 1, n, Hkv, D)
        if i == 0:
            cache.append(dev_bf16(k), dev_bf16(v))
            oc.append(k, v)
            continue
        q = soft_q(i, n, Hq, D)
        scale = 0.3 / np.sqrt(D)
        out = cache.prefill_step(dev_bf16(k), dev_bf16(v), dev_bf16(q), scale, dtype=torch.float32)
        rows = sorted({*range(min(n, 4)), n // 2, n - 2 if n > 1 else 0, n - 1})
        err = np.abs(out.cpu().numpy().astype(np.float64)[rows] - oc.prefill(k, v, q, scale, rows=rows))
        assert torch.isfinite(out).all()
        assert err.max() < (2e-2 if mode == 1 else 4e-3) and err.mean() < 1.2e-4, (
            f"start {oc.offset - n} n {n}: {err.max():.2e} {err.mean():.2e}")
    check_codes(*cache.read_codes(), oc, what=f"mode {mode} D {D} W {W}")
