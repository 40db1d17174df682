"""The partials of key-split prefill calls: one buffer per GPU, shared by its
handles, ordered among streams and threads. Calls of few rows after some
thousands of positions, which are split; results compared bit for bit with
the same call made alone."""
import gc
import threading

import pytest

from gpu_util import dev_bf16, fast_kv, fast_q

pytestmark = pytest.mark.gpu

SHAPES = [(512, 8, 0), (256, 4, 0), (128, 3, 1), (256, 16, 2)]  # D, bits, mode


class Call:
    """A cache of 3000 positions and one prefill of n rows after them."""

    def __init__(self, gpu, D, bits, mode, n=5, seed=1):
        import torch

        Hkv, Hq, T = 1, 8, 3000
        self.cache = gpu.KVCache(gpu.make_desc(Hkv, D, bits, 0, T + 64 * n, mode))
        k, v = fast_kv(seed, T + n, Hkv, D), fast_kv(seed + 1, T + n, Hkv, D)
        self.cache.append(dev_bf16(k[:T]), dev_bf16(v[:T]))
        self.args = [dev_bf16(k[T:]), dev_bf16(v[T:]), dev_bf16(fast_q(seed, n, Hq, Hkv, D)), 0.02]
        self.out = torch.empty((n, Hq, D), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()

    def run(self):
        self.cache.prefill_step(*self.args, out=self.out)
        return self.out


def test_prefill_scratch_is_shared_and_bounded(gpu):
    import torch

    calls = [Call(gpu, D, bits, mode, n) for D, bits, mode in SHAPES for n in (3, 40)]
    calls[0].run()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for c in calls:
        c.run()
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free, "a later split call took device memory"


def test_first_split_prefill_while_another_stream_captures(gpu):
    """The first split call of a GPU's handles, eager, inside the capture of
    another stream: the capture survives and the result is the usual one."""
    import torch

    alone = Call(gpu, 512, 8, 0)
    want = alone.run().clone()  # (also loads the kernels)
    x = torch.zeros(4, device="cuda")
    del alone
    gc.collect()
    c = Call(gpu, 512, 8, 0)
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        x.add_(1)
        with torch.cuda.stream(side):
            c.run()
        x.add_(1)
    torch.cuda.synchronize()
    assert torch.equal(c.out, want)
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, torch.full_like(x, 2.0 * (i + 1)))


def test_split_prefills_on_streams_and_threads(gpu):
    """Split calls of several handles, in turn on two streams without a wait
    between them, then from one thread per handle, each on a stream of its
    own: every result as alone."""
    import torch

    def fresh():
        return [Call(gpu, D, bits, mode, seed=7 * i + 1) for i, (D, bits, mode) in enumerate(SHAPES)]

    want = []
    for c in fresh():
        outs = []
        for _ in range(12):
            outs.append(c.run().clone())
            torch.cuda.synchronize()
        want.append(outs)
    torch.cuda.synchronize()

    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    calls, got = fresh(), [[] for _ in SHAPES]
    for r in range(12):
        for i, c in enumerate(calls):
            with torch.cuda.stream(streams[i % 2]):
                got[i].append(c.run().clone())
    torch.cuda.synchronize()
    for i in range(len(SHAPES)):
        assert all(torch.equal(a, b) for a, b in zip(got[i], want[i])), f"streams: {SHAPES[i]}"

    calls, got, errors = fresh(), [[] for _ in SHAPES], []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(12):
                    got[i].append(calls[i].run().clone())
            s.synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(SHAPES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(len(SHAPES)):
        assert all(torch.equal(a, b) for a, b in zip(got[i], want[i])), f"threads: {SHAPES[i]}"
