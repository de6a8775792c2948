"""Launches captured into a graph and replayed after later uploads: a batch of the
same rows cut differently, and the first one again.  Every replay works on the batch
uploaded last, as eager calls do."""
import numpy as np
import pytest

from gpu_helpers import to_gpu

pytestmark = pytest.mark.gpu

H, HKV, HD, LAYERS, PAGES = 4, 2, 128, 2, 48


def batch(lens, max_pages, seed):
    rng = np.random.default_rng(seed)
    return rng.permutation(PAGES)[:len(lens) * max_pages].astype(np.int32).reshape(len(lens), max_pages), lens


@pytest.mark.parametrize("wider", [0, 3])
def test_prefill_replays_follow_uploads(wider):
    import torch

    import nitrorag_amd as na

    print(f"prefill replays over uploads, tables {wider} wider", flush=True)
    # 192 rows each: as many 128-row work items, other numbers of 64-row ones
    # (wider tables only for the append alone: attention captures their width)
    first, second = batch([64, 128], 8, 1), batch([96, 96], 8 + wider, 2)
    rng = np.random.default_rng(3)
    q, k, v = (to_gpu(rng.standard_normal((192, n * HD)).astype(np.float32)) for n in (H, HKV, HKV))
    start = [to_gpu(rng.standard_normal((PAGES, LAYERS, 16, HKV * HD)).astype(np.float32)) for _ in range(2)]
    pools = [t.clone() for t in start]
    pool = na.KVPool.wrap(*pools)
    out = torch.full_like(q, float("nan"))

    def upload(b):
        pool.upload_prefill_batch(b[0], [0] * len(b[1]), b[1])

    def step(o):
        pool.kv_append_prefill(1, k, v)
        if not wider:
            pool.prefill(1, q, o, H, HKV, HD)

    def reset():
        for t, s in zip(pools, start):
            t.copy_(s)
        out.fill_(float("nan"))

    upload(second)  # sizes every buffer
    upload(first)
    step(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(out)
    for i, b in enumerate((first, second, first, second, second)):
        upload(b)
        reset()
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in (*pools, out)]
        reset()
        step(out)
        torch.cuda.synchronize()
        for name, g, w in zip(("K pool", "V pool", "output"), got, (*pools, out)):
            assert torch.equal(g.nan_to_num(7.0), w.nan_to_num(7.0)), f"replay {i}: {name}"
    del graph
    assert pool.take_device_errors() == 0
