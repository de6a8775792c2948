"""Q8 products over many activation rows (the large-tile kernel): ragged rows,
outputs and blocks around its tiles against 64 bits, and a layer whose four
launches (RoPE + append, residual, SwiGLU) all take it against the oracle."""
import numpy as np
import pytest

from test_gpu_model import check_logits
from test_gpu_q8 import run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,batch", [
    (96, 8200, 130),     # 3 blocks (no flush), rows of x past two panels, a partial column tile
    (256, 1000, 1000),   # one flush exactly
    (2080, 4104, 257),   # 65 blocks: flushes, a pair and an odd block; one row in the last panel
    (288, 16390, 513),   # the 128-row tile, 9 blocks
    (32, 16384, 127),    # one block
])
def test_many_rows(n, d, batch):
    print(f"q8 gemm n {n} d {d} batch {batch}", flush=True)
    rng = np.random.default_rng(n + d + batch)
    q = rng.integers(-127, 128, (d, n // 32, 32)).astype(np.int8)
    scale = (rng.random((d, n // 32)) * 0.02 + 1e-3).astype(np.float32)
    w = np.concatenate((scale[..., None].view(np.uint8), q.view(np.uint8)), axis=-1).reshape(-1)
    x = rng.standard_normal((batch, n)).astype(np.float32)
    got = run_gpu(w, x, d, 0)
    want = x.astype(np.float64) @ (q.astype(np.float64) * scale[..., None]).reshape(d, n).T
    # n products rounded to 2^-24 of a sum whose size they share: independent
    # roundings add as their root, twice which bounds the 2-norm
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2 * np.sqrt(n) * 2.0 ** -24, err


def test_layer_of_many_rows():
    import torch

    import nitrorag_amd as na
    from nitrorag_amd.model import FULL_ROWS, synthetic_model_file
    from oracle import model as om

    # 43 blocks of hidden columns, grouped heads, 2000 rows of three prompts
    dim, hid, H, Hkv, V, S = 512, 1376, 8, 2, 300, 1024
    lens = [1000, 777, 223]
    print(f"layer of {sum(lens)} rows", flush=True)
    blob = om.scale_residual_outputs(synthetic_model_file(dim, hid, 1, H, Hkv, V, S, seed=5), 64.0)
    model, ora = na.Model(blob), om.OracleModel(blob)
    need = [-(-n // 16) for n in lens]
    pages = sum(need) + 3
    order = np.random.default_rng(6).permutation(pages).astype(np.int32)
    tables = np.zeros((3, max(need)), np.int32)
    for b, n in enumerate(need):
        tables[b, :n] = order[sum(need[:b]):sum(need[:b]) + n]
    dk = torch.zeros((pages, 1, 16, model.kv_dim), device="cuda")
    dv = torch.zeros_like(dk)
    pool = na.KVPool.wrap(dk, dv)
    toks = np.random.default_rng(7).integers(0, V, sum(lens)).astype(np.int32)
    pool.upload_prefill_batch(tables, [0, 0, 0], lens)
    got = model.forward_prefill(pool, toks, semantics=FULL_ROWS).cpu().numpy()
    assert pool.take_device_errors() == 0
    k = np.zeros((pages, 1, 16, model.kv_dim), np.float32)
    v = np.zeros_like(k)
    ends = np.cumsum(lens)
    want = np.stack([ora.forward_prefill_chunk(k, v, tables[b], 0, toks[ends[b] - n:ends[b]], bulk=False)
                     for b, n in enumerate(lens)])
    check_logits(got, want, "layer of many rows")
    for g, r in ((dk, k), (dv, v)):
        assert np.abs(g.cpu().numpy() - r).max() <= 1e-4 + 1e-3 * np.abs(r).max()


@pytest.mark.parametrize("n,d,batch", [(2080, 8200, 400), (4096, 4200, 1000)])
def test_equal_rows_give_equal_bits(n, d, batch):
    """Activation rows that are the same, in any panel, and weight rows that are the
    same, in any column tile, give the same bits: an output's sums are added in an
    order that depends on n alone."""
    print(f"q8 equal rows n {n} d {d} batch {batch}", flush=True)
    rng = np.random.default_rng(n)
    q = rng.integers(-127, 128, (5, n // 32, 32)).astype(np.int8)
    scale = (rng.random((5, n // 32)) * 0.02 + 1e-3).astype(np.float32)
    few = np.concatenate((scale[..., None].view(np.uint8), q.view(np.uint8)), axis=-1).reshape(5, -1)
    x = rng.standard_normal((7, n)).astype(np.float32)
    got = run_gpu(few[np.arange(d) % 5].reshape(-1), x[np.arange(batch) % 7], d, 0)
    assert np.array_equal(got, got[:7, :5][np.arange(batch) % 7][:, np.arange(d) % 5])
