"""Q8 products over many activation rows (the large-tile kernel): ragged rows,
outputs and blocks around its tiles against 64 bits, and a layer whose four
launches (RoPE + append, residual, SwiGLU) all take it against the oracle; each of
its forms at both tile widths, which nitro_q8_tile_rows confirms."""
import numpy as np
import pytest

from nitrorag_amd.q8 import MATMUL, QKV, RESIDUAL, SWIGLU, tile_rows
from test_gpu_model import check_logits
from test_gpu_q8 import run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,batch,tile", [
    (96, 8500, 130, 128),    # 3 blocks (no flush), rows of x past two panels, a partial column tile
    (256, 1100, 1000, 128),  # one flush exactly
    (2080, 4300, 257, 128),  # 65 blocks: flushes, a pair and an odd block; one row in the last panel
    (288, 16390, 513, 128),  # 9 blocks
    (32, 16384, 127, 128),   # one block
    (288, 29000, 515, 64),   # the narrow tile, 9 blocks
])
def test_many_rows(n, d, batch, tile):
    print(f"q8 gemm n {n} d {d} batch {batch}", flush=True)
    assert tile_rows(batch, n, d, MATMUL) == tile
    rng = np.random.default_rng(n + d + batch)
    q = rng.integers(-127, 128, (d, n // 32, 32)).astype(np.int8)
    scale = (rng.random((d, n // 32)) * 0.02 + 1e-3).astype(np.float32)
    w = np.concatenate((scale[..., None].view(np.uint8), q.view(np.uint8)), axis=-1).reshape(-1)
    x = rng.standard_normal((batch, n)).astype(np.float32)
    got = run_gpu(w, x, d, 0)
    want = x.astype(np.float64) @ (q.astype(np.float64) * scale[..., None]).reshape(d, n).T
    # An add's rounding is at most 2^-24 of its result (2^-24 / sqrt(3) in the mean
    # square), and partial sums of random terms grow as their root.  Adds of block
    # sums, in chains of 8: 4.5 in units of the output's square; of chains: blocks /
    # 16; within a block, about 6.  Roundings add as their root, twice which is the
    # bound.  (x without its lowest part would be off by 5e-6.)
    bound = 2 * 2.0 ** -24 * np.sqrt((10.5 + n / 32 / 16) / 3)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"error {err:.3g} of {bound:.3g}", flush=True)
    assert err <= bound, (err, bound)


def layer_tiles(rows, dim, hid, kv):
    """Tile widths of a layer's wo, w2, w1 + w3, wq + wk + wv."""
    return [tile_rows(rows, dim, dim, RESIDUAL), tile_rows(rows, hid, dim, RESIDUAL), tile_rows(rows, dim, hid, SWIGLU),
            tile_rows(rows, dim, dim, QKV, kv)]


def test_layer_of_wide_tiles():
    """A layer of 8271 rows of nine prompts, all four launches with 128 weight rows
    per workgroup, against the same layer in 64 bits."""
    import torch

    from perf import cases

    case = {"kind": "model_prefill", "dim": 768, "hidden": 1376, "layers": 1, "heads": 8, "kv_heads": 8, "vocab": 500,
            "seq_len": 1024, "batch": 9, "new_min": 826, "new_max": 1000, "lengths": 0, "semantics": 0}
    rows = 8271
    print(f"layer of {rows} rows", flush=True)
    assert layer_tiles(rows, 768, 1376, 768) == [128, 128, 128, 128]
    state = cases.prepare(case, 11)
    assert int(state["count"].sum()) == rows
    got = cases.run(state)
    want = cases.exact(case, 11)
    torch.cuda.synchronize()
    for name, g, w in zip(("logits", "K pool", "V pool"), got, want):
        err = ((g.double() - w.double()).norm() / w.double().norm()).item()
        print(f"{name}: error {err:.3g}", flush=True)
        # three products in a row, attention (head size 96: at 24 bits), the norms and
        # the classifier: six steps, each within 2.7e-7 as test_many_rows has it, whose
        # errors add as their root
        assert err <= np.sqrt(6) * 2.7e-7, (name, err)


def test_layer_of_many_rows():
    import torch

    import nitrorag_amd as na
    from nitrorag_amd.model import FULL_ROWS, synthetic_model_file
    from oracle import model as om

    # 43 blocks of hidden columns, grouped heads, 2000 rows of three prompts
    dim, hid, H, Hkv, V, S = 512, 1376, 8, 2, 300, 1024
    lens = [1000, 777, 223]
    print(f"layer of {sum(lens)} rows", flush=True)
    assert layer_tiles(sum(lens), dim, hid, dim * Hkv // H) == [64, 64, 64, 64]
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
