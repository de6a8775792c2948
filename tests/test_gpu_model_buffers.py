"""Device memory that a model's forwards take: one copy of the SwiGLU output, in the
form the products read, and nothing in split form for a model that never runs
full-row products of more than 4 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIM, HIDDEN, HEADS, VOCAB, SEQ = 256, 8192, 4, 64, 1024
PROMPTS, TOKENS = 8, 1000
ROWS = PROMPTS * TOKENS


def test_forward_buffers():
    import torch

    import nitrorag_amd as na
    from nitrorag_amd.model import FULL_ROWS, LAST_BLOCK, synthetic_model_file

    print("model buffers", flush=True)
    model = na.Model(synthetic_model_file(DIM, HIDDEN, 1, HEADS, HEADS, VOCAB, SEQ, seed=3))
    need = -(-TOKENS // 16)
    pages = torch.zeros((PROMPTS * need, 1, 16, model.kv_dim), device="cuda")
    pool = na.KVPool.wrap(pages, torch.zeros_like(pages))
    tables = np.arange(PROMPTS * need, dtype=np.int32).reshape(PROMPTS, need)
    tokens = np.random.default_rng(4).integers(0, VOCAB, ROWS).astype(np.int32)
    logits = torch.empty((PROMPTS, VOCAB), device="cuda")
    pool.upload_prefill_batch(tables, [0] * PROMPTS, [TOKENS] * PROMPTS)
    torch.cuda.synchronize()
    free = [torch.cuda.mem_get_info()[0]]
    outs = []
    for semantics in (LAST_BLOCK, FULL_ROWS, LAST_BLOCK):
        model.forward_prefill(pool, tokens, logits, semantics)
        torch.cuda.synchronize()
        outs.append(logits.clone())
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    assert torch.equal(outs[0], outs[2]) and torch.isfinite(outs[1]).all()
    assert pool.take_device_errors() == 0
    taken = [free[0] - f for f in free[1:]]
    floats = 4 * ROWS * (3 * DIM + DIM // 16 + HIDDEN)     # x, attention, q, partial sums, hb
    split = 6 * ROWS * DIM + 2 * ROWS * HIDDEN             # x in split form; hb grows from 4 to 6 bytes a value
    weights = 2 * (2 * HIDDEN + HIDDEN + 4 * DIM) * DIM    # the tile layout, below 2 bytes a weight
    slack = 48 << 20                                       # allocation granules, kernels loaded on first use
    print(f"taken {taken}, floats {floats}, split {split}", flush=True)
    assert taken[0] <= floats + slack
    assert taken[1] <= floats + split + weights + slack
    assert taken[2] <= taken[1] + slack
