"""Device memory that a model's forwards take: the SwiGLU output held once where
every product reads one form of it, nothing in split form for a model that never runs
full-row products of more than 4 rows, and no buffer moved by a forward of other
semantics."""
import numpy as np
import pytest

from nitrorag_amd.model import FULL_ROWS, LAST_BLOCK, synthetic_model_file

pytestmark = pytest.mark.gpu

DIM, HIDDEN, HEADS, VOCAB, SEQ = 256, 8192, 4, 64, 1024
PROMPTS, TOKENS = 8, 1000
ROWS = PROMPTS * TOKENS
HB = 4 * ROWS * HIDDEN                              # SwiGLU's output as floats
ROW_BUFFERS = 4 * ROWS * (3 * DIM + DIM // 16 + 1)  # x, attention, q, partial sums, tokens
SPLIT = 6 * ROWS * (DIM + HIDDEN)                   # x and SwiGLU's output in split form
WEIGHTS = 2 * (3 * HIDDEN + 4 * DIM) * DIM          # the tile layout, below 2 bytes a weight
SLACK = 48 << 20                                    # allocation granules, kernels loaded on first use


@pytest.mark.parametrize("order,most", [
    ([LAST_BLOCK, LAST_BLOCK], [ROW_BUFFERS + HB] * 2),
    ([FULL_ROWS, LAST_BLOCK, FULL_ROWS], [ROW_BUFFERS + SPLIT + WEIGHTS] * 3),
    ([LAST_BLOCK, FULL_ROWS, LAST_BLOCK], [ROW_BUFFERS + HB] + [ROW_BUFFERS + HB + SPLIT + WEIGHTS] * 2),
])
def test_forward_buffers(order, most):
    import torch

    import nitrorag_amd as na

    print(f"model buffers, semantics {order}", flush=True)
    model = na.Model(synthetic_model_file(DIM, HIDDEN, 1, HEADS, HEADS, VOCAB, SEQ, seed=3))
    need = -(-TOKENS // 16)
    pages = torch.zeros((PROMPTS * need, 1, 16, model.kv_dim), device="cuda")
    pool = na.KVPool.wrap(pages, torch.zeros_like(pages))
    tables = np.arange(PROMPTS * need, dtype=np.int32).reshape(PROMPTS, need)
    tokens = np.random.default_rng(4).integers(0, VOCAB, ROWS).astype(np.int32)
    logits = torch.empty((PROMPTS, VOCAB), device="cuda")
    pool.upload_prefill_batch(tables, [0] * PROMPTS, [TOKENS] * PROMPTS)
    torch.cuda.synchronize()
    free, outs = torch.cuda.mem_get_info()[0], {}
    for semantics, bound in zip(order, most):
        model.forward_prefill(pool, tokens, logits, semantics)
        torch.cuda.synchronize()
        assert torch.isfinite(logits).all()
        assert torch.equal(logits, outs.setdefault(semantics, logits.clone()))
        torch.cuda.synchronize()
        taken = free - torch.cuda.mem_get_info()[0]
        print(f"semantics {semantics}: {taken} of {bound}", flush=True)
        assert taken <= bound + SLACK
    assert pool.take_device_errors() == 0
