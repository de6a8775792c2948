"""Q8 products whose activations reach past 2^32 bytes: every row of x is the
one its output is made of, just below, at and above the limit of a 32-bit byte
offset."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, D = 4096, 48
LIMIT_ROWS = (1 << 30) // N  # x of 2^32 bytes


@pytest.mark.parametrize("rows", [LIMIT_ROWS - 1, LIMIT_ROWS, LIMIT_ROWS + 1, LIMIT_ROWS + 1000])
def test_rows_past_32_bit_byte_offsets(rows):
    import torch

    import nitrorag_amd as na

    print(f"q8 n {N} d {D} rows {rows}", flush=True)
    rng = np.random.default_rng(rows)
    q = rng.integers(-127, 128, (D, N // 32, 32)).astype(np.int8)
    scale = (rng.random((D, N // 32)) * 0.02 + 1e-3).astype(np.float32)
    w = np.concatenate((scale[..., None].view(np.uint8), q.view(np.uint8)), axis=-1).reshape(-1)
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    x = torch.randn(rows, N, generator=g, device="cuda")
    out = torch.full((rows, D), float("nan"), device="cuda")
    na.q8_matmul(torch.from_numpy(w).cuda(), x, out)
    dense = torch.from_numpy((q.astype(np.float64) * scale[..., None]).reshape(D, N)).cuda()
    step = 16384
    for a in range(0, rows, step):
        want = x[a:a + step].double() @ dense.T
        err = ((out[a:a + step].double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
        # a sum of N products, each rounded to 2^-24 (independent roundings add
        # as their root); a row made of another row's x is off by about 1.4
        assert err <= 4 * np.sqrt(N) * 2.0 ** -24, (a, err)
    assert torch.isfinite(out).all()
