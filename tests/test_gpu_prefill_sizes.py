"""Prefill attention at head sizes around the widths its kernels are built for
(32, 64, 96, 128, 256 columns): fresh prompts, chunks after cached keys, ragged
lengths around the query and key tiles, grouped-query heads, against 64-bit
attention.  The scatter + attention pair and the append call agree exactly."""
import numpy as np
import pytest

from gpu_helpers import to_gpu
from test_gpu_prefill import prefill_batch_case

pytestmark = pytest.mark.gpu


def exact(c, k, v):
    """Causal attention in 64 bits over the appended pools."""
    H, Hkv, hd, layer = c["H"], c["Hkv"], c["hd"], c["layer"]
    out, row = np.zeros(c["q"].shape), 0
    for b, (start, n) in enumerate(zip(c["starts"], c["lens"])):
        pos = np.arange(int(start + n))
        kk, vv = (p[c["tables"][b][pos // 16], layer, pos % 16].astype(np.float64).reshape(len(pos), Hkv, hd) for p in (k, v))
        q = c["q"][row:row + n].astype(np.float64).reshape(int(n), H, hd)
        seen = pos[None, :] <= int(start) + np.arange(int(n))[:, None]
        for h in range(H):
            s = np.where(seen, q[:, h] @ kk[:, h * Hkv // H].T / np.sqrt(hd), -np.inf)
            p = np.exp(s - s.max(axis=1, keepdims=True))
            out[row:row + n, h * hd:(h + 1) * hd] = (p / p.sum(axis=1, keepdims=True)) @ vv[:, h * Hkv // H]
        row += int(n)
    return out


def run(c, append):
    import torch

    import nitrorag_amd as na

    k, v = to_gpu(c["k"]), to_gpu(c["v"])
    pool = na.KVPool.wrap(k, v)
    pool.upload_prefill_batch(c["tables"], c["starts"], c["lens"])
    q, kc, vc = to_gpu(c["q"]), to_gpu(c["kc"]), to_gpu(c["vc"])
    out = torch.full_like(q, float("nan"))
    if append:
        pool.prefill_append(c["layer"], q, kc, vc, out, c["H"], c["Hkv"], c["hd"])
    else:
        pool.kv_append_prefill(c["layer"], kc, vc)
        pool.prefill(c["layer"], q, out, c["H"], c["Hkv"], c["hd"])
    torch.cuda.synchronize()
    assert pool.take_device_errors() == 0
    return out.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy()


# (lengths lo, hi, starts lo, hi): single tokens, around a key tile (32, 64) and
# a query item (64, 128), chunks after cached keys that start inside a page, and
# batches past 256 keys (two K/V buffers at heads of 65..128)
SHAPES = [(1, 1, 0, 0), (31, 33, 0, 0), (127, 130, 0, 0), (1, 140, 1, 200), (260, 300, 0, 0), (1, 40, 240, 270)]


@pytest.mark.parametrize("hd", [4, 28, 36, 60, 68, 80, 92, 96, 100, 124, 128, 132, 252, 256])
def test_head_sizes(hd):
    for i, (lo, hi, slo, shi) in enumerate(SHAPES):
        print(f"prefill hd {hd} lengths {lo}-{hi} after {slo}-{shi}", flush=True)
        c = prefill_batch_case(100 + i, 3, lo, hi, 4, 2, hd, 2, 1, slo, shi)
        got, gk, gv = run(c, False)
        fused, fk, fv = run(c, True)
        assert np.array_equal(got, fused) and np.array_equal(gk, fk) and np.array_equal(gv, fv)
        want = exact(c, gk, gv)
        # An add rounds to 2^-24 / sqrt(3) of its result in the mean square, and sums of
        # random terms grow as their root, so a chain of n adds is off by sqrt(n / 2)
        # of that: six products per 32 columns for a score (of size 1, entering its
        # weight directly), six per 32 keys (at most 340) for an output, and about 6
        # in units of its square for exp2, the weights' sum and the division.  They
        # add as their root, twice which is the bound.  (hd 128 holds V and the
        # weights to 16 bits: 2^-16 of each, 2^-15 in all; a lost part anywhere else
        # shows as 1e-5 too.)
        adds = 6 * -(-hd // 32) / 2 + 6 * 340 / 32 / 2 + 6
        bound = 2 * 2.0 ** -24 * np.sqrt(adds / 3) + (2.0 ** -15 if hd == 128 else 0)
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"error {err:.3g} of {bound:.3g}", flush=True)
        assert err <= bound, (hd, lo, hi, err, bound)
