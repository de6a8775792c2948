"""Prefill attention over infinities and NaN at the head sizes that hold V and
the weights to 24 bits (all but 32, 64 and 128): as fp32 arithmetic has it.  A
score of minus infinity has weight 0, an infinite V an infinite output, a key
past a row's position does not reach it, and rows that meet none of them are the
rows of finite inputs."""
import numpy as np
import pytest

from test_gpu_prefill import prefill_batch_case
from test_gpu_prefill_sizes import run

pytestmark = pytest.mark.gpu


def attended(c, k, v):
    """Causal attention in 64 bits over the appended pools, keys past a row's position left out."""
    H, Hkv, hd, layer = c["H"], c["Hkv"], c["hd"], c["layer"]
    out, row = np.zeros(c["q"].shape), 0
    for b, (start, n) in enumerate(zip(c["starts"], c["lens"])):
        pos = np.arange(int(start + n))
        kk, vv = (p[c["tables"][b][pos // 16], layer, pos % 16].astype(np.float64).reshape(len(pos), Hkv, hd) for p in (k, v))
        for t in range(int(n)):
            seen = int(start) + t + 1
            for h in range(H):
                q = c["q"][row + t, h * hd:(h + 1) * hd].astype(np.float64)
                s = (kk[:seen, h * Hkv // H] * q).sum(axis=1) / np.sqrt(hd)
                p = np.where(s == -np.inf, 0.0, np.exp(s - s.max()))
                out[row + t, h * hd:(h + 1) * hd] = (p[:, None] * vv[:seen, h * Hkv // H]).sum(axis=0) / p.sum()
        row += int(n)
    return out


def put(c, pool, new, b, pos, col, value):
    """Sets column col of sequence b's K or V row at `pos`, cached or new."""
    start, off = int(c["starts"][b]), int(np.sum(c["lens"][:b]))
    if pos < start:
        c[pool][c["tables"][b][pos // 16], c["layer"], pos % 16, col] = value
    else:
        c[new][off + pos - start, col] = value


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("lo,hi,slo,shi", [(20, 45, 0, 0), (30, 150, 3, 40), (260, 280, 0, 0)])
@pytest.mark.parametrize("hd", [16, 48, 80, 96, 112, 160, 256])
def test_infinities_and_nan(hd, lo, hi, slo, shi):
    print(f"prefill non-finite hd {hd} lengths {lo}-{hi} after {slo}-{shi}", flush=True)
    c = prefill_batch_case(hd + lo, 5, lo, hi, 4, 2, hd, 2, 1, slo, shi)
    off = np.concatenate(([0], np.cumsum(c["lens"])))
    ends = [int(s + n) for s, n in zip(c["starts"], c["lens"])]
    # sequence 0: an infinite V early and one of the other sign late, in different heads
    put(c, "v", "vc", 0, 2, 5, np.inf)
    put(c, "v", "vc", 0, ends[0] - 4, hd + hd // 2, -np.inf)
    # sequence 1: an infinite K, so that each query's score there is one of both infinities
    put(c, "k", "kc", 1, 1, 3, np.inf)
    # sequence 2: an infinite query row, and a NaN in a later one
    c["q"][off[2] + 7, 1] = np.inf
    c["q"][off[2] + 11, 3 * hd + 2] = np.nan
    # sequence 3: NaN in V near the end of the chunk
    put(c, "v", "vc", 3, ends[3] - 9, hd - 1, np.nan)
    # sequence 4 stays finite
    got, gk, gv = run(c, False)
    fused, fk, fv = run(c, True)
    for a, b in ((got, fused), (gk, fk), (gv, fv)):
        assert np.array_equal(a, b, equal_nan=True)
    want = attended(c, gk, gv)
    assert np.isfinite(want[off[4]:]).all() and np.isposinf(want).any() and np.isneginf(want).any()
    assert np.isnan(want).any() and np.isfinite(want[off[1]:off[2]]).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0))
    ok = np.isfinite(want)
    # as in test_gpu_prefill_sizes; the rows computed again add their products one
    # by one (hd in a score, a key each in an output)
    adds = hd / 2 + max(ends) / 2 + 6
    bound = 2 * 2.0 ** -24 * np.sqrt(adds / 3)
    err = np.linalg.norm(got[ok] - want[ok]) / np.linalg.norm(want[ok])
    assert err <= bound, (err, bound)
