"""Uploads read from host memory by a kernel, in a process whose runtime is told to
give out non-coherent host memory by default (HIP_HOST_COHERENT=0): the device
arrays hold every upload's own values, though all are staged at the same
addresses."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import numpy as np, torch
import nitrorag_amd as na

B, MAX_PAGES, KV = 24, 9, 64
PAGES = B * MAX_PAGES
k = torch.zeros(PAGES, 1, 16, KV, device="cuda")
v = torch.zeros_like(k)
pool = na.KVPool.wrap(k, v)
rng = np.random.default_rng(1)
for step in range(60):
    tables = rng.permutation(PAGES).astype(np.int32).reshape(B, MAX_PAGES)
    pos = rng.integers(0, 16 * MAX_PAGES, B).astype(np.int32)
    pool.upload_decode_batch(tables, pos)
    row = torch.full((B, KV), float(step + 1), device="cuda")
    pool.kv_append(0, row, -row)
    want = np.zeros((PAGES, 16), bool)
    want[tables[np.arange(B), pos // 16], pos % 16] = True
    got = (k[:, 0, :, 0] == step + 1).cpu().numpy()
    assert np.array_equal(got, want), f"step {step}: rows elsewhere than the last upload has them"
assert pool.take_device_errors() == 0
print("uploads ok", flush=True)
"""


def test_uploads_without_coherent_default():
    print("uploads under HIP_HOST_COHERENT=0", flush=True)
    env = dict(os.environ, HIP_HOST_COHERENT="0", PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100, env=env, cwd=ROOT)
    assert r.returncode == 0 and "uploads ok" in r.stdout, r.stdout + r.stderr
