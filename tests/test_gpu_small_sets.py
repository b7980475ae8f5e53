"""Rows of the general records whose candidates number about 64 (the one-pass finish over the blocks' lists takes up to 64)
against the CPU oracle: below, at and past that count, spread over the blocks or in one, with a top-p threshold, a min-p
cut, a top-k past the set, and no cut at all; the rest of the vocabulary below the weight window, just inside it, or masked."""
import pytest
import torch

import qwen_warp_amd as q
from test_gpu_parity import check_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 200])
@pytest.mark.parametrize("where", ["spread", "one block", "block ends"])
def test_small_sets(sampler, n, where, dtype):
    V = 12 * 8192 + 520
    g = torch.Generator().manual_seed(n)
    params = [dict(top_p=0.9), dict(min_p=0.2), dict(min_p=0.02, top_p=0.8), dict(top_k=1000, top_p=0.95), dict(top_k=1000, min_p=0.1), dict(), dict(top_p=0.9999999),
              dict(top_p=1e-6)]
    rows, x = [], torch.empty(2 * len(params), V)
    for b in range(2 * len(params)):
        base = [-60.0, -18.0][b % 2]  # below the weight window of 35 powers of two; inside it
        x[b] = base + torch.randn(V, generator=g) * 0.3
        if b % 4 == 3:
            x[b] = float("-inf")
        ids = torch.randperm(V, generator=g)[:n] if where == "spread" else 8192 + torch.randperm(8192, generator=g)[:n] if where == "one block" else \
            torch.tensor([(i // 2) % 13 * 8192 + (0 if i % 2 == 0 else 519) - (i // 26 if i % 2 else -(i // 26)) for i in range(n)])
        x[b, ids] = torch.rand(n, generator=g) * 4.0
        rows.append(q.RowSpec(temperature=[1.0, 0.6][b // 2 % 2], seed=b, position=b, row_key=b, **params[b // 2]))
    check_rows(sampler, x.to(dtype), rows, label=f"n={n} {where}")
