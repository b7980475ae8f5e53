"""Rows whose top_k is at most 64 (top-list records: each block's best candidates from a bound on the threads' largest
elements) against the CPU oracle, where the selection can go wrong: ties at the bound, the best tokens crowded into few
threads, fewer candidates than top_k, the smallest and the widest vocabularies, both k_scan widths."""
import pytest
import torch

import qwen_warp_amd as q
from test_gpu_parity import check_rows

pytestmark = pytest.mark.gpu


def _logits(kind, B, V, g):
    x = torch.randn(B, V, generator=g) * 3.0
    if kind == "equal":        # one value everywhere: the bound is tied in every thread
        x[:] = 1.25
    elif kind == "tied":       # ten values: ties at the bound across threads and blocks
        x = x.clamp(-3, 3).round()
    elif kind == "crowded":    # the best tokens are neighbours: they lie in few threads of one block
        x[:, : min(V, 200)] += 20.0
    elif kind == "sorted":
        x = x.sort(dim=1, descending=True).values
    elif kind == "sparse":     # few candidates, some of them infinite or NaN
        keep = torch.randperm(V, generator=g)[: 40]
        y = torch.full_like(x, float("-inf"))
        y[:, keep] = x[:, keep]
        y[:, keep[0]] = float("nan")
        x = y
    elif kind == "none":
        x[:] = float("-inf")
    elif kind == "signed":     # zeros of both signs at the bound
        x = torch.where(torch.rand(B, V, generator=g) < 0.5, torch.tensor(0.0), torch.tensor(-0.0))
        x[:, :: max(V // 20, 1)] = 1.0
    return x


@pytest.mark.parametrize("kind", ["normal", "equal", "tied", "crowded", "sorted", "sparse", "none", "signed"])
@pytest.mark.parametrize("V", [8, 8200, 66000, 524288])
def test_top_list_rows(sampler, kind, V):
    g = torch.Generator().manual_seed(V + len(kind))
    B = 12 if V == 8200 else 5 if V < 500000 else 3
    x = _logits(kind, B, V, g)
    for dt in (torch.float32, torch.bfloat16):
        rows = [q.RowSpec(temperature=[1.0, 0.7, 1.3][b % 3], top_k=[64, 1, 20, 63, 50][b % 5], top_p=[1.0, 0.9, 1e-7, 0.95][b % 4], min_p=0.05 * (b % 2),
                          seed=9 + b, position=b, row_key=b) for b in range(B)]
        check_rows(sampler, x.to(dt), rows, label=f"{kind} V={V} {dt}")


@pytest.mark.parametrize("B", [7, 40])
def test_top_list_rows_with_processors(sampler, B):
    """Both k_scan widths (7 x 31 and 40 x 31 workgroups) with penalties, biases past the bound and masked tokens; rows
    beside rows that take the general records."""
    V = 248320
    g = torch.Generator().manual_seed(B)
    x = torch.randn(B, V, generator=g) * 3.0
    rows = []
    for b in range(B):
        hist = torch.randint(0, V, (500,), generator=g).tolist()
        bias = {int(i): 30.0 for i in torch.randperm(V, generator=g)[:70]} if b % 3 == 0 else None
        allowed = torch.randperm(V, generator=g)[:45].tolist() if b % 5 == 4 else None
        rows.append(q.RowSpec(temperature=0.8, top_k=[20, 64, 0, 50, 65][b % 5], top_p=0.95, repetition=1.2, presence=0.3, gen=hist, bias=bias, allowed=allowed,
                              seed=b, row_key=b))
    check_rows(sampler, x, rows, dense=False)
