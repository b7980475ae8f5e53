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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("blocks,crowd", [(17, 3), (31, 3), (32, 3), (33, 6), (64, 7), (64, 9)])
def test_top_list_rows_crowded_blocks(sampler, blocks, crowd, dtype):
    """The best tokens crowded into a few blocks whose lists are held by fewer threads than top_k (16 threads per block up to
    32 blocks, 8 past them; nine blocks of 64: by the 72 a bound of top_k 64 accepts): the resolver's bound falls below all of
    them, more than 128 entries reach it, and they are reduced before they are ranked."""
    V, tpb = blocks * 8192, 16 if blocks <= 32 else 8
    assert (crowd * tpb < 58 or crowd * tpb == 72) and crowd * 58 > 128
    g = torch.Generator().manual_seed(blocks)
    B = 10
    x = torch.randn(B, V, generator=g) * 2.0
    rows = []
    for b in range(B):
        for k in torch.randperm(blocks, generator=g)[:crowd].tolist():
            x[b, k * 8192 + torch.randperm(8192, generator=g)[:300]] += 30.0
        rows.append(q.RowSpec(temperature=[1.0, 8.0][b % 2], top_k=[64, 58, 64, 64, 60][b % 5], top_p=[1.0, 0.9][b // 2 % 2], seed=b, position=b, row_key=b))
    check_rows(sampler, x.to(dtype), rows, label=f"blocks={blocks}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,threads", [(2, 1024), (130, 512)])
@pytest.mark.parametrize("hot", [63, 64, 65])
def test_top_list_rows_whole_threads(sampler, B, threads, hot, dtype):
    """Every element of 63, 64 (the most a block's bound accepts) or 65 threads of a scan workgroup far above all others: the
    bound lists them all, and the list is cut to what a record holds.  Both scan widths (2 x 2 and 130 x 2 workgroups)."""
    vec, V = 4 if dtype == torch.float32 else 8, 16384
    g = torch.Generator().manual_seed(hot)
    x = torch.randn(B, V, generator=g)
    for lo in (0, 8192):
        t = torch.arange(8192) // vec % threads  # the thread that holds each token of a block
        x[:, lo:lo + 8192] += torch.where(torch.isin(t, torch.randperm(threads, generator=g)[:hot]), 25.0, 0.0)
    rows = [q.RowSpec(temperature=[1.0, 4.0][b % 2], top_k=[64, 63, 20][b % 3], top_p=[1.0, 0.95][b // 2 % 2], seed=b, position=b, row_key=b) for b in range(B)]
    check_rows(sampler, x.to(dtype), rows, dense=B == 2, label=f"hot={hot}")


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
