"""The resolver's batched rescans of blocks (raw logits, a bitmap of masked and processed tokens, the patches' values)
against the CPU oracle: more blocks than one batch, a ragged last block, blocks with no, 1,024 (all the patches hold) and
1,025 processed tokens, banned and allowed masks."""
import numpy as np
import pytest
import torch

import qwen_warp_amd as q
from test_gpu_parity import check_rows

pytestmark = pytest.mark.gpu
BLK = 8192


def _mask(V, g, density):
    bits = (torch.rand(V, generator=g) < density).numpy()
    m = np.zeros((V + 31) // 32, np.uint32)
    i = np.nonzero(bits)[0]
    np.bitwise_or.at(m, i >> 5, np.uint32(1) << (i & 31).astype(np.uint32))
    return m


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("blocks", [1, 8, 9, 20])
def test_rescans(sampler, blocks, dtype):
    V = blocks * BLK - (BLK - 40 if blocks == 9 else 0)
    g = torch.Generator().manual_seed(blocks)
    x = torch.randn(6, V, generator=g) * 2.5
    hot = torch.randint(0, V, (6, 24), generator=g)
    x.scatter_add_(1, hot, torch.full(hot.shape, 8.0))
    x = x.to(dtype)
    few = torch.randint(0, V, (700,), generator=g).tolist()
    full = torch.randperm(min(BLK, V), generator=g)[:1024].tolist()          # block 0: 1,024 distinct tokens
    over = full + [int(i) + BLK for i in torch.randperm(min(BLK, V - BLK), generator=g)[:1025]] if V > BLK + 1025 else full  # block 1: 1,025
    pen = dict(repetition=1.2, presence=0.4, frequency=0.2)
    allowed = torch.randperm(V, generator=g)[: V // 2].tolist()
    rows = [dict(top_p=0.95), dict(top_p=0.9, banned=_mask(V, g, 0.05)), dict(top_p=0.95, gen=few, **pen), dict(top_p=0.97, gen=full, banned=_mask(V, g, 0.01), **pen),
            dict(top_p=0.95, gen=over, allowed=allowed, **pen), dict(top_p=0.99, top_k=1000, min_p=0.001, gen=few, **pen)]
    for flags in (q.TF_RESCAN, 0):
        specs = [q.RowSpec(temperature=1.0 - 0.05 * b, seed=b, position=b, row_key=b, test_flags=flags, **r) for b, r in enumerate(rows)]
        info = check_rows(sampler, x, specs, label=f"blocks={blocks} flags={flags}")
        if flags and blocks >= 8:  # the top-p rows' cut bins were rescanned (fewer blocks, or the last row's cuts: a bin of one element)
            assert info.tolist()[:5] == [1] * 5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("slow", [(1,), (0, 7, 11)])
def test_rescans_with_bitmaps_before_staged_blocks(sampler, slow, dtype):
    """One row's cut bin rescanned both from blocks with masked and processed tokens (bitmaps) and from blocks with more
    processed tokens than patches (staged afterwards in the bitmaps' LDS): every block holds 60 tokens of the bin, half of
    them banned or penalised out of it, which must not come back with their raw values."""
    blocks, V, n = 12, 12 * BLK, 60
    params = [dict(top_p=0.5), dict(top_p=0.9), dict(top_k=150), dict(top_k=300, top_p=0.8), dict(min_p=0.998), dict(top_p=0.3, min_p=0.5)]
    g = torch.Generator().manual_seed(len(slow))
    x = torch.randn(2 * len(params), V, generator=g) - 9.0
    rows = []
    for b in range(2 * len(params)):
        hot = torch.stack([k * BLK + torch.randperm(BLK, generator=g)[:n] for k in range(blocks)])  # per block: 15 banned, 15 penalised, 30 kept
        x[b, hot.flatten()] = 5.0 + 0.004 * torch.rand(blocks * n, generator=g)  # a bin is 0.0108 wide at T = 1
        out, gen = hot[:, :15].flatten(), hot[:, 15:30].flatten().tolist()
        for k in slow:
            cold = torch.ones(BLK, dtype=torch.bool)
            cold[hot[k] - k * BLK] = False
            gen += (k * BLK + torch.nonzero(cold).flatten()[:1025]).tolist()
        touched = np.bincount(np.asarray(gen) // BLK, minlength=blocks)
        assert all((touched[k] > 1024) == (k in slow) for k in range(blocks))
        mask = np.zeros((V + 31) // 32, np.uint32)
        np.bitwise_or.at(mask, out.numpy() >> 5, np.uint32(1) << (out.numpy() & 31).astype(np.uint32))
        masks = dict(banned=mask) if b % 2 else dict(allowed=[i for i in range(V) if not (int(mask[i >> 5]) >> (i & 31)) & 1])
        rows.append(q.RowSpec(temperature=1.0, repetition=1.2, presence=0.4, gen=gen, seed=b, position=b, row_key=b, test_flags=q.TF_RESCAN, **masks, **params[b // 2]))
    info = check_rows(sampler, x.to(dtype), rows, label=f"slow={slow}")
    assert info.tolist() == [1] * len(rows)  # every row's cut lies in the rescanned bin


def test_min_p_below_a_top_k_cut(sampler):
    """A min-p cut far below the top-k cut is not looked up: no rescans (out_info 0), the same tokens; at and around the count
    above the min-p cut's bin both cuts still apply."""
    V = 31 * BLK
    g = torch.Generator().manual_seed(3)
    x = torch.randn(8, V, generator=g) * 2.5
    rows = [q.RowSpec(temperature=1.0, top_k=[1000, 1000, 400, 300, 200, 120, 80, 70][b], min_p=[1e-3, 1e-2, 0.03, 0.03, 0.03, 0.03, 0.03, 0.03][b],
                      top_p=[0.9, 1.0][b % 2], seed=b, row_key=b) for b in range(8)]
    info = check_rows(sampler, x, rows)
    assert int(info[0]) == 0
