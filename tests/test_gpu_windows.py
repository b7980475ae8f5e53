"""The listed windows of the general records: rows of many shapes against the CPU oracle, and rows of one value
distribution in all blocks, whose cuts lie where every block lists, resolved without rescans (out_info 0): min-p floors deep
in a flat row (the bins above each block's own cut), near its top, top-p boundaries in dense bins of a peaked row."""
import pytest
import torch

import qwen_warp_amd as q
from test_gpu_parity import check_rows

pytestmark = pytest.mark.gpu
V = 31 * 8192


def _logits(kind, B, g):
    u = torch.rand(B, V, generator=g)
    if kind == "uniform":
        return 12.0 * u
    if kind == "laplace":
        u = u - 0.5
        return -torch.sign(u) * torch.log1p(-2 * u.abs().clamp(max=0.4999999))
    if kind == "zipf":
        return -1.2 * torch.log(u.argsort(1).float() + 1.0)
    if kind == "mixture":
        return torch.where(u < 0.01, torch.randn(B, V, generator=g) * 2 + 6, torch.randn(B, V, generator=g))
    return float(kind) * torch.randn(B, V, generator=g)


@pytest.mark.parametrize("kind,params", [
    ("uniform", [dict(min_p=0.1), dict(min_p=0.01), dict(min_p=0.001), dict(min_p=0.9)]),
    ("0.5", [dict(temperature=1.2, min_p=0.05), dict(temperature=0.7, min_p=0.01), dict(temperature=1.3, min_p=0.001), dict(temperature=0.3, min_p=0.05)]),
    ("3.0", [dict(min_p=0.01), dict(min_p=0.1), dict(top_p=0.9), dict(top_p=0.5)])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_cuts_inside_every_window(sampler, kind, params, dtype):
    g = torch.Generator().manual_seed(len(kind))
    rows = [q.RowSpec(**{"temperature": 1.0, **p}, seed=b, position=b, row_key=b) for b, p in enumerate(params * 2)]
    info = check_rows(sampler, _logits(kind, len(rows), g).to(dtype), rows, label=kind)
    # min-p looked up in a bin that a block lists is no rescan; one value distribution in every block: no misses
    assert int((info == 1).sum()) <= 1, info.tolist()


@pytest.mark.parametrize("kind", ["laplace", "zipf", "mixture", "1.0", "1.5"])
def test_windows_of_other_shapes(sampler, kind):
    g = torch.Generator().manual_seed(len(kind))
    params = [dict(top_p=0.9), dict(top_p=0.99), dict(min_p=0.001), dict(min_p=0.01), dict(top_p=0.95, min_p=0.01), dict(top_p=0.99, min_p=0.001),
              dict(top_k=1000, min_p=0.003), dict(top_k=500, top_p=0.9)]
    rows = [q.RowSpec(temperature=[1.3, 0.8][b // len(params)], seed=b, position=b, row_key=b, **p) for b, p in enumerate(params * 2)]
    check_rows(sampler, _logits(kind, len(rows), g), rows, dense=False, label=kind)
