"""Verify rows whose kept set is listed (at most 64 tokens: the residual drawn from the list, without the blocks) beside
rows whose set is not, against verify_seq: set sizes around 64, 12 sequences of four blocks (1,024-thread verify kernels) and
300 of one block (512-thread ones), draft probabilities that leave no residual, NaN and zero ones, the broken-residual
control."""
import pytest
import torch

import qwen_warp_amd as q
from test_gpu_verify import _case, check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("top_k,B,K,V,Vd", [*((k, 12, 5, 3 * 8192 + 64, 4096) for k in (1, 2, 63, 64, 65)), (63, 300, 2, 1024, 600)])
def test_listed_kept_sets(top_k, B, K, V, Vd, dtype):
    tl, dp, idmap, drafts, g = _case(top_k, B, K, V, Vd, dtype, agree=0.8, noise=0.7)
    dp[1] = 0.0
    dp[2] = float("nan")
    dp[3] = 1.0  # q >= p on every token of the draft table
    dp[4].clamp_(min=1e-3)
    sm = q.Sampler("cuda")
    seqs = [q.RowSpec(temperature=[1.0, 0.6][b % 2], top_k=0 if b % 5 == 4 else top_k, top_p=[1.0, 0.9][b // 2 % 2], min_p=0.02 * (b % 3 == 1), seed=b, position=b,
                      row_key=b, test_flags=q.TF_BROKEN if b == 7 else 0) for b in range(B)]
    check_against_oracle(sm, tl, dp, idmap, drafts, seqs, f"top_k={top_k}")
