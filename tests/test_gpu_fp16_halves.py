"""fp16 pages with P in two fp16 halves, and in one where the kernels with four
query tiles at head_dim 128 keep it (batches that fill the grid), against
float64. Rounding the output to fp16 alone has a relative 2-norm of 2.0e-4 to
2.1e-4 (2^-11 times 0.41); the halves add 2^-22, one half of P up to about 1.8e-4
in quadrature."""

import pytest
import torch

from engine.attention import VerifyPlan, verify_attention
from oracle import attention as ref_attn

from test_gpu_attention import _dense_pool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,Hq,Hkv,d,hi,bound", [
    (3, 7, 16, 2, 128, 500, 2.4e-4),     # four tiles at 128, the smallest piece sets the split
    (6, 9, 16, 2, 128, 20, 2.4e-4),      # one piece per segment, two row groups
    (24, 7, 16, 2, 128, 3000, 3.0e-4),   # longer pieces fill the grid: one half
    (130, 8, 16, 2, 128, 90, 3.0e-4),    # the cost-balanced split
    (4, 6, 12, 2, 128, 700, 2.4e-4),
    (4, 1, 14, 2, 64, 3000, 2.4e-4),
    (130, 9, 14, 2, 64, 200, 2.4e-4),
])
def test_error_against_float64(cuda, B, C, Hq, Hkv, d, hi, bound):
    g = torch.Generator().manual_seed(B + hi)
    lens = [hi] + [int(x) for x in torch.randint(0, hi + 1, (B - 1,), generator=g)]
    gpu, keys, values = _dense_pool(cuda, lens, C, Hkv, d, 16, torch.float16, seed=hi)
    q = torch.randn(B, C, Hq, d, generator=g).to(torch.float16)
    out = verify_attention(q.to(cuda), gpu, 0, list(range(B)), lens, max(lens) + C)
    plan = VerifyPlan(gpu, list(range(B)), lens, C, Hq, max(lens) + C)
    assert torch.equal(verify_attention(q.to(cuda), gpu, 0, list(range(B)), lens, max(lens) + C, plan=plan), out)
    want = ref_attn.extend_attention_dense(q.float(), [k.float() for k in keys], [v.float() for v in values], lens, Hq)
    err = float((out.cpu().double() - want.double()).norm() / want.double().norm())
    assert err <= bound, err


@pytest.mark.parametrize("B,C,lo,hi", [
    (16, 7, 256, 4096),   # even share 4 pages, smallest piece 24
    (16, 7, 64, 4096),
    (20, 8, 700, 3000),   # even share 9, smallest piece 20
    (9, 7, 16, 12000),    # smallest piece 41
])
def test_ragged_batches_with_four_tiles_at_128(cuda, B, C, lo, hi):
    """One long context among short ones: the batch's own pages leave the grid
    unfilled, though B times the longest context would fill it. The pieces are the
    smallest ones, so P is in two halves; a looser max_ctx changes nothing."""
    lens = [lo] * (B // 2) + [hi] + [lo] * (B - 1 - B // 2)
    gpu, keys, values = _dense_pool(cuda, lens, C, 2, 128, 16, torch.float16, seed=hi)
    q = torch.randn(B, C, 16, 128, generator=torch.Generator().manual_seed(B + lo)).to(torch.float16)
    out = verify_attention(q.to(cuda), gpu, 0, list(range(B)), lens, hi + C)
    want = ref_attn.extend_attention_dense(q.float(), [k.float() for k in keys], [v.float() for v in values], lens, 16)
    err = float((out.cpu().double() - want.double()).norm() / want.double().norm())
    assert err <= 2.2e-4, err  # the output's rounding, 2.0e-4 to 2.1e-4; one half of P would add 1.2e-4 or more in quadrature
    for more in (1.5, 4):
        assert torch.equal(verify_attention(q.to(cuda), gpu, 0, list(range(B)), lens, int(hi * more)), out), more


def test_loose_max_ctx_leaves_a_full_grid_alone(cuda):
    """One half of P (the batch fills the grid): the same bits whatever max_ctx."""
    lens, C = [300 + 97 * b for b in range(28)], 7
    gpu, _, _ = _dense_pool(cuda, lens, C, 2, 128, 16, torch.float16, seed=3)
    q = torch.randn(28, C, 16, 128, generator=torch.Generator().manual_seed(4)).to(torch.float16).to(cuda)
    out = verify_attention(q, gpu, 0, list(range(28)), lens, max(lens) + C)
    assert torch.equal(verify_attention(q, gpu, 0, list(range(28)), lens, 20000), out)
