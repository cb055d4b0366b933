"""fp32 pages with fp32 queries on the fp32 matrix instructions (head_dim 64 and
128, block size 16), against float64: one to four query tiles, row groups past
the tile limit, pieces merged across workgroups, the cost-balanced split, and a
call whose workspace only covers the general path."""

import math

import pytest
import torch

from engine import _hip
from engine.attention import verify_attention
from oracle import attention as ref_attn
from test_gpu_attention import _dense_pool

pytestmark = pytest.mark.gpu


def _check(out, q, keys, values, lens, Hq):
    # fp32 sums of up to n products of O(1) terms: a few 2^-24 in the 2-norm
    want = ref_attn.extend_attention_dense(q.double(), [k.double() for k in keys], [v.double() for v in values],
                                           lens, Hq)
    err = float((out.cpu().double() - want).norm() / want.norm())
    assert err <= 1e-6, err
    assert torch.allclose(out.cpu().double(), want.double(), atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("B,C,Hq,Hkv,d,lo,hi", [
    (1, 1, 2, 2, 64, 0, 0),          # one key
    (4, 5, 4, 2, 64, 37, 129),       # 10 rows
    (2, 9, 14, 2, 64, 300, 1003),    # 63 rows: four tiles
    (3, 11, 14, 2, 64, 1, 77),       # 77 rows: two row groups
    (3, 8, 12, 2, 128, 15, 400),     # 48 rows at head_dim 128: two row groups
    (2, 3, 16, 4, 128, 16, 250),     # 12 rows
    (1, 6, 4, 1, 128, 9000, 9000),   # pieces over several workgroups, merged
    (140, 2, 4, 2, 64, 3, 300),      # more segments than workgroups: the cost-balanced split
    (140, 5, 12, 2, 128, 3, 200),
])
def test_fp32_shapes(cuda, B, C, Hq, Hkv, d, lo, hi):
    g = torch.Generator().manual_seed(B * 100 + C)
    lens = [lo + int(float(u) * (hi - lo + 0.999)) for u in torch.rand(B, generator=g)]
    lens[0] = hi
    gpu, keys, values = _dense_pool(cuda, lens, C, Hkv, d, 16, torch.float32, seed=C, nan_fill=True)
    q = torch.randn(B, C, Hq, d, generator=g) * math.sqrt(2.0)
    out = verify_attention(q.to(cuda), gpu, 0, list(range(B)), lens, max(lens) + C)
    _check(out, q, keys, values, lens, Hq)


@pytest.mark.parametrize("d", [64, 128])
def test_fp32_without_workspace_takes_the_general_path(cuda, d):
    lens, C, Hq, Hkv = [17, 60], 3, 4, 2
    gpu, keys, values = _dense_pool(cuda, lens, C, Hkv, d, 16, torch.float32, seed=1)
    q = torch.randn(2, C, Hq, d, generator=torch.Generator().manual_seed(2))
    qd, out = q.to(cuda), torch.empty(2, C, Hq, d, device=cuda)
    sid, st = _hip.i32([0, 1], cuda), _hip.i32(lens, cuda)
    p = _hip.ptr
    _hip.call("spv_verify_attn", p(out), p(qd), _hip.SPV_F32, p(gpu.k_pool), p(gpu.v_pool), _hip.SPV_F32, None,
              p(gpu.tables_dev), gpu.max_blocks_per_seq, p(sid), p(st), p(gpu.lens_dev), p(gpu.allocator.ctr), 2, C,
              Hq, Hkv, d, 16, 0, gpu.allocator.capacity, max(lens) + C, 1.0 / math.sqrt(d), None, 0,
              _hip.stream_of(cuda))
    _check(out, q, keys, values, lens, Hq)
