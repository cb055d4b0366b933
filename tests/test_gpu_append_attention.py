"""A later layer's append and attention in one launch (``append_verify_attention``)
against the two calls it stands for (a planned write, then planned attention):
pools and outputs bit-equal. Chunks inside one page, across pages, across the
pieces of a segment, longer than the eight tokens a wave loads at once; row
groups that each write the page they read; the cost-balanced split; an
exhausted pool; shapes and types the planned kernels do not take; an output
that shares memory with the new keys."""

import pytest
import torch

from engine import _hip
from engine.attention import VerifyPlan, append_verify_attention, verify_attention
from engine.kv import BlockExhaustedError, PagedKVCache, WritePlan

pytestmark = pytest.mark.gpu


def _pools(cuda, lens, C, Hkv, d, dtype, layers, seed, cap=None):
    g = torch.Generator().manual_seed(seed)
    need = sum(-(-(n + C) // 16) for n in lens)
    perm = torch.randperm(cap or need + 8, generator=g).tolist()
    kvs = [PagedKVCache(layers, Hkv, d, len(perm), 16, cuda, dtype, max_seqs=len(lens)) for _ in range(2)]
    for kv in kvs:
        kv.k_pool.fill_(float("nan"))
        kv.v_pool.fill_(float("nan"))
        kv.allocator.load_free_list(perm)
        for s in range(len(lens)):
            kv.add_sequence(s)
    for layer in range(layers):
        for s, n in enumerate(lens):
            if n:
                k, v = (torch.randn(1, n, Hkv, d, generator=g).to(dtype).to(cuda) for _ in range(2))
                for kv in kvs:
                    kv.write_block(layer, [s], [0], k, v)
    return kvs, g


def _same(a, b):
    return torch.equal(a.view(torch.int16 if a.element_size() == 2 else torch.int32),
                       b.view(torch.int16 if b.element_size() == 2 else torch.int32))


def _compare(cuda, kvs, g, lens, C, Hq, Hkv, d, qdtype, dtype, layers=3):
    B = len(lens)
    sid, st = _hip.i32(list(range(B)), cuda), _hip.i32(lens, cuda)
    mc = max(lens) + C
    qkv = [tuple(torch.randn(B, C, h, d, generator=g).to(t).to(cuda) for h, t in ((Hq, qdtype), (Hkv, dtype), (Hkv, dtype)))
           for _ in range(layers)]
    outs = []
    for kv, fused in zip(kvs, (False, True)):
        wplan, plan, o = WritePlan(), None, []
        for layer, (q, k, v) in enumerate(qkv):
            if layer and fused:
                o.append(append_verify_attention(q, k, v, kv, layer, sid, st, mc, plan, wplan))
                continue
            kv.write_block_device(layer, sid, st, k, v, alloc=layer == 0, plan=wplan)
            plan = plan or VerifyPlan(kv, sid, st, C, Hq, mc)
            o.append(verify_attention(q, kv, layer, sid, st, mc, plan=plan))
        outs.append(o)
    for a, b in zip(*outs):
        assert _same(a, b)
    assert _same(kvs[0].k_pool, kvs[1].k_pool) and _same(kvs[0].v_pool, kvs[1].v_pool)
    return outs[1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,C,Hq,Hkv,d", [
    ([0, 1, 15, 16, 17, 127], 1, 14, 2, 64),              # one token: first, last and only place of a page
    ([0, 10, 14, 255, 256, 1000], 6, 12, 2, 128),         # within and across pages
    ([12, 4090, 700], 9, 14, 2, 64),                      # four query tiles; merged pieces
    ([3, 250, 16 * 31 + 13], 9, 4, 2, 128),
    ([5, 300], 40, 4, 2, 64),                             # 80 rows: two row groups write the same pages
    ([4100, 8190 - 7], 33, 2, 2, 128),                    # a chunk over three or four pages, two pieces
    ([7 + 11 * i for i in range(140)], 3, 14, 2, 64),     # cost-balanced split
    ([1 + 3 * i for i in range(130)], 6, 12, 2, 128),
    ([9, 100], 64, 1, 1, 64),                             # the longest planned chunk
    ([20, 31], 7, 16, 2, 128),                            # four query tiles at 128: two launches
])
def test_equals_write_then_attend(cuda, dtype, lens, C, Hq, Hkv, d):
    kvs, g = _pools(cuda, lens, C, Hkv, d, dtype, 3, seed=C + d)
    for o in _compare(cuda, kvs, g, lens, C, Hq, Hkv, d, dtype, dtype):
        assert bool(torch.isfinite(o).all())


@pytest.mark.parametrize("qdtype,dtype", [(torch.float32, torch.float32), (torch.float16, torch.bfloat16)])
def test_types_without_a_planned_kernel(cuda, qdtype, dtype):
    lens, C = [20, 33, 64], 5
    kvs, g = _pools(cuda, lens, C, 2, 64, dtype, 3, seed=3)
    _compare(cuda, kvs, g, lens, C, 4, 2, 64, qdtype, dtype)


def test_exhausted_pool_writes_what_the_two_calls_write(cuda):
    lens, C = [30 + 3 * s for s in range(12)], 7
    cap = sum(-(-n // 16) for n in lens) + 2  # the chunk needs more blocks than are left
    kvs, g = _pools(cuda, lens, C, 2, 128, torch.bfloat16, 3, seed=5, cap=cap)
    _compare(cuda, kvs, g, lens, C, 12, 2, 128, torch.bfloat16, torch.bfloat16)
    for kv in kvs:
        with pytest.raises(BlockExhaustedError):
            kv.seq_lengths


def test_output_over_the_new_keys(cuda):
    # the write reads the keys before the attention overwrites them
    lens, C = [40, 70], 4
    (a, b), g = _pools(cuda, lens, C, 2, 64, torch.bfloat16, 2, seed=7)
    sid, st = _hip.i32([0, 1], cuda), _hip.i32(lens, cuda)
    q, k, v = (torch.randn(2, C, 2, 64, generator=g).to(torch.bfloat16).to(cuda) for _ in range(3))
    outs = []
    for kv in (a, b):
        wplan = WritePlan()
        kv.write_block_device(0, sid, st, k, v, alloc=True, plan=wplan)
        plan = VerifyPlan(kv, sid, st, C, 2, 70 + C)
        k1 = k.clone()
        outs.append(append_verify_attention(q, k1, v, kv, 1, sid, st, 70 + C, plan, wplan,
                                            out=k1 if kv is b else None))
    assert torch.equal(outs[0], outs[1]) and _same(a.k_pool, b.k_pool)


@pytest.mark.parametrize("which", ["keys", "values"])
def test_output_over_the_new_keys_through_another_storage(cuda, which):
    # half of the output lies over half of the new keys (values), in a storage of its own
    lens, C = [40, 70, 9], 4
    (a, b), g = _pools(cuda, lens, C, 2, 64, torch.bfloat16, 2, seed=8)
    sid, st = _hip.i32([0, 1, 2], cuda), _hip.i32(lens, cuda)
    q, k, v = (torch.randn(3, C, 2, 64, generator=g).to(torch.bfloat16).to(cuda) for _ in range(3))
    n = q.numel()
    outs = []
    for kv in (a, b):
        wplan = WritePlan()
        kv.write_block_device(0, sid, st, k, v, alloc=True, plan=wplan)
        plan = VerifyPlan(kv, sid, st, C, 2, 70 + C)
        buf = torch.zeros(2 * n, dtype=torch.bfloat16, device=cuda)
        new = buf[:n].copy_((k if which == "keys" else v).reshape(-1)).view_as(k)
        out = torch.from_dlpack(buf[n // 2:n // 2 + n]).view_as(k)
        assert out.untyped_storage().data_ptr() != new.untyped_storage().data_ptr()
        kn, vn = (new, v) if which == "keys" else (k, new)
        outs.append(append_verify_attention(q, kn, vn, kv, 1, sid, st, 70 + C, plan, wplan,
                                            out=out if kv is b else None))
    assert torch.equal(outs[0], outs[1]) and _same(a.k_pool, b.k_pool) and _same(a.v_pool, b.v_pool)
