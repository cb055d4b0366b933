"""The filtered sampler's workspace holder on the CPU: a batch that grows one
sequence at a time leaves replaced buffers (kept for graphs captured earlier)
that together stay below the one in use."""

import torch

from engine import _hip
from engine import spec_scheduler as es

STEP = 9000


def test_replaced_buffers_stay_below_the_live_one():
    ws, cpu = _hip.Workspace(es._filter_workspace._factor), torch.device("cpu")
    for b in range(1, 65):
        buf = ws.get(b * STEP, cpu, stream=0)
        assert b * STEP <= buf.numel() <= 2 * b * STEP and not bool(buf.any())
        assert sum(t.numel() for t in ws._retired) <= buf.numel()
    assert ws.get(STEP, cpu, stream=0) is buf
    assert ws.get(10 * buf.numel(), cpu, stream=0).numel() == 10 * buf.numel()
    assert ws.get(STEP, cpu, stream=1).numel() == STEP
