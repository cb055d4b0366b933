"""Host integers carried to the device by a launch (``_hip.i32s``,
spv_put_ints) against ``torch.tensor``: the edges of the two argument sizes,
several lists in one launch, tensors among them, values that are not plain
32-bit integers, and a list changed right after the call."""

import pytest
import torch

from engine import _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (16, 17), (100, 28), (128,), (129,), (3, 960), (960,), (961,), (944, 16),
                                   (945, 16), (2000, 5, 7), (0, 4)])
def test_lists_arrive(cuda, sizes):
    lists = [[(-1) ** i * (i * 2654435761 % 2 ** 31) for i in range(k, k + n)] for k, n in enumerate(sizes)]
    t = torch.arange(5, device=cuda)
    got = _hip.i32s(cuda, *lists, t)
    want = [torch.tensor(x, dtype=torch.int32, device=cuda) for x in lists]
    for x in lists:
        x[:] = [7] * len(x)
    for a, b in zip(got, want + [t.int()]):
        assert a.dtype == torch.int32 and a.is_contiguous() and torch.equal(a, b)


def test_other_values_are_torch_tensors_affair(cuda):
    assert _hip.i32([True, False], cuda).tolist() == [1, 0]
    assert _hip.i32((x for x in (3, 4)), cuda).tolist() == [3, 4]
    assert _hip.i32([2 ** 31 - 1, -2 ** 31], cuda).tolist() == [2 ** 31 - 1, -2 ** 31]
    assert _hip.i32([2.0, 3.0], cuda).tolist() == torch.tensor([2.0, 3.0], dtype=torch.int32).tolist()
    with pytest.raises((RuntimeError, OverflowError)):
        _hip.i32([2 ** 40], cuda)
