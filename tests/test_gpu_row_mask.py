"""The rows that hold tokens: one launch against the three it replaces, around the 16 rows of a thread and the 4096 of a
workgroup, with counts past, at and short of the buffer, negative ones, and calls that keep torch's own operations."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _want(lens, rows):
    return torch.arange(rows, device=lens.device) < lens.sum()


@pytest.mark.parametrize("rows", [0, 1, 15, 16, 17, 255, 4095, 4096, 4097, 70001])
@pytest.mark.parametrize("lens", [[0], [5], [7, 0, 9], [16, 4080], [4096, 1, -1], [-3, 2], [100000], [3] * 700])
def test_mask(gpu, rows, lens):
    from primus_amd.pytorch import ops

    t = torch.tensor(lens, dtype=torch.int64, device=gpu)
    got = ops.tokens_per_expert_to_mask(t, rows)
    assert got.dtype == torch.bool and got.shape == (rows,) and torch.equal(got, _want(t, rows))


def test_other_calls(gpu):
    from torch._subclasses.fake_tensor import FakeTensorMode

    from primus_amd.pytorch import ops

    t = torch.tensor([3, 0, 4], dtype=torch.int64, device=gpu)
    for other in (t.int(), t.cpu(), torch.stack([t, t], 1)[:, 0], t.view(1, 3)):
        assert torch.equal(ops.tokens_per_expert_to_mask(other, 9), _want(other, 9))
    batch = torch.stack([t, t + 1])
    got = torch.func.vmap(lambda v: ops.tokens_per_expert_to_mask(v, 9))(batch)
    assert torch.equal(got, torch.stack([_want(v, 9) for v in batch]))
    with FakeTensorMode() as mode:
        fake = mode.from_tensor(t)
        assert ops.tokens_per_expert_to_mask(fake, 9).shape == (9,)
