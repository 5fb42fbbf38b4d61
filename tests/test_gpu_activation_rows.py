"""swiglu_with_probs / geglu_with_probs at the row lengths where the workgroup's size changes (2560, 4104, 6656 and 8200 columns), one
chunk to either side of them and of whole passes of 512 and 1024 threads, against the oracle with test_gpu_activation's bounds."""

import pytest
import torch

from tests.test_gpu_activation import test_forward_backward_vs_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("activation", ["silu", "gelu"])
@pytest.mark.parametrize("f", [2552, 2560, 4088, 4096, 4104, 6648, 6656, 8184, 8192, 8200])
def test_every_workgroup_size(gpu, activation, f):
    check(gpu, activation, 9, f, torch.float32)
