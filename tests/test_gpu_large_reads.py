"""Passes that read large tensors past the caches, at the lines of their rules."""
import pytest
import torch

import test_gpu_delta_rows as delta

pytestmark = pytest.mark.gpu


# output rows of 128 MB and a little less
@pytest.mark.parametrize("lens,D", [([5, 131067], 128), ([5, 131066], 128), ([70000, 262144 - 70000], 64)])
def test_delta_of_every_row_at_the_line(lens, D):
    delta.test_delta_of_every_row(lens, 4, D, torch.bfloat16)
