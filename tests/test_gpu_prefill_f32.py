"""Prompt portions in float32 with one, two and four key groups a block (chosen from the number of (tile, head) pairs): tiles of all
heights, walks shorter and longer than a step, a window."""
import pytest
import torch

from test_gpu_kernels import _attention_case, _close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkvh,dh,page", [(1, 1, 64, 16), (15, 5, 64, 64), (16, 8, 64, 64), (70, 10, 64, 32), (71, 71, 64, 64),
                                             (2, 1, 128, 64), (25, 5, 128, 32), (26, 2, 128, 64)])
@pytest.mark.parametrize("window", [None, 70])
def test_key_groups(nh, nkvh, dh, page, window):
    lens = [(0, 2), (0, 31), (0, 129), (130, 65), (257, 160), (31, 97), (700, 33)]          # ten tiles
    got, want = _attention_case(torch.float32, nh, nkvh, dh, page, lens, window, 61, "prefill")
    _close(got, want, torch.float32, factor=3)
