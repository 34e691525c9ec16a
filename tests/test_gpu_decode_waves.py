"""Attention of single tokens with grouped queries at the sizes where the number of waves of a block changes: one split of few (row, kv
head) pairs, just below and above the line; many splits of heads of 128, more of them than there are key tiles."""
import pytest
import torch

from test_gpu_kernels import _attention_case, _close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkvh,dh,rows,n_split", [(6, 2, 64, 64, 1), (6, 2, 64, 65, 1), (16, 8, 64, 16, 1), (8, 2, 128, 5, 23), (8, 2, 128, 5, 24),
                                                     (32, 2, 128, 3, 32), (4, 1, 128, 5, 64)])
@pytest.mark.parametrize("window", [None, 100])
def test_grouped_queries_with_four_and_eight_waves(nh, nkvh, dh, rows, n_split, window):
    lens = [((0, 31, 32, 255, 256, 257, 511, 1031)[i % 8] + i // 8, 1) for i in range(rows)]
    got, want = _attention_case(torch.bfloat16, nh, nkvh, dh, 64, lens, window, 51, "decode", n_split=n_split)
    _close(got, want, torch.bfloat16, factor=3)


@pytest.mark.parametrize("page", [1, 2, 3, 48, 2047, 2048])          # a key's page by a multiplication, where ids are staged and exact
@pytest.mark.parametrize("dtype,nh,nkvh,dh", [(torch.bfloat16, 6, 2, 64), (torch.bfloat16, 3, 3, 64), (torch.bfloat16, 4, 2, 128),
                                              (torch.float32, 6, 2, 64)])
def test_page_sizes(page, dtype, nh, nkvh, dh):
    lens = [(n, 1) for n in (0, page - 1, page, 46, 95, 96, 500, min(1031, 1000 * page))]
    got, want = _attention_case(dtype, nh, nkvh, dh, page, lens, None, 52, "decode", n_split=3)
    _close(got, want, dtype, factor=3)
