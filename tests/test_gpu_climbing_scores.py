"""Attention where scores climb along the keys: the accumulators are rescaled only in steps where some row's maximum grew, and rows of
one wave climb, fall and stay level at once."""
import math

import pytest
import torch

import plain_model as P
from test_gpu_kernels import _paged

pytestmark = pytest.mark.gpu
KEYS, PAST = 460, 140


def _inputs(dh, climb):
    """One request, 2 heads over one kv head.  Keys climb by ``climb`` powers of two every 64 keys; queries follow them up, down or not."""
    g = torch.Generator().manual_seed(dh + int(climb))
    k, v = torch.randn(KEYS, 1, dh, generator=g) * 0.5, torch.rand(KEYS, 1, dh, generator=g) * 2 - 1
    k[:, 0, 0] = torch.arange(KEYS) * (climb / 64)
    q = torch.randn(KEYS - PAST, 2, dh, generator=g)
    q[:, :, 0] = torch.tensor([1.0, -1.0, 0.0])[torch.randint(0, 3, q.shape[:2], generator=g)]
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


@pytest.mark.parametrize("kernel", ["prefill", "span", "decode"])
@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("climb", [1.0, 7.75, 8.0, 8.25, 40.0])
def test_climbing_scores(kernel, dh, climb):
    from infinicore_infer_amd.kernels import ops
    q, k, v = _inputs(dh, climb)
    scale, n = math.log(2.0), KEYS - PAST                  # a score of one is one power of two
    want = P.plain_attention(q, k, v, scale, PAST, None).reshape(n, 2 * dh).double()
    kc, vc, bt = _paged(k, v, 64, torch.bfloat16, seed=3)
    qd, kc, vc, bt = q.reshape(n, 2 * dh).cuda(), kc.cuda(), vc.cuda(), bt[None].cuda()
    out = torch.full_like(qd, float("nan"))
    rows = ops.attention_prefill_tile_rows()
    tiles = torch.tensor([[0, o, min(rows, n - o), PAST + o] for o in range(0, n, rows)], dtype=torch.int32).cuda()
    if kernel == "decode":
        part = [torch.empty(n * 2 * 3 * m, device="cuda") for m in (dh, 2)]
        rows = torch.arange(PAST, KEYS, dtype=torch.int32).cuda()
        ops.attention_decode(qd, out, kc, vc, bt, None, n, torch.zeros_like(rows), rows, *part, 2, 1, dh, 64, scale, 0, 3)
    elif kernel == "prefill":
        ops.attention_prefill(qd, out, kc, vc, bt, tiles, len(tiles), 2, 1, dh, 64, scale, 0, 1)
    else:
        ops.attention_span_prefill(qd, out, None, kc, vc, bt, tiles, len(tiles), 2, 1, dh, dh, 64, scale, 0, 0, None, 0.0)
    # Weights are rounded to bfloat16 (2^-9 of each, so at most 2^-9 of max|v| <= 1), the result once more; float32 scores of up to 2^9
    # with sums of dh products are good to about 2^-12 of a power of two: 2^-8 in all, doubled.
    err = float((out.cpu().double() - want).abs().max())
    assert err <= 2.0 ** -7, err
