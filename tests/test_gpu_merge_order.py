"""The order and rounding of the sums that merge running-softmax states: fixed, whichever kernel they are in."""
import pytest
import torch

from infinicore_infer_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _fma(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _case(dtype, nh, nkvh, dh, rows, keys, seed, portion=0):
    """(q, k, v, tables, positions): one request a row of up to `keys` keys, and one with a portion of that many tokens behind them."""
    g, page = torch.Generator().manual_seed(seed), 64
    per = -(-max(keys, portion) // page)
    T = rows + portion
    k, v = (torch.randn((rows + 1) * per, nkvh, page, dh, generator=g).to(dtype).cuda() for _ in range(2))
    q = (1.5 * torch.randn(T, (nh + 2 * nkvh) * dh, generator=g)).to(dtype).cuda()
    tables = torch.arange((rows + 1) * per, dtype=torch.int32).view(rows + 1, per).cuda()
    positions = torch.tensor([keys - 1 - 3 * i for i in range(rows)] + list(range(portion)), dtype=torch.int32).cuda()
    requests = torch.tensor(list(range(rows)) + [rows] * portion, dtype=torch.int32).cuda()
    return q, k, v, tables, positions, requests, page


@pytest.mark.parametrize("nh,nkvh,dh", [(6, 6, 64), (4, 4, 128), (8, 2, 64)])
@pytest.mark.parametrize("splits", [2, 5, 9, 33, 64])
def test_merge_of_splits(nh, nkvh, dh, splits):
    """float32, bit for bit: weights exp(m - max); the weighted sums' total by halves of the wave, where a lane's own product enters the first sum unrounded;
    thread group j of 256 / head size takes splits j, j + groups, .. one after the other."""
    rows, groups = 3, 256 // dh
    q, k, v, tables, positions, requests, page = _case(torch.float32, nh, nkvh, dh, rows, 2064, 7 * splits + dh)
    out = torch.empty(rows, nh * dh, device="cuda")
    acc, ml = torch.empty(rows, nh, splits, dh, device="cuda"), torch.empty(rows, nh, splits, 2, device="cuda")
    ops.attention_decode(q, out, k, v, tables, None, rows, requests, positions, acc, ml, nh, nkvh, dh, page, dh ** -0.5, 0, splits)
    m = torch.full((rows, nh, 64), float("-inf"), device="cuda")
    l = torch.zeros(rows, nh, 64, device="cuda")
    m[..., :splits], l[..., :splits] = ml[..., 0], ml[..., 1]
    w = torch.exp(m - m.amax(-1, keepdim=True))
    lanes = torch.arange(64, device="cuda")
    s = _fma(l, w, (l * w)[..., lanes ^ 32])
    for d in (16, 8, 4, 2, 1):
        s = s + s[..., lanes ^ d]
    want = None
    for j in range(groups):
        a = torch.zeros(rows, nh, dh, device="cuda")
        for i in range(j, splits, groups):
            a = _fma(acc[:, :, i], w[..., i, None], a)
        want = a if want is None else want + a
    want = want * (1.0 / s[..., torch.arange(dh, device="cuda") % 64])      # (lanes i and i ^ 32 may differ in their totals' last bit)
    assert torch.equal(out.view(rows, nh, dh), want)


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("keys", [40, 700, 2064])
def test_states_of_single_tokens_are_the_same_in_both_launches(dh, keys):
    """Ungrouped bfloat16 heads: alone and beside a prompt's tiles the splits' float32 states are the same bits."""
    nh, rows, portion, splits = 6, 5, 70, 3
    q, k, v, tables, positions, requests, page = _case(torch.bfloat16, nh, nh, dh, rows, keys, keys + dh, portion)
    listed = torch.arange(rows, dtype=torch.int32).cuda()
    tiles = torch.tensor([(rows, rows, portion, 0)], dtype=torch.int32).cuda()
    states = []
    for together in (False, True):
        out = torch.zeros(rows + portion, nh * dh, dtype=torch.bfloat16, device="cuda")
        acc, ml = torch.zeros(rows, nh, splits, dh, device="cuda"), torch.zeros(rows, nh, splits, 2, device="cuda")
        if together:
            ops.attention_mixed(q, out, k, v, tables, listed, rows, requests, positions, acc, ml, splits, tiles, 1, nh, nh, dh, page, dh ** -0.5)
        else:
            ops.attention_decode(q, out, k, v, tables, listed, rows, requests, positions, acc, ml, nh, nh, dh, page, dh ** -0.5, 0, splits)
        states.append((acc, ml, out[:rows]))
    for alone, beside in zip(*states):
        assert torch.equal(alone, beside)
