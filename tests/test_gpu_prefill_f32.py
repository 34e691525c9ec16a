"""Prompt portions in float32 with two and four key groups a block (chosen from the number of (tile, head) pairs; one group and the lines
between them: test_prefill_f32_groups.py): tiles of all heights, walks shorter and longer than a step, a window."""
import pytest
import torch

from test_gpu_kernels import _attention_case, _close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkvh,dh,page", [(1, 1, 64, 16), (15, 5, 64, 64), (16, 8, 64, 64), (70, 10, 64, 32), (71, 71, 64, 64),
                                             (2, 1, 128, 64), (25, 5, 128, 32), (26, 2, 128, 64)])
@pytest.mark.parametrize("window", [None, 70])
def test_key_groups(nh, nkvh, dh, page, window):
    lens = [(0, 2), (0, 31), (0, 129), (130, 65), (257, 160), (31, 97), (700, 33)]          # nine tiles
    got, want = _attention_case(torch.float32, nh, nkvh, dh, page, lens, window, 61, "prefill")
    _close(got, want, torch.float32, factor=3)


@pytest.mark.parametrize("nh,nkvh,dh,lens", [(2, 1, 64, [(40, 150)]), (26, 13, 64, [(0, 640)]), (72, 9, 64, [(3, 1300)]), (4, 2, 128, [(40, 150)]), (41, 41, 128, [(0, 1300)])])
def test_products_of_parts(nh, nkvh, dh, lens):
    """Error against 64 bits with one, two and four key groups: that of float32 sums whose roundings are of either sign, one per 16 keys
    and four for the score, the softmax and the way out, 2^-24 each (float32 instructions 2.0..4.3e-7, parts of which one product of three is left out 2^-18.5).  A key with an infinity, whose parts are no numbers, counts as a score of -inf."""
    from infinicore_infer_amd.kernels import ops
    dev, ps, (past, n) = "cuda", 64, lens[0]
    g = torch.Generator().manual_seed(dh + n)
    pages = -(-(past + n) // ps)
    for infinite in (False, True):
        k, v = (torch.randn(pages, nkvh, ps, dh, generator=g).to(dev) for _ in range(2))
        q = torch.randn(n, (nh + 2 * nkvh) * dh, generator=g).to(dev)
        if infinite:
            q[:, :nh * dh:dh] = q[:, :nh * dh:dh].abs() + 0.5
            k[pages // 2, :, 5, 0] = float("-inf")
        tiles = torch.tensor([(0, i, min(128, n - i), past + i) for i in range(0, n, 128)][::-1], dtype=torch.int32, device=dev)
        table = torch.arange(pages, dtype=torch.int32, device=dev)[None]
        out = torch.empty(n, nh * dh, device=dev)
        ops.attention_prefill(q, out, k, v, table, tiles, len(tiles), nh, nkvh, dh, ps, dh ** -0.5, 0)
        seen = torch.arange(past + n)[None] <= past + torch.arange(n)[:, None]
        wrong = total = 0.0
        for h in range(0, nh, max(1, nh // 4)):
            kh, vh = (x[:, h // (nh // nkvh)].reshape(-1, dh)[:past + n].double().cpu() for x in (k, v))
            s = (q[:, h * dh:(h + 1) * dh].double().cpu() @ kh.t() * dh ** -0.5).masked_fill(~seen, float("-inf"))
            want = torch.softmax(s, -1) @ vh
            wrong += float((out[:, h * dh:(h + 1) * dh].double().cpu() - want).square().sum())
            total += float(want.square().sum())
        assert (wrong / total) ** 0.5 < 2 ** -24 * (4 + ((past + n) / 16) ** 0.5)


@pytest.mark.parametrize("nh,dh", [(100, 64), (400, 64), (800, 64), (100, 128), (500, 128)])
def test_products_of_parts_err_to_both_sides(nh, dh):
    """Values that are all one number whose lower 16 bits are ones: every result is that number, off by the roundings of two sums of at most 16 terms (one chunk of keys, so
    that no small product meets a large sum), to either side: 2^-24 a rounding.  Parts cut off instead of rounded are off by 2^-23.4 on average, towards zero (rounded: 2^-26.3)."""
    from infinicore_infer_amd.kernels import ops
    dev, n, ps = "cuda", 16, 64
    x = torch.tensor(0x3f80ffff, dtype=torch.int32).view(torch.float32).item()
    g = torch.Generator().manual_seed(dh + nh)
    k, q = torch.randn(1, nh, ps, dh, generator=g).to(dev), torch.randn(n, 3 * nh * dh, generator=g).to(dev)
    tiles, out = torch.tensor([(0, 0, n, 0)], dtype=torch.int32, device=dev), torch.empty(n, nh * dh, device=dev)
    ops.attention_prefill(q, out, k, torch.full_like(k, x), torch.zeros(1, 1, dtype=torch.int32, device=dev), tiles, 1, nh, nh, dh, ps, dh ** -0.5, 0)
    off = out.double() / float(x) - 1.0
    assert abs(float(off.mean())) < 2.0 ** -24 and float(off.abs().max()) < 32 * 2.0 ** -24


@pytest.mark.parametrize("nh,dh", [(100, 64), (400, 64), (800, 64), (100, 128), (500, 128)])
def test_tiny_values(nh, dh):
    """Values under 2^-110, whose third part no bfloat16 number holds: the first token's result is its one value, and the others' keep a float32 sum's error."""
    from infinicore_infer_amd.kernels import ops
    dev, n, ps = "cuda", 16, 64
    g = torch.Generator().manual_seed(dh + nh)
    k, q = torch.randn(1, nh, ps, dh, generator=g).to(dev), torch.randn(n, 3 * nh * dh, generator=g).to(dev)
    v = (torch.randn(1, nh, ps, dh, generator=g) * 2.0 ** -113).to(dev)
    tiles, out = torch.tensor([(0, 0, n, 0)], dtype=torch.int32, device=dev), torch.empty(n, nh * dh, device=dev)
    ops.attention_prefill(q, out, k, v, torch.zeros(1, 1, dtype=torch.int32, device=dev), tiles, 1, nh, nh, dh, ps, dh ** -0.5, 0)
    first = v[0, :, 0].reshape(-1).double()
    whole = first.abs() > 2.0 ** -120
    assert float((out[0].double() / first - 1.0).abs()[whole].max()) < 2.0 ** -23
    s = (q[:, :dh].double().cpu() @ k[0, 0, :n].double().cpu().t() * dh ** -0.5).masked_fill(~torch.ones(n, n).tril().bool(), float("-inf"))
    p, v0 = torch.softmax(s, -1), v[0, 0, :n].double().cpu()
    assert bool(((out[:, :dh].double().cpu() - p @ v0).abs() <= (64 + 2 * dh ** 0.5) * 2.0 ** -24 * (p @ v0.abs())).all())
