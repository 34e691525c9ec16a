"""The few-row products with an epilogue at the sizes where the kernel for up to 8 rows can go wrong: one line of K and its
longest, widths that are no multiple of its groups of 8 weight rows, one and several groups a block, rows that do not exist."""
import pytest
import torch

import plain_model as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ops():
    from infinicore_infer_amd.kernels import ops
    return ops


def _bound(a, w):
    """What a product rounded to bfloat16 may be off by: half a unit in the last place of the result, and the float32 sum's own
    error (K additions of terms that are exact products)."""
    exact = a.double() @ w.double().t()
    return exact, exact.abs() * 2.0 ** -8 + (a.double().abs() @ w.double().abs().t()) * (a.shape[1] * 2.0 ** -24)


def _inputs(seed, M, N, K):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(M, K, generator=g).to(torch.bfloat16), (torch.randn(N, K, generator=g) * 0.1).to(torch.bfloat16), g)


@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(5, 64), (256, 128), (250, 192), (2304, 2304), (2300, 704), (4096, 1088), (4090, 64), (1536, 8128), (1001, 5760)])
def test_residual_epilogue(M, N, K):
    ops = _ops()
    a, w, g = _inputs(M + N + K, M, N, K)
    x, gw = torch.randn(M, N, generator=g), torch.rand(N, generator=g) + 0.5
    xd, y = x.to(DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    sumsq = torch.full((ops.residual_parts(N), 16), float("nan"), device=DEV)
    ops.gemm_nt(a.to(DEV), w.to(DEV), y, residual=(xd, gw.to(DEV), 0.5, sumsq))
    exact, tol = _bound(a, w)
    got = xd.cpu().double()
    assert bool(((got - x.double() - 0.5 * exact).abs() <= 0.5 * tol + got.abs() * 2.0 ** -23 + x.double().abs() * 2.0 ** -23).all())
    assert bool(((y.cpu().double() - got * gw.double()).abs() <= (got * gw.double()).abs() * 2.0 ** -8).all())
    ss = sumsq.cpu().double().sum(0)
    assert bool(((ss[:M] - (got * got).sum(1)).abs() <= (got * got).sum(1) * (N * 2.0 ** -24 + 1e-6)).all())
    assert bool((ss[M:] == 0).all())                 # rows that do not exist add nothing


@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("di,K", [(3, 64), (2048, 128), (2041, 192), (3840, 1536), (4100, 64), (5760, 2304), (6143, 192), (8200, 128), (40, 8128)])
def test_gate_up_epilogue(M, di, K):
    ops = _ops()
    a, w, _ = _inputs(M + di + K, M, 2 * di, K)
    out = torch.full((M, di), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_nt(a.to(DEV), w.to(DEV), out, swiglu_output=True)
    exact, tol = _bound(a, w)
    (gate, up), (tg, tu) = exact.split(di, 1), tol.split(di, 1)
    want = P.plain_swiglu(gate, up)
    # |d silu / d gate| <= 1.1; the activation's own two hardware functions and its rounding are one more unit
    limit = 1.1 * up.abs() * tg + P.plain_swiglu(gate, torch.ones_like(up)).abs() * tu + 1.1 * tg * tu + want.abs() * 2.0 ** -7
    assert bool(((out.cpu().double() - want).abs() <= limit).all())


@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("nh,nkvh,dh,K,page", [(1, 1, 32, 64, 16), (24, 8, 64, 1536, 64), (36, 36, 64, 128, 32), (5, 1, 128, 8128, 64),
                                               (3, 3, 96, 192, 16), (32, 2, 128, 4096, 64)])
def test_rotary_and_cache_write_epilogue(M, nh, nkvh, dh, K, page):
    ops = _ops()
    H = (nh + 2 * nkvh) * dh
    a, w, g = _inputs(M + H + K, M, H, K)
    pos = torch.randint(0, 300, (M,), generator=g, dtype=torch.int32)
    slots = torch.randperm(5 * page, generator=g)[:M].to(torch.int32)
    if M > 2:
        slots[1] = -1                                # a row without a cache slot writes nothing
    sin, cos = (t.float() for t in P.plain_rope_tables(dh, 10000.0, 300))
    kc = torch.zeros(5, nkvh, page, dh, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    qkv = torch.zeros(M, H, dtype=torch.bfloat16, device=DEV)
    ops.gemm_qkv_rope(a.to(DEV), w.to(DEV), qkv, pos.to(DEV), slots.to(DEV), cos.to(DEV), sin.to(DEV), kc, vc, nh, nkvh, dh, page)
    exact, tol = _bound(a, w)
    half, c, s = dh // 2, cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
    e, t = exact.view(M, -1, dh), tol.view(M, -1, dh)
    lo, hi = e[..., :half] * c - e[..., half:] * s, e[..., half:] * c + e[..., :half] * s
    rot = torch.cat([lo, hi], -1)
    rtol = torch.cat([t[..., :half] * c.abs() + t[..., half:] * s.abs(), t[..., half:] * c.abs() + t[..., :half] * s.abs()], -1) + rot.abs() * 2.0 ** -7 + 1e-6
    assert bool(((qkv.cpu().double().view(M, -1, dh)[:, :nh] - rot[:, :nh]).abs() <= rtol[:, :nh]).all())
    kc, vc = kc.cpu().double(), vc.cpu().double()
    written = torch.zeros(5, page, dtype=torch.bool)
    for m, slot in enumerate(slots.tolist()):
        if slot < 0:
            continue
        written[slot // page, slot % page] = True
        k, v = kc[slot // page, :, slot % page], vc[slot // page, :, slot % page]
        assert bool(((k - rot[m, nh:nh + nkvh]).abs() <= rtol[m, nh:nh + nkvh]).all())
        assert bool(((v - e[m, nh + nkvh:]).abs() <= t[m, nh + nkvh:]).all())
    assert float(kc.permute(0, 2, 1, 3)[~written].abs().sum()) == 0 and float(vc.permute(0, 2, 1, 3)[~written].abs().sum()) == 0
