"""Kernels that send several rounds of loads ahead, at the widths where a round or a run of rounds ends, and the few-token grids."""
import pytest
import torch

import plain_mezinex as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 4, 5])                           # four, two and one round ahead
@pytest.mark.parametrize("d", [4, 1020, 1024, 1028, 2052, 4096, 4100, 8200, 1023])
def test_streams_at_the_edges_of_rounds(S, d):
    from infinicore_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(d)
    r = lambda *shape: torch.randn(*shape, generator=g)
    xs, y, mix, ow, iw, nw = r(S, 3, d), r(3, d).bfloat16(), r(S, S), r(S), r(S), r(d)
    new = P.hyper_write(xs.double(), y.double(), mix.double(), ow.double())
    u = P.hyper_read(new, iw.double())
    x, h = xs.cuda(), torch.full((3, d), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.hc_step(x, y=y.cuda(), mix=mix.cuda(), out_w=ow.cuda(), in_w=iw.cuda(), norm_w=nw.cuda(), eps=1e-5, h=h)
    # sums of S + 1 float32 terms of at most `size`: 8 of their roundings; the norm's factor adds two more, bfloat16 rounds to 2^-9
    size = float((mix.abs().T @ xs.abs().flatten(1)).max() + (ow.abs().max() * y.abs().max()))
    assert float((x.cpu().double() - new).abs().max()) <= 8 * 2.0 ** -24 * size
    want = P.rms(u, 1e-5) * nw.double()
    assert ((h.cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()
    total = torch.full((3, d), float("nan"), device="cuda")
    ops.hc_step(x, in_w=torch.ones(S, device="cuda"), h=total)        # the read alone, no norm
    assert float((total.cpu().double() - new.sum(0)).abs().max()) <= 32 * 2.0 ** -24 * size * S


@pytest.mark.parametrize("T", [1, 64, 65])                            # an item a thread, and a loop over a token's items
@pytest.mark.parametrize("Rq,R", [(255, 256), (2048, 512), (2049, 8), (2500, 257)])
@pytest.mark.parametrize("cached", [True, False])
def test_latent_rows(T, Rq, R, cached):
    from infinicore_infer_amd.kernels import ops
    E, rot, H, dim = 12, 8, 50, 4
    g = torch.Generator().manual_seed(Rq)
    rows = torch.randn(T, Rq + R + E, generator=g)
    qn, kn, pos = torch.randn(Rq, generator=g), torch.randn(R, generator=g), torch.randint(0, 200, (T,), generator=g, dtype=torch.int32)
    hi = torch.rand(rot // 2, generator=g)
    freq = torch.cat([hi, torch.zeros(rot // 2)])
    slots = torch.randperm(T, generator=g).to(torch.int32)

    def turned(v):                                                    # v [T, ..., E]
        ang = pos.double().view(-1, *[1] * (v.dim() - 1)) * hi.double()
        a, b = v[..., 0:rot:2], v[..., 1:rot:2]
        out = v.clone()
        out[..., 0:rot:2], out[..., 1:rot:2] = a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()
        return out

    cq = torch.full((T, Rq), float("nan"), device="cuda")
    cache = torch.zeros(T, 1, 1, R + E, device="cuda")
    ops.latent_prep(rows.cuda(), Rq, R, E, qn.cuda(), kn.cuda(), 1e-5, freq.cuda(), rot, pos.cuda(), cq, cache, slots.cuda() if cached else None)
    x = rows.double()
    # float32 sums of squares over at most 2,500 columns (error far below 1e-5 of them), products of values below 20; angles below 200
    assert torch.allclose(cq.cpu().double(), P.rms(x[:, :Rq], 1e-5) * qn.double(), rtol=2e-5, atol=1e-5)
    if cached:
        want = torch.cat([P.rms(x[:, Rq:Rq + R], 1e-5) * kn.double(), turned(x[:, Rq + R:])], -1)
        assert torch.allclose(cache.cpu().double().view(T, -1)[slots.long()], want, rtol=2e-5, atol=5e-5)
    else:
        assert not cache.any()
    q = torch.randn(T, H, dim + E, generator=g)
    qa = torch.zeros(T, H * (R + E), device="cuda")
    ops.latent_q_rotate(q.view(T, -1).cuda(), dim, E, R, H, freq.cuda(), rot, pos.cuda(), qa)
    got = qa.cpu().double().view(T, H, R + E)
    assert torch.allclose(got[..., R:], turned(q[..., dim:].double()), atol=5e-5) and not got[..., :R].any()
