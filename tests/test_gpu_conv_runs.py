"""The convolution per channel of long steps, a run of tokens a thread: against the kernel of short steps (same sums in the same order, so the
same bits), which rows that are not aligned still take, and against the plain convolution."""
import pytest
import torch

import plain_mezinex as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [64, 4100])                               # a block's channels in part, and the last of five blocks in part
@pytest.mark.parametrize("act", ["none", "silu"])
def test_runs_of_tokens(dtype, C, act):
    from infinicore_infer_amd.kernels import ops
    lens = [1, 2, 3, 8, 7, 12, (1 << 20) // C + 5]                     # requests that begin at, just before and just after a run's edge
    T, g = sum(lens), torch.Generator().manual_seed(C)
    w, b, ib = torch.randn(C, 4, generator=g).cuda(), torch.randn(C, generator=g).cuda(), torch.randn(C, generator=g).cuda()
    rows = torch.randn(T, C, generator=g).to(dtype).cuda()
    state = torch.randn(9, 3 * C + 7, generator=g).cuda()
    starts = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    req = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).cuda()
    slots = torch.tensor([8, 0, 3, 5, 1, 7, 2], dtype=torch.int32).cuda()
    got = []
    for off in (0, 1):                                                # whole 4-element pieces, and not
        x = torch.zeros(T, C + 4, dtype=dtype, device="cuda")
        x[:, off:off + C] = rows
        st, out = state.clone(), torch.full((T, C), float("nan"), device="cuda")
        copy = torch.zeros(T, C, dtype=dtype, device="cuda")
        ops.causal_conv(x[:, off:off + C], w, b, out, st, 5, req, starts, slots, len(lens), in_bias=ib, out_copy=copy, act=act)
        got.append((out, copy, st))
    for one, other in zip(*got):
        assert torch.equal(one, other)
    # float32 sums of five terms, each term and sum good to 2^-24 of at most sum |w| |x| + |b|; silu's slope is below 1.1
    for i, s in enumerate(starts[:-1].tolist()):
        before = state[slots[i].long(), 5:5 + 3 * C].view(3, C).double()
        seq = torch.cat([before, rows[s:s + lens[i]].double() + ib.double()])
        pick = slice(0, C, 997)
        y = P.causal_conv(seq[:, pick].cpu(), w[pick].double().cpu(), b[pick].double().cpu())[3:]
        size = P.causal_conv(seq[:, pick].abs().cpu(), w[pick].abs().double().cpu(), b[pick].abs().double().cpu())[3:]
        want = P.silu(y) if act == "silu" else y
        assert ((got[0][0][s:s + lens[i], pick].cpu().double() - want).abs() <= 1e-6 * (1 + size)).all()
