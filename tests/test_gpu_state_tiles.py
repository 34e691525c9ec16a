"""The matrix state recurrence of prompt portions, chunk by chunk, at every split of a state over a block's threads: chunks of all
remainders of the tokens staged at a time, chunks of one token, step sizes and fixed decays, rows in both types."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _recurrence(x, B, C, dt, decay, D, S):
    """One request in float64: x [T, H, P], B, C [T, H, N], dt, decay [T, H], S [H, N, P]; returns (y, S)."""
    y = torch.empty_like(x)
    for t in range(x.shape[0]):
        S = decay[t][:, None, None] * S + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None, :]
        y[t] = (S * C[t][:, :, None]).sum(1) + D[:, None] * x[t]
    return y, S


@pytest.mark.parametrize("P,N", [(32, 128), (64, 64), (64, 128), (128, 32), (128, 128), (256, 64), (64, 96)])     # the last: the other kernel
@pytest.mark.parametrize("steps,dtype", [(True, torch.bfloat16), (True, torch.float32), (False, torch.bfloat16)])
def test_chunked_portions(P, N, steps, dtype):
    from infinicore_infer_amd.kernels import ops
    H, G, lens, chunk = 4, 2 if steps else 4, [67, 1, 34, 101], 33
    g = torch.Generator().manual_seed(P + N)
    T, R, inner = sum(lens), len(lens), H * P
    rows = (torch.randn(T, inner + 2 * G * N, generator=g) * 0.5).to(dtype)
    dt_raw = torch.randn(T, H, generator=g).to(dtype) if steps else None
    bias = torch.randn(H, generator=g) - 1.0 if steps else None
    rate = -torch.exp(torch.randn(H, generator=g) * 0.5) if steps else torch.rand(H, generator=g) * 0.3 + 0.7
    skip = torch.rand(H, generator=g) if steps else None
    state = torch.randn(R + 1, inner * N, generator=g) * 0.3
    slots, starts = [2, 0, 4, 1], [0, 67, 68, 102, 203]
    d64 = rows.double()
    act = lambda v: v if steps else v * torch.sigmoid(v)              # linear attention's rows come with silu on the way in
    x = act(d64[:, :inner]).view(T, H, P)
    B = act(d64[:, inner:inner + G * N]).view(T, G, N).repeat_interleave(H // G, 1)
    C = act(d64[:, inner + G * N:]).view(T, G, N).repeat_interleave(H // G, 1)
    if steps:
        dt = torch.nn.functional.softplus(dt_raw.double() + bias.double())
        decay = torch.exp(rate.double() * dt)
    else:
        dt, decay = torch.ones(T, H, dtype=torch.float64), rate.double().expand(T, H)
    D = skip.double() if steps else torch.zeros(H, dtype=torch.float64)
    st, y = state.to(DEV), torch.full((T, inner), float("nan"), device=DEV)
    most = (max(lens) + chunk - 1) // chunk
    scratch = (chunk, most, torch.full((R * most * inner * N,), float("nan"), device=DEV), torch.full((R * most * H,), float("nan"), device=DEV))
    dev = lambda t: None if t is None else t.to(DEV)
    ops.ssm_scan(rows.to(DEV), dev(dt_raw), dev(bias), rate.to(DEV), dev(skip), H, P, N, G, y, st, 0,
                 torch.tensor(starts, dtype=torch.int32, device=DEV), torch.tensor(slots, dtype=torch.int32, device=DEV), R, chunks=scratch,
                 in_act=None if steps else "silu")
    y, st = y.cpu().double(), st.cpu().double()
    for r, (a, n) in enumerate(zip(starts, lens)):
        at = slice(a, a + n)
        wy, ws = _recurrence(x[at], B[at], C[at], dt[at], decay[at], D, state[slots[r]].double().view(H, N, P))
        # float32 throughout: a state entry is a sum of n terms that each carry a few roundings of 2^-24 (the decays' products up to n),
        # an output a sum of N of them
        mag_s = float((state[slots[r]].abs().max() + (B[at].abs().amax() * x[at].abs().amax() * dt[at].amax()) * min(n, 40)))
        assert float((st[slots[r]].view(H, N, P) - ws).abs().max()) <= mag_s * (n + 8) * 2.0 ** -24
        mag_y = float((C[at].abs().sum(-1).max()) * ws.abs().max().clamp(min=1.0)) + float(x[at].abs().max())
        assert float((y[at].view(n, H, P) - wy).abs().max()) <= mag_y * (n + 8) * 2.0 ** -24
    assert torch.equal(st[3], state[3].double())                       # a slot that no request owns
