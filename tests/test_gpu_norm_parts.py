"""Float32 rows that reach a product of parts already split: the norm and the gated unit that write the parts, and a product's slices that the norm adds up, against the kernels
that do each by itself, bit for bit (the same values in the same order)."""
import pytest
import torch

from infinicore_infer_amd.kernels import ops
from infinicore_infer_amd.kernels.lib import get_lib

pytestmark = pytest.mark.gpu
STREAM = 0


def _randn(g, *shape):
    return torch.randn(*shape, generator=g).cuda()


def _products(rows, parts, weight):
    """The product of the rows, split by itself and from the parts that are there."""
    lib, (M, K), N = get_lib(), rows.shape, weight.shape[0]
    apart, ready = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    own = torch.empty(parts.numel(), dtype=torch.uint8, device="cuda")
    for out, ws, flag in ((apart, own, 0), (ready, parts, 1)):
        assert lib.ic_gemm_f32_between(rows.data_ptr(), weight.data_ptr(), out.data_ptr(), M, N, K, K, K, N, ws.data_ptr(), ws.numel(), flag, 0, STREAM) == 0
    return apart, ready


# one row of threads for two rows and for one, several vectors a thread, the narrowest and the widest row; rows short of and beyond whole tiles of 16
@pytest.mark.parametrize("d", [32, 96, 1536, 2048, 2304, 4160, 8224, 16384])
@pytest.mark.parametrize("M,slices", [(1, 1), (15, 2), (16, 1), (33, 4), (130, 3)])
def test_norm_with_slices_and_parts(d, M, slices):
    lib, g = get_lib(), torch.Generator().manual_seed(d * 1000 + M)
    x, y, w = _randn(g, M, d), _randn(g, slices, M, d), _randn(g, d)
    weight = _randn(g, 64, d)
    total = y[0].clone()
    for s in range(1, slices):
        total += y[s]
    want_x, want = x.clone(), torch.empty_like(x)
    ops.add_rmsnorm(want_x, total, 0.3, w, want, 1e-5)
    parts = torch.full((lib.ic_gemm_f32_parts_bytes(M, d),), 255, dtype=torch.uint8, device="cuda")
    got = torch.empty_like(x)
    rest = x.clone()
    assert lib.ic_norm_parts_f32(rest.data_ptr(), y.data_ptr(), slices, 0.3, w.data_ptr(), got.data_ptr(), 0, M, d, 1e-5, STREAM) == 0
    assert torch.equal(rest, want_x) and torch.equal(got, want)
    got.zero_()
    assert lib.ic_norm_parts_f32(x.data_ptr(), y.data_ptr(), slices, 0.3, w.data_ptr(), got.data_ptr(), parts.data_ptr(), M, d, 1e-5, STREAM) == 0
    assert torch.equal(x, want_x) and torch.equal(got, want)
    apart, ready = _products(got, parts, weight)
    assert torch.equal(apart, ready)


@pytest.mark.parametrize("di", [32, 96, 3840])
@pytest.mark.parametrize("M", [1, 16, 33, 130])
def test_swiglu_with_parts(di, M):
    lib, g = get_lib(), torch.Generator().manual_seed(di * 1000 + M)
    gate_up, weight = _randn(g, M, 2 * di), _randn(g, 64, di)
    want, got = torch.empty(M, di, device="cuda"), torch.empty(M, di, device="cuda")
    ops.swiglu(gate_up, want)
    parts = torch.full((lib.ic_gemm_f32_parts_bytes(M, di),), 255, dtype=torch.uint8, device="cuda")
    assert lib.ic_swiglu_parts_f32(gate_up.data_ptr(), got.data_ptr(), parts.data_ptr(), M, di, STREAM) == 0
    assert torch.equal(got, want)
    apart, ready = _products(got, parts, weight)
    assert torch.equal(apart, ready)


def test_slices_that_a_product_leaves():
    """Behind A's parts, [slice][row][column]; their sum is the product's own result."""
    lib, (M, N, K) = get_lib(), (517, 1536, 3840)
    g = torch.Generator().manual_seed(5)
    a, w, c = _randn(g, M, K), _randn(g, N, K), torch.zeros(M, N, device="cuda")
    ws = torch.empty(lib.ic_gemm_f32_workspace_bytes(M, N, K), dtype=torch.uint8, device="cuda")
    args = (a.data_ptr(), w.data_ptr(), c.data_ptr(), M, N, K, K, K, N, ws.data_ptr(), ws.numel())
    slices = lib.ic_gemm_f32_whole(*args)
    assert slices > 1
    assert lib.ic_gemm_f32_between(*args, 0, 1, STREAM) == 0
    at = lib.ic_gemm_f32_parts_bytes(M, K)
    left = ws[at:at + 4 * slices * M * N].view(torch.float32).view(slices, M, N)
    total = left[0].clone()
    for s in range(1, slices):
        total += left[s]
    assert not c.any()
    assert lib.ic_gemm_f32_between(*args, 1, 0, STREAM) == 0
    assert torch.equal(c, total)
    # not in parts: few rows, or room for some of the rows only
    assert lib.ic_gemm_f32_whole(*args[:3], 32, *args[4:]) == 0
    assert lib.ic_gemm_f32_whole(*args[:10], lib.ic_gemm_f32_parts_bytes(64, K)) == 0
    assert lib.ic_gemm_f32_between(*args[:10], lib.ic_gemm_f32_parts_bytes(64, K), 1, 0, STREAM) != 0


def test_steps_in_parts_equal_steps_product_by_product(tmp_path_factory):
    """A float32 step issued natively (parts from the norms and the gated unit, slices added by the norm) and kernel by kernel, on three layers of the 1B shape: bit for bit."""
    import os

    import helpers as H
    from infinicore_infer_amd.engine import Engine, StepEntry
    from infinicore_infer_amd.weights import write_random_model
    cfg = dict(model_type="minicpm", vocab_size=5003, hidden_size=1536, num_hidden_layers=3, num_attention_heads=24, num_key_value_heads=8, intermediate_size=3840,
               max_position_embeddings=1024, rms_norm_eps=1e-5, rope_theta=10000.0, scale_emb=12, dim_model_base=256, scale_depth=1.4, tie_word_embeddings=True, eos_token_id=2)
    folder = os.path.join(str(tmp_path_factory.getbasetemp()), "model_norm_parts")
    write_random_model(folder, cfg, seed=3, std=0.02)
    a, b = [Engine.from_dir(folder, dtype=torch.float32, max_tokens=4096, use_native=n, page_size=64, max_requests=8) for n in (True, False)]
    assert a.native is not None and b.native is None
    for j, n in enumerate((517, 33, 130, 300)):
        ents = [StepEntry("p%d" % j, H.random_tokens(5003, n, j), [0, n - 1])] + [StepEntry("p%d" % i, [9 + i], [0]) for i in range(j)]
        assert torch.equal(a.step(ents), b.step(ents))


def test_norm_weights_that_are_not_aligned():
    """The norms without parts take any weight, and a step with such weights runs as it did: bit for bit the one issued kernel by kernel."""
    import helpers as H
    from infinicore_infer_amd.engine import StepEntry
    from test_gpu_large import SHAPE_1B, _engine_and_weights
    cfg = dict(SHAPE_1B, vocab_size=2003, num_hidden_layers=4)
    engines = [_engine_and_weights(cfg, 21, 0.02, 4096, 8, dtype=torch.float32, use_native=False)[0] for _ in range(2)]
    from infinicore_infer_amd.engine.native import NativeDecoder
    for e in engines:
        for i, norm in enumerate(n for l in e.model.layers for n in (l.mixer_norm, l.feed_forward_norm)):
            if i % 3 != 2:                                   # (aligned ones beside them: a product's slices and parts, or none)
                off = torch.empty(norm.weight.numel() + 1, device="cuda")
                off[1:].copy_(norm.weight)
                norm.weight = off[1:]
    engines[0].native = NativeDecoder.try_build(engines[0])
    assert engines[0].native is not None
    for n in (517, 130):
        got, want = [e.step([StepEntry("p%d" % n, H.random_tokens(2003, n, 3), [0, n - 1])]).clone() for e in engines]
        assert torch.equal(got, want)
    assert engines[0].native_steps == 2
