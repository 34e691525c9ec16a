"""Float32 products of several threads on one stream: what one product's kernels hand on to the next is not another's."""
import os
import threading

import pytest
import torch

import helpers as H
from infinicore_infer_amd.kernels import ops
from infinicore_infer_amd.kernels.lib import get_lib


def _together(calls):
    """Runs the calls in a thread each, started at the same time; their results."""
    start, out, wrong = threading.Barrier(len(calls)), [None] * len(calls), []

    def run(i):
        try:
            start.wait()
            out[i] = calls[i]()
        except BaseException as e:
            wrong.append(e)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if wrong:
        raise wrong[0]
    return out


def test_scratch_bytes():
    """Scratch memory grows with the rows (recorded steps share what the largest needs), holds 16 rows' parts at least, and none is asked for few rows."""
    lib = get_lib()
    for N, K in ((4, 32), (1536, 1536), (7680, 1536), (4096, 16384), (122753, 2304)):
        sizes = [lib.ic_gemm_f32_workspace_bytes(M, N, K) for M in (1, 32, 33, 48, 64, 65, 130, 517, 2048, 30000)]
        assert sizes[:2] == [0, 0] and sizes == sorted(sizes) and sizes[-1] <= 64 << 20
        assert all(s >= lib.ic_gemm_f32_parts_bytes(16, K) for s in sizes[2:])


@pytest.mark.gpu
def test_products_of_two_threads():
    M, N, K, n = 130, 7680, 1536, 60
    assert get_lib().ic_gemm_f32_pays(M, N, K)
    g = torch.Generator().manual_seed(5)
    w = torch.randn(N, K, generator=g).cuda()
    rows = [torch.randn(M, K, generator=g).cuda() for _ in range(2)]
    want = [ops.product(a, w, torch.empty(M, N, device="cuda")).clone() for a in rows]
    outs = [[torch.zeros(M, N, device="cuda") for _ in range(n)] for _ in rows]
    torch.cuda.synchronize()
    _together([lambda i=i: [ops.product(rows[i], w, o) for o in outs[i]] for i in range(2)])
    for i in range(2):
        assert all(torch.equal(o, want[i]) for o in outs[i])


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_engines_of_two_threads(tmp_path_factory, native):
    """Two float32 engines that step portions of 130 tokens on one stream: the same logits as one after the other."""
    from infinicore_infer_amd.engine import Engine, StepEntry
    from infinicore_infer_amd.weights import write_random_model
    cfg = dict(model_type="minicpm", vocab_size=2003, hidden_size=1536, num_hidden_layers=2, num_attention_heads=24, num_key_value_heads=8,
               intermediate_size=3840, max_position_embeddings=2048, rms_norm_eps=1e-5, rope_theta=10000.0, scale_emb=12, dim_model_base=256,
               scale_depth=1.4, tie_word_embeddings=True, eos_token_id=2)
    folder = os.path.join(str(tmp_path_factory.getbasetemp()), "model_two_threads")
    if not os.path.isdir(folder):
        write_random_model(folder, cfg, seed=7, std=0.02)
    steps = 10
    engines = [Engine.from_dir(folder, dtype=torch.float32, max_tokens=130 * steps, page_size=64, max_requests=2, use_native=native) for _ in range(2)]
    tokens = [H.random_tokens(cfg["vocab_size"], 130 * steps, 11 + i) for i in range(2)]

    def go(i):
        out = [engines[i].step([StepEntry("r", tokens[i][130 * s:130 * s + 130], list(range(0, 130, 3)))]).clone() for s in range(steps)]
        engines[i].free("r")
        return out
    want = [go(0), go(1)]
    torch.cuda.synchronize()
    for _ in range(3):
        got = _together([lambda i=i: go(i) for i in range(2)])
        for i in range(2):
            assert all(torch.equal(a, b) for a, b in zip(got[i], want[i]))
    assert all((e.native_steps > 0) == native for e in engines)
