"""The order in which a step of single tokens starts its rows: longest first, and the same logits as in the rows' own order."""
import os

import pytest
import torch

import helpers as H
from test_gpu_native import _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 1024])
@pytest.mark.parametrize("values", [5, 100000])                       # many equal positions, and few
def test_rows_by_length(n, values):
    from infinicore_infer_amd.kernels import ops
    from infinicore_infer_amd.kernels.lib import get_lib
    pos = torch.randint(0, values, (n,), generator=torch.Generator().manual_seed(n), dtype=torch.int32).cuda()
    order = torch.full((n + 1,), -7, dtype=torch.int32).cuda()
    assert get_lib().ic_attn_decode_order(pos.data_ptr(), order.data_ptr(), n, ops.current_stream()) == 0
    assert order[:n].tolist() == torch.argsort(pos, descending=True, stable=True).tolist() and int(order[n]) == -7


def test_more_rows_than_an_order_holds_are_refused():
    from infinicore_infer_amd.kernels.lib import get_lib
    pos = torch.zeros(1025, dtype=torch.int32).cuda()
    assert get_lib().ic_attn_decode_order(pos.data_ptr(), pos.data_ptr(), 1025, None) != 0


@pytest.mark.parametrize("graphs", [False, True])
def test_steps_of_ordered_rows(tmp_path_factory, graphs):
    """Two layers of 36 heads, 7 rows (252 blocks, at most one a compute unit) and 20 rows (720) of ragged lengths: native steps, which
    order their rows, against steps issued from Python, which do not; eager and, with every position moved on, replayed."""
    from infinicore_infer_amd.engine import StepEntry
    from infinicore_infer_amd.weights import write_random_model
    cfg = dict(model_type="minicpm", vocab_size=5003, hidden_size=2304, num_hidden_layers=2, num_attention_heads=36,
               num_key_value_heads=36, intermediate_size=5760, max_position_embeddings=512, rms_norm_eps=1e-5,
               rope_theta=10000.0, scale_emb=12, dim_model_base=256, scale_depth=1.4, tie_word_embeddings=True,
               eos_token_id=2)
    folder = os.path.join(str(tmp_path_factory.getbasetemp()), "model_decode_order")
    write_random_model(folder, cfg, seed=3, std=0.02)
    a, b = _pair(folder, torch.bfloat16, 24 * 512, page_size=64, max_requests=24, use_graphs=graphs)
    ids = ["q%d" % i for i in range(20)]
    for eng in (a, b):
        eng.step([StepEntry(r, H.random_tokens(5003, 2 + (37 * i) % 200, i), []) for i, r in enumerate(ids)])
    for n in (7, 20):
        for j in range(4):
            ents = [StepEntry(r, [7 + i + j], [0]) for i, r in enumerate(ids[:n])]
            assert torch.equal(a.step(ents), b.step(ents)), (n, j)
    if graphs:
        assert a.graph_replays == b.graph_replays > 0
