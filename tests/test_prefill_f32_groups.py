"""Prompt portions in float32 at both sides of every line between one, two and four key groups a block: which one runs is asked of the rule that the
launcher asks, so that none of them goes untested when a line moves."""
import pytest
import torch

LENS = [(0, 2), (0, 31), (0, 129), (130, 65), (257, 160), (31, 97), (5, 128), (700, 33)]          # ten tiles of 128 rows
TILES = sum(-(-n // 128) for _, n in LENS)


def _groups(dh, heads, tiles=TILES):
    from infinicore_infer_amd.kernels.lib import get_lib
    return get_lib().ic_attn_prefill_f32_groups(dh, heads * tiles)


def test_lines_between_the_groups():
    assert TILES == 10
    assert [_groups(64, h) for h in (1, 12, 13, 70, 71, 1000)] == [4, 4, 2, 2, 1, 1]
    assert [_groups(128, h) for h in (1, 40, 41, 1000)] == [2, 2, 1, 1]
    assert _groups(64, 8, 16) == 4 and _groups(64, 129, 1) == 2 and _groups(64, 700, 1) == 2 and _groups(64, 701, 1) == 1
    assert _groups(128, 400, 1) == 2 and _groups(128, 401, 1) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkvh,dh,page,groups", [(1, 1, 64, 16, 4), (12, 4, 64, 64, 4), (13, 13, 64, 32, 2), (70, 10, 64, 32, 2), (71, 71, 64, 64, 1),
                                                    (2, 1, 128, 64, 2), (40, 8, 128, 32, 2), (41, 41, 128, 64, 1)])
@pytest.mark.parametrize("window", [None, 70])
def test_key_groups(nh, nkvh, dh, page, groups, window):
    from test_gpu_kernels import _attention_case, _close
    assert _groups(dh, nh) == groups
    got, want = _attention_case(torch.float32, nh, nkvh, dh, page, LENS, window, 61, "prefill")
    _close(got, want, torch.float32, factor=3)


@pytest.mark.gpu
def test_row_groups_without_work_do_not_crowd_the_others():
    """Heads of 128, one block a unit, two key groups: of portions of two tokens every second block has no rows.  12 portions of 16 heads (192 pairs, 192 blocks with work for 256
    units) take about as long as of 8; with empty and full blocks in turn they took 2.1 times as long, since the full ones met on half the units."""
    from infinicore_infer_amd.kernels import ops
    ps, dh, past, n = 64, 128, 2000, 12
    pages = -(-(past + 2) // ps)
    assert _groups(dh, 16, n) == 2

    def fastest(nh):
        k, v = (torch.randn(n * pages, nh, ps, dh, device="cuda") for _ in range(2))
        q, out = torch.randn(2 * n, 3 * nh * dh, device="cuda"), torch.empty(2 * n, nh * dh, device="cuda")
        table = torch.arange(n * pages, dtype=torch.int32, device="cuda").view(n, pages)
        tiles = torch.tensor([(r, 2 * r, 2, past) for r in range(n)], dtype=torch.int32, device="cuda")
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                ops.attention_prefill(q, out, k, v, table, tiles, n, nh, nh, dh, ps, dh ** -0.5, 0)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    assert fastest(16) < 1.6 * fastest(8)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkvh,dh,lens", [(100, 20, 128, [(0, 2), (0, 33), (31, 34), (62, 2), (63, 130), (0, 65)]), (120, 24, 64, [(0, 2), (0, 33), (31, 34), (62, 2), (63, 130), (0, 65)]),
                                             (90, 30, 128, [(0, 130)] * 2), (3, 3, 128, [(0, 2)] * 88 + [(40, 20)])])
@pytest.mark.parametrize("window", [None, 20])
def test_half_steps_and_rounds(nh, nkvh, dh, lens, window):
    """One group: the last step's second half of keys beyond, at and before a wave's last row.  Two groups of heads of 128: rounds of 3 and of 86 tiles, and what is left."""
    from test_gpu_kernels import _attention_case, _close
    assert _groups(dh, nh, sum(-(-n // 128) for _, n in lens)) == (1 if nh >= 100 else 2)
    got, want = _attention_case(torch.float32, nh, nkvh, dh, 64, lens, window, 61, "prefill")
    _close(got, want, torch.float32, factor=3)
