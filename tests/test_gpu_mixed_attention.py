"""A mixed step's attention in one launch against float64, and the rule that chooses it."""
import pytest
import torch

from infinicore_infer_amd.kernels import ops
from infinicore_infer_amd.kernels.lib import get_lib

BF16 = torch.bfloat16


def test_rule_cpu():
    def rule(dtype=BF16, nh=24, nkv=8, dh=64, ps=64, stride=33, rows=40, tiles=8, pos=1023, window=0, parts=3):
        return ops.rule_attention_together(dtype, nh, nkv, dh, ps, stride, rows, tiles, pos, window, parts, 256)
    assert rule() and rule(nh=36, nkv=36) and rule(nh=32, nkv=2, dh=128, ps=128)
    assert not rule(dtype=torch.float32) and not rule(dh=80) and not rule(ps=32) and not rule(ps=96) and not rule(stride=1025)
    assert not rule(rows=0) and not rule(tiles=0)
    # few tiles with long walks keep their two wave groups; a window makes walks short, many tiles have one group anyway
    assert not rule(parts=1, tiles=6, pos=3199) and rule(parts=1, tiles=6, pos=1000) and rule(parts=1, tiles=6, pos=3199, window=512)
    assert rule(parts=1, tiles=40, pos=3199)


def _packed(lens, starts, page_size=64, nh=32, nkv=2, dh=128):
    """The description of a step of requests with `lens` new tokens from `starts` on, as the C packer lays it out (host code only)."""
    import ctypes
    import numpy as np
    from infinicore_infer_amd.kernels.lib import IcDecoderMeta, IcHostBatch, IcLayer, IcRunEntry, IcStepBatch
    lib, room = get_lib(), ctypes.create_string_buffer(64)
    at = ctypes.addressof(room)
    layer, entry, meta = IcLayer(), IcRunEntry(k_cache=at, v_cache=at, writes_cache=1), IcDecoderMeta()
    a = layer.attention
    a.n_heads, a.n_kv_heads, a.head_dim, a.w_qkv, a.w_o = nh, nkv, dh, at, at
    layer.mixer_norm.weight = layer.ffn_norm.weight = at
    layer.ffn.intermediate, layer.ffn.w_gate_up, layer.ffn.w_down = 128, at, at
    meta.dtype, meta.hidden, meta.vocab, meta.page_size, meta.n_layers, meta.n_entries, meta.n_groups = 1, nh * dh, 64, page_size, 1, 1, 1
    meta.embed_table = meta.head_weight = meta.final_norm.weight = meta.final_norm_scaled = at
    dec = lib.ic_decoder_create(ctypes.byref(meta), ctypes.byref(layer), ctypes.byref(entry))
    assert dec, lib.ic_decoder_create_error()
    try:
        i32 = lambda x: np.asarray(x, dtype=np.int32)
        toks, ln, st, want = i32([1] * sum(lens)), i32(lens), i32(starts), i32([0] * len(lens))
        tables = [i32(range((s + n + page_size - 1) // page_size)) for n, s in zip(lens, starts)]
        ptrs, tlen = (ctypes.c_void_p * len(lens))(*[t.ctypes.data for t in tables]), i32([len(t) for t in tables])
        hb = IcHostBatch(len(toks), len(lens), toks.ctypes.data, ln.ctypes.data, st.ctypes.data, want.ctypes.data, None,
                         ctypes.cast(ptrs, ctypes.c_void_p), tlen.ctypes.data, lib.ic_attn_prefill_tile_rows(), 0)
        n = lib.ic_decoder_step_ints(dec, ctypes.byref(hb))
        staging, out = np.zeros(n, dtype=np.int32), IcStepBatch()
        assert lib.ic_decoder_pack(dec, ctypes.byref(hb), staging.ctypes.data, staging.ctypes.data, n, ctypes.byref(out)) == 0
        return out
    finally:
        lib.ic_decoder_destroy(dec)


def test_long_chats_beside_short_prompts_cpu():
    """How far the prompt tiles walk is told apart from how far the single tokens do: 60 rows of up to 3,000 keys beside portions that
    end at position 699 (32:2 heads of 128) measured 45.1 us apart and 38.9 together."""
    b = _packed([1] * 60 + [600, 200, 50], [3000 - 40 * i for i in range(60)] + [100, 0, 0])
    assert (b.n_decode_rows, b.n_prefill_tiles, b.max_position, b.max_tile_position) == (60, 8, 3000, 699)
    parts, _ = ops.attention_prefill_parts_of_step(BF16, b.n_prefill_tiles, 32, 128, b.max_tile_position, 0, 256)
    together = lambda end: ops.rule_attention_together(BF16, 32, 2, 128, 64, 47, b.n_decode_rows, b.n_prefill_tiles, end, 0, parts, 256)
    assert parts == 1 and together(b.max_tile_position) and not together(b.max_position)
    assert _packed([1, 1], [5, 700]).max_tile_position == 0
    # a walk that the tiles alone leave whole is cut in two here from 12 key tiles on, while the blocks are few enough for it
    cut = lambda nh, dh, tiles, end, entry=ops.attention_mixed_parts_of_step: entry(BF16, tiles, nh, dh, end, 0, 256)
    alone = ops.attention_prefill_parts_of_step
    assert cut(24, 64, 8, 1023, alone)[0] == 1 and cut(24, 64, 8, 1023) == (2, 11) and cut(32, 128, 10, 767) == (2, 11) and cut(32, 128, 10, 2047) == (2, 16)
    assert cut(24, 64, 8, 703) == cut(24, 64, 8, 703, alone) == (1, 11) and cut(32, 128, 11, 1023)[0] == 1
    assert cut(24, 64, 4, 1023) == cut(24, 64, 4, 1023, alone) and cut(24, 64, 4, 1023)[0] == 3
    assert _packed([300, 1], [2000, 7]).max_tile_position == 2299


def _case(nh, nkv, dh, ps, held, portions, window, n_split, parts, part_len):
    g = torch.Generator().manual_seed(nh + dh + len(held))
    lens = [p + 1 for p in held] + [a + b for a, b in portions]
    pages = [-(-n // ps) for n in lens]
    ids = torch.randperm(sum(pages), generator=g).tolist()
    bt = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    for r, n in enumerate(pages):
        bt[r, :n] = torch.tensor(ids[:n], dtype=torch.int32)
        ids = ids[n:]
    pos, req, tiles, row = list(held), list(range(len(held))), [], len(held)
    for i, (a, b) in enumerate(portions):
        tiles += [(len(held) + i, row + o, min(128, b - o), a + o) for o in range(0, b, 128)]
        pos += range(a, a + b)
        req += [len(held) + i] * b
        row += b
    rnd = lambda *s: torch.randn(*s, generator=g).to(BF16)
    q, k, v = rnd(row, (nh + 2 * nkv) * dh), rnd(sum(pages), nkv, ps, dh), rnd(sum(pages), nkv, ps, dh)
    scale = dh ** -0.5
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    dev = dict(q=q.cuda(), k=k.cuda(), v=v.cuda(), bt=bt.cuda(), pos=i32(pos), req=i32(req), tl=i32(tiles).view(-1, 4),
               rows=i32(sorted(range(len(held)), key=lambda i: -held[i])))
    n = len(held)
    acc = torch.empty(n * nh * n_split * dh, device="cuda")
    ml = torch.empty(n * nh * n_split * 2, device="cuda")
    scratch = torch.empty(max(4, ops.attention_prefill_scratch_floats(len(tiles), nh, dh, parts)), device="cuda")
    counters = torch.zeros(ops.attention_prefill_counter_ints(), dtype=torch.int32, device="cuda")
    args, cut = (nh, nkv, dh, ps, scale, window), dict(parts=parts, part_len=part_len, scratch=scratch, counters=counters)
    out = torch.full((row, nh * dh), 3.0, dtype=BF16, device="cuda")
    single = (dev["rows"], n, dev["req"], dev["pos"], acc, ml)
    for _ in range(2):                          # twice: the counters are back at zero
        ops.attention_mixed(dev["q"], out, dev["k"], dev["v"], dev["bt"], *single, n_split, dev["tl"], len(tiles), *args, **cut)
    assert (counters == 0).all()
    got = out.cpu().double().view(row, nh, dh)
    q, k, v = q.double(), k.double(), v.double()
    for t in list(range(n)) + list(range(n, row, 37)) + [row - 1]:
        p, r = pos[t], req[t]
        keys = torch.arange(max(0, p - window + 1) if window else 0, p + 1)
        pg, at = bt[r].long()[keys // ps], keys % ps
        for h in range(nh):
            kv = h // (nh // nkv)
            s = (k[pg, kv, at] @ q[t, h * dh:(h + 1) * dh]) * scale
            w = s.softmax(0)
            want, size = w @ v[pg, kv, at], w @ v[pg, kv, at].abs()
            # probabilities and the result rounded to bfloat16 (2^-9 each), scores of float32 sums
            assert ((got[t, h] - want).abs() - size * 2.0 ** -7 - 1e-6).max() <= 0, (t, h)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,dh", [(6, 2, 64), (3, 3, 64), (4, 1, 128), (2, 2, 128), (20, 1, 64)])
@pytest.mark.parametrize("ps", [64, 256])
def test_mixed_against_float64(nh, nkv, dh, ps):
    _case(nh, nkv, dh, ps, [0], [(0, 2)], 0, 1, 1, 0)                                   # the smallest step
    _case(nh, nkv, dh, ps, [3, 700, 64, 63], [(0, 130), (300, 257)], 0, 1, 1, 0)
    _case(nh, nkv, dh, ps, [500, 129, 1], [(700, 140), (0, 5)], 0, 3, 3, 4)             # splits and cut walks
    _case(nh, nkv, dh, ps, [500, 129, 1], [(700, 140), (0, 5)], 100, 2, 1, 0)           # a window


@pytest.mark.gpu
def test_refused_arguments():
    lib = get_lib()
    x = torch.zeros(1 << 12, device="cuda")
    p = x.data_ptr()
    good = dict(q=p, qs=512, out=p, os=256, dt=1, k=p, v=p, bt=p, bts=4, rows=p, req=p, pos=p, acc=p, ml=p, n=1, ns=1, tl=p, nt=1, nh=4, nkv=4, dh=64,
                ps=64, scale=0.1, window=0, parts=1, plen=0, scratch=None, nf=0, cnt=None, stream=0)
    for bad, status in ((dict(dt=0), -2), (dict(dh=80), -2), (dict(ps=32), -2), (dict(bts=2000), -2), (dict(rows=None), -1), (dict(n=0), -1),
                        (dict(nt=0), -1), (dict(ns=65), -1), (dict(q=p + 2), -1), (dict(parts=2, plen=4), -1), (dict(ns=2, acc=None), -1)):
        assert lib.ic_attn_mixed(*dict(good, **bad).values()) == status, bad


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_both_step_paths_ask_with_the_portions_end(native, tmp_path_factory, monkeypatch):
    import helpers as H
    from infinicore_infer_amd.engine import Engine, StepEntry
    folder = H.make_model_dir(tmp_path_factory.getbasetemp(), "C")
    eng = Engine.from_dir(folder, dtype=BF16, max_tokens=1024, page_size=64, max_requests=4, use_native=native)
    vocab = H.CONFIGS["C"][0]["vocab_size"]
    eng.step([StepEntry("a", H.random_tokens(vocab, 400, 1), [399])])
    seen = []
    build = Engine._build_context
    monkeypatch.setattr(Engine, "_build_context", lambda self, *a: seen.append(build(self, *a)) or seen[-1])
    rule = ops.rule_attention_together
    asked = []
    monkeypatch.setattr(ops, "rule_attention_together", lambda *a: asked.append(a[8]) or rule(*a))
    eng.step([StepEntry("a", [5], [0]), StepEntry("b", H.random_tokens(vocab, 70, 2), [69])])
    if native:
        assert eng.native is not None and (eng.native._batch.max_position, eng.native._batch.max_tile_position) == (400, 69)
    else:
        assert seen[-1].max_position == 400 and seen[-1].max_tile_position == 69 and asked and set(asked) == {69}
