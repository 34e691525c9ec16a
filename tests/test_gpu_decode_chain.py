"""Decode steps whose layers run in one launch (decode_chain.hip): against the plain implementation and the same steps kernel by kernel, over row counts and lengths at
the edges of what is dealt to the blocks; recorded and eager steps, steps with fewer blocks than compute units and steps of two streams at once, to the bit."""
import threading

import pytest
import torch

import helpers as H
from test_gpu_large import SHAPE_1B, SHAPE_2B, _engine_and_weights

pytestmark = pytest.mark.gpu

LAYERS = 4
SHAPES = {"1b": dict(SHAPE_1B, vocab_size=2003, num_hidden_layers=LAYERS, max_position_embeddings=4096),
          "2b": dict(SHAPE_2B, vocab_size=2003, num_hidden_layers=LAYERS)}


# (hidden, heads, kv heads, inner): groups of 1..4 in both of the kernel's sizes, with the least and the most columns of a block, and rows of which waves have unlike shares
OTHERS = [(1536, 12, 12, 2112), (2048, 32, 16, 4096), (1024, 15, 5, 2752), (1088, 16, 4, 2176), (4096, 40, 40, 4160), (2112, 64, 32, 6144), (3072, 48, 16, 4352), (2304, 64, 16, 6080)]
for _d, _h, _kv, _di in OTHERS:
    SHAPES["%d-%d-%d-%d" % (_d, _h, _kv, _di)] = dict(SHAPE_1B, vocab_size=2003, num_hidden_layers=3, hidden_size=_d, num_attention_heads=_h, num_key_value_heads=_kv,
                                                      head_dim=64, intermediate_size=_di)


def _engine(shape, **kw):
    return _engine_and_weights(SHAPES[shape], 21, 0.02, 16 * 2304, 12, **kw)


def _chained(engine):
    return bool(engine.native._lib.ic_decoder_takes_chain(engine.native._h, engine.native._batch_ref))


def _hold(engine, doc, lens):
    from infinicore_infer_amd.engine import StepEntry
    engine.step([StepEntry("doc", doc, [])])
    for i, n in enumerate(lens):
        engine.fork("doc", "r%d" % i, n)
    engine.free("doc")


def _decode(engine, tokens):
    from infinicore_infer_amd.engine import StepEntry
    return engine.step([StepEntry("r%d" % i, [t], [0]) for i, t in enumerate(tokens)]).clone()


def _drop(engine, n):
    for i in range(n):
        engine.free("r%d" % i)


LENS = [[1], [62], [63], [64], [257], [320], [384], [600], [1100], [2063], [1, 300], [64, 63, 65], [900, 20], [400, 300, 200, 100], [2000, 1, 1, 1],
        [700, 3, 1290, 40, 511], [1500] * 6, [2000, 1000, 500, 250, 125, 60, 30], [1] * 8, [2250, 1, 2, 3, 4, 5, 6, 7]]


@pytest.mark.parametrize("page_size", [16, 64])
@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_rows_and_lengths(shape, page_size):
    """Each path rounds to bfloat16 some ten times a layer and is 1e-2 off the plain implementation at most (checked below); two of them differ by twice that."""
    a, _ = _engine(shape, page_size=page_size, use_graphs=False)
    b, _ = _engine(shape, page_size=page_size, use_native=False)
    doc = H.random_tokens(2003, 2260, 4)
    taken = 0
    for k, lens in enumerate(LENS):
        for e in (a, b):
            _hold(e, doc, lens)
        for j in range(3):
            toks = H.random_tokens(2003, len(lens), 100 * k + j)
            la, lb = _decode(a, toks), _decode(b, toks)
            taken += _chained(a)
            err = float((la - lb).norm() / lb.norm())
            assert err < 2e-2, (shape, lens, j, err)
        for e in (a, b):
            _drop(e, len(lens))
    assert taken == 3 * sum(len(lens) <= (7 if shape == "2b" else 8) for lens in LENS)      # (more rows of the wide shape are faster kernel by kernel)


@pytest.mark.parametrize("shape", ["%d-%d-%d-%d" % o for o in OTHERS])
def test_other_sizes(shape):
    a, _ = _engine(shape, use_graphs=False)
    b, _ = _engine(shape, use_native=False)
    doc = H.random_tokens(2003, 1300, 4)
    for k, lens in enumerate([[1], [257], [600, 40], [1200, 1, 64, 700]]):
        for e in (a, b):
            _hold(e, doc, lens)
        for j in range(2):
            toks = H.random_tokens(2003, len(lens), 100 * k + j)
            la, lb = _decode(a, toks), _decode(b, toks)
            err = float((la - lb).norm() / lb.norm())
            assert _chained(a) and err < 2e-2, (shape, lens, j, err)
        for e in (a, b):
            _drop(e, len(lens))


@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_against_the_plain_implementation(shape):
    from plain_model import plain_forward, round_bf16
    engine, sd = _engine(shape, use_graphs=False)
    doc = H.random_tokens(2003, 700, 8)
    lens, steps = [650, 63, 257], 3
    _hold(engine, doc, lens)
    new = [H.random_tokens(2003, len(lens), 50 + j) for j in range(steps)]
    got = []
    for j in range(steps):
        got.append(_decode(engine, new[j]))
        assert _chained(engine)
    for i, n in enumerate(lens):
        tokens = doc[:n] + [new[j][i] for j in range(steps)]
        want = plain_forward(SHAPES[shape], sd, tokens, rnd=round_bf16, rows=list(range(n, n + steps))).cpu()
        have = torch.stack([got[j][i] for j in range(steps)]).double().cpu()
        err = float((have - want).abs().max() / want.abs().max())
        assert err < H.BF16_TOL, (shape, n, err)


@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_recorded_and_eager_steps_are_equal(shape):
    """Several replays with the engine's own eager work between them; lengths cross the border of a unit of keys and of a recorded step's range."""
    from infinicore_infer_amd.engine import StepEntry
    a, _ = _engine(shape, graph_after=1)
    b, _ = _engine(shape, use_graphs=False)
    doc = H.random_tokens(2003, 700, 9)
    for e in (a, b):
        _hold(e, doc, [254, 61, 640])
    for j in range(8):
        toks = H.random_tokens(2003, 3, 70 + j)
        la, lb = _decode(a, toks), _decode(b, toks)
        assert _chained(b) and torch.equal(la, lb), j
        if j % 3 == 2:
            for e in (a, b):
                e.step([StepEntry("other", H.random_tokens(2003, 40, j), [])])
                e.free("other")
            torch.cuda.synchronize()
    assert a.graph_replays >= 5


@pytest.mark.parametrize("absent", [1, 100, 240])
@pytest.mark.parametrize("lens", [[257], [600, 40], [1500] * 3])
@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_blocks_that_find_no_room(shape, lens, absent):
    """The others do their work, with the same results to the bit."""
    a, _ = _engine(shape, use_graphs=False)
    b, _ = _engine(shape, use_graphs=False)
    forward = a.native._lib.ic_decoder_forward_absent
    doc = H.random_tokens(2003, 1600, 3)
    for e in (a, b):
        _hold(e, doc, lens)
    a.native._forward = lambda *args: forward(*args[:-1], absent, args[-1])
    for j in range(2):
        toks = H.random_tokens(2003, len(lens), 30 + j)
        la, lb = _decode(a, toks), _decode(b, toks)
        assert _chained(a) and torch.equal(la, lb), (shape, lens, absent, j)


def test_two_streams_at_once():
    """Two engines decode on streams of their own at the same time: neither keeps the other from ending, and each has the logits that it has alone."""
    engines = [_engine("1b")[0], _engine("1b", graph_after=1)[0]]
    doc = H.random_tokens(2003, 700, 5)
    toks = [H.random_tokens(2003, 2, 10 + j) for j in range(12)]

    def hold():
        for e in engines:
            _hold(e, doc, [600, 257])
        torch.cuda.synchronize()

    def go(i):
        out = [_decode(engines[i], t) for t in toks]
        torch.cuda.current_stream().synchronize()
        _drop(engines[i], 2)
        return out
    hold()
    want = [go(0), go(1)]
    assert all(torch.equal(x, y) for x, y in zip(*want))
    for _ in range(3):
        hold()
        got, wrong, start = [None, None], [], threading.Barrier(2)

        def run(i):
            try:
                with torch.cuda.stream(torch.cuda.Stream()):
                    start.wait()
                    got[i] = go(i)
            except BaseException as e:
                wrong.append(e)
        threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, wrong
        bad = [(i, j) for i in range(2) for j in range(len(toks)) if not torch.equal(got[i][j], want[i][j])]
        assert not bad, bad


def test_weights_that_are_not_numbers():
    """A NaN of that pattern in an embedding row makes the logits of its request NaN (and ends: what is handed on is never what stands for "not there yet"), the others' stay."""
    engine, _ = _engine("1b", use_graphs=False)
    doc = [t for t in H.random_tokens(2003, 300, 6) if t != 5]
    _hold(engine, doc, [200, 100])
    want = _decode(engine, [7, 9])
    _drop(engine, 2)
    table = engine.model.embedding.table
    row = table[5].clone()
    table[5].view(torch.int16).fill_(-1)                     # all ones: a NaN whose bits stand for "not there yet"
    _hold(engine, doc, [200, 100])
    got = _decode(engine, [7, 5])
    table[5].copy_(row)
    got[0, 5] = want[0, 5]                                   # (the table is the head's too)
    assert _chained(engine) and torch.equal(got[0], want[0]) and bool(got[1].isnan().all())


def test_the_table_of_an_engine_made_on_a_stream_of_its_own():
    """Work is queued on that stream when the table is handed over: it holds the layers' addresses all the same (looked at, not run)."""
    from infinicore_infer_amd.engine.native import NativeDecoder
    engine, _ = _engine("1b")
    lib = engine.native._lib
    host = torch.empty(lib.ic_decoder_table_bytes(LAYERS), dtype=torch.uint8)
    assert lib.ic_decoder_layer_table(engine.native._h, host.data_ptr()) == 1
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(40):
            a = a @ a
            a /= a.norm()
        made = NativeDecoder.try_build(engine)
    stream.synchronize()
    own = torch.empty_like(host)                             # (the scaled final norm is this decoder's own)
    assert lib.ic_decoder_layer_table(made._h, own.data_ptr()) == 1
    assert torch.equal(own[:-64], host[:-64]) and torch.equal(made._layer_table.cpu(), own)


@pytest.mark.parametrize("lens", [[1024], [64], [1024, 320, 640]])
@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_pieces_whose_scores_are_all_minus_infinity(shape, lens):
    """Keys of weight 0 beside others, in pieces of their own among others: whether their scores are -inf or finite and far below is one to the bit.  The step's own key (a
    unit of its own: the lengths are multiples of 64) and the last unit's cached ones, in the first layer: its keys are minus its queries, times 4e37 and 1e10."""
    engine, _ = _engine(shape, use_graphs=False)
    doc, toks = H.random_tokens(2003, 1100, 4), H.random_tokens(2003, len(lens), 9)
    mixer = engine.model.layers[0].mixer
    w, nh, nkv = mixer.w_qkv, mixer.nh, mixer.nkvh
    keep = w.clone()
    out = []
    for size in (4e37, 1e10):
        w.copy_(keep)
        _hold(engine, doc, lens)
        q = w[:nh * 64].view(nkv, nh // nkv, 64, -1)
        q.copy_(q[:, :1].clone().expand_as(q))               # a group's heads alike
        w[nh * 64:(nh + nkv) * 64].view(nkv, 64, -1).copy_(q[:, 0].float() * -size)
        _decode(engine, toks)
        keys = engine.storage.kv(0)[0]                       # [page, kv head, place, 64]
        for i, n in enumerate(lens):
            page = lambda p: engine.cache.block_table("r%d" % i, 0)[p // 64]
            own = keys[page(n), :, n % 64].clone()
            assert n % 64 == 0 and bool(own.isfinite().all())
            if n > 64:
                keys[page(n - 64)] = own[:, None]
            engine.cache.truncate("r%d" % i, n)
        out.append(_decode(engine, toks))
        assert _chained(engine)
        _drop(engine, len(lens))
    assert bool(out[1].isfinite().all()) and torch.equal(*out)


@pytest.mark.parametrize("lens", [[1100], [700, 3, 1290]])
@pytest.mark.parametrize("shape", ["1b", "2b"])
def test_waits_that_are_given_up(shape, lens):
    """No question is asked twice, so that most blocks give up at their first wait: the step ends, sampling its tokens raises, the cache holds nothing that came of it (what
    the first layers wrote is right), and later steps are as ever."""
    from infinicore_infer_amd.kernels.lib import KernelError
    engine, _ = _engine(shape, use_graphs=False)
    toks, doc = H.random_tokens(2003, len(lens), 7), H.random_tokens(2003, 1400, 3)
    planes = [plane.zero_() for s in range(LAYERS) for plane in engine.storage.kv(s)]        # (pages that nobody holds have what the memory held)
    _hold(engine, doc, lens)
    want = _decode(engine, toks)
    back = lambda: [engine.cache.truncate("r%d" % i, n) for i, n in enumerate(lens)]
    back()
    forward, usual = engine.native._lib.ic_decoder_forward_tries, engine.native._forward
    for sample in (engine.sample, lambda logits: engine.sample_ahead(logits)[1](), lambda logits: (torch.cuda.synchronize(), _decode(engine, toks))):
        engine.native._forward = lambda *args: forward(*args[:-1], 0, args[-1])
        got = _decode(engine, toks)
        engine.native._forward = usual
        assert _chained(engine) and bool(got.isnan().all())
        with pytest.raises(KernelError, match="gave up"):
            sample(got)
        assert all(bool(plane.isfinite().all()) for plane in planes)
        back()
        assert torch.equal(_decode(engine, toks), want)
        engine.sample(got)                                   # (told once)
        back()


@pytest.mark.parametrize("native", [True, False])
def test_steps_ahead_of_rows_that_sampled_no_token(native):
    """Logits of NaN sample what is no token of the vocabulary.  A step that takes it from the device looks up the last one (whose logits nobody wants) and nothing beyond."""
    from infinicore_infer_amd.engine import StepEntry
    engine, _ = _engine("1b", graph_after=1, use_native=native)
    doc, V = H.random_tokens(2003, 90, 3), 2003
    _hold(engine, doc, [70, 50])
    nan = torch.full((2, V), float("nan"), device="cuda")
    sampled, wait = engine.sample_ahead(nan)
    assert all(not 0 <= t < V for t in wait())
    ents = [StepEntry("r%d" % i, [0], [0]) for i in range(2)]
    want = engine.step([StepEntry("r%d" % i, [V - 1], [0]) for i in range(2)]).clone()      # recorded here
    for i, n in enumerate([70, 50]):
        engine.cache.truncate("r%d" % i, n)
    got = engine.step_ahead(ents, sampled)
    assert got is not None and torch.equal(got, want)


@pytest.mark.parametrize("absent,rounds", [(1, 1), (100, 1), (192, 3), (240, 15)])
def test_how_long_blocks_wait_for_others(absent, rounds):
    """A round of the tasks beyond the first costs a step's time; blocks wait that long (a millisecond at least) for those that would spare it, before they begin without."""
    engine, _ = _engine("1b", use_graphs=False)
    _hold(engine, H.random_tokens(2003, 300, 3), [257])
    forward = engine.native._lib.ic_decoder_forward_absent
    engine.native._forward = lambda *args: forward(*args[:-1], absent, args[-1])
    if engine.cu_count != 256:
        pytest.skip("rounds are counted for 256 units")
    took = []
    for j in range(4):
        events = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda.synchronize()
        events[0].record()
        _decode(engine, [5])
        events[1].record()
        torch.cuda.synchronize()
        took.append(events[0].elapsed_time(events[1]))
    assert _chained(engine) and rounds * 0.999 < min(took[1:]) < rounds * 1.0 + 5.0, took       # (ms; the clock is 100 MHz, the step itself under 3 ms with 16 blocks)


def test_steps_issued_before_one_was_found_without_results():
    """While the host has not seen a step's tokens, the step after it is under way from them: it is refused too, and so is one that would go on from it; then the flag (set here by the
    host, as the device does) is forgotten."""
    from infinicore_infer_amd.engine import StepEntry
    from infinicore_infer_amd.kernels.lib import KernelError
    engine, _ = _engine("1b", graph_after=1)
    _hold(engine, H.random_tokens(2003, 90, 3), [70, 50])
    ents = [StepEntry("r%d" % i, [0], [0]) for i in range(2)]
    engine.sample(_decode(engine, [5, 6]))                   # recorded
    first, wait_first = engine.sample_ahead(_decode(engine, [7, 8]))
    second, wait_second = engine.sample_ahead(engine.step_ahead(ents, first))
    assert _chained(engine)
    torch.cuda.synchronize()
    engine.native._gave_up[0] = 1
    held = engine.length("r0")
    for refused in (wait_first, wait_second, lambda: engine.step_ahead(ents, second)):
        with pytest.raises(KernelError, match="gave up|without results"):
            refused()
    assert engine.length("r0") == held and engine.native._gave_up[0] == 0
    logits = engine.step([StepEntry("r0", [3], [0])])
    assert len(engine.sample(logits)) == 1
