"""Which decoders and steps run all layers in one launch (decode_chain.hip), and the table that this takes: host code alone, on pointers that nothing follows."""
import ctypes

import numpy as np
import pytest

from infinicore_infer_amd.kernels.lib import IcDecoderMeta, IcLayer, IcRunEntry, IcStepBatch, get_lib

FIELDS = ("w_qkv", "w_o", "w_gate_up", "w_down", "norm_in", "norm_mid", "k_cache", "v_cache")


class Decoder:
    """Layers of one size; the pointers of layer i count on from 1 << 20 times i + 1."""

    def __init__(self, layers=4, hidden=1536, heads=24, kv=8, inner=3840, dim=64, page=64, units=256, change=None):
        self.lib, self.n = get_lib(), layers
        at = lambda i, k: (i + 1 << 20) + 4096 * k
        self.want = [[at(i, k) for k in range(8)] for i in range(layers)] + [[0, 0, 0, 0, 4096, 0, 0, 0]]
        arr, runs, meta = (IcLayer * layers)(), (IcRunEntry * layers)(), IcDecoderMeta()
        for i in range(layers):
            l, a = arr[i], arr[i].attention
            a.n_heads, a.n_kv_heads, a.head_dim, a.rot_dim, a.max_positions, a.softmax_scale, a.cos, a.sin = heads, kv, dim, dim, 4096, 0.125, 256, 512
            a.w_qkv, a.w_o, l.ffn.w_gate_up, l.ffn.w_down, l.mixer_norm.weight, l.ffn_norm.weight = self.want[i][:6]
            l.mixer_norm.eps = l.ffn_norm.eps = 1e-5
            l.ffn.intermediate, l.residual_scale = inner, 0.2
            runs[i] = IcRunEntry(i, 1, 0, *self.want[i][6:])
        meta.dtype, meta.hidden, meta.vocab, meta.page_size, meta.n_layers, meta.n_entries, meta.n_groups, meta.compute_units = 1, hidden, 2003, page, layers, layers, 1, units
        meta.embed_table, meta.head_weight, meta.final_norm.weight, meta.final_norm_scaled = 1024, 1024, 2048, 4096
        if change:
            change(meta, arr, runs)
        self.h = self.lib.ic_decoder_create(ctypes.byref(meta), arr, runs)
        assert self.h, self.lib.ic_decoder_create_error()
        self.h = ctypes.c_void_p(self.h)

    def __enter__(self):
        return self

    def __exit__(self, *_):
        self.lib.ic_decoder_destroy(self.h)

    def table(self):
        host = np.full(self.lib.ic_decoder_table_bytes(self.n) // 8, -1, dtype=np.int64)
        return host.reshape(-1, 8).tolist() if self.lib.ic_decoder_layer_table(self.h, host.ctypes.data) == 1 else None

    def use(self):
        return self.lib.ic_decoder_use_layer_table(self.h, 1 << 16, None)

    def step(self, rows=1, keys=258):
        b = IcStepBatch()
        b.n_tokens = b.n_requests = b.n_want = b.n_decode_rows = rows
        b.want_rows_identity = b.decode_rows_identity = 1
        b.max_position, b.max_context = keys - 1, keys
        return b

    def takes(self, rows=1, keys=258, **fields):
        b = self.step(rows, keys)
        for k, v in fields.items():
            setattr(b, k, v)
        return bool(self.lib.ic_decoder_takes_chain(self.h, ctypes.byref(b)))


def test_the_table_is_made_without_the_device():
    """Making a decoder writes nothing to the device (the table was copied there on a stream of its own, which nothing ordered with the caller's fill of the same
    memory): its bytes are handed out, and steps use them only once the caller says that they are on the device."""
    with Decoder() as d:
        assert d.table() == d.want
        assert not d.takes()
        before = d.lib.ic_decoder_workspace_bytes(d.h, ctypes.byref(d.step()))
        assert d.lib.ic_decoder_use_layer_table(d.h, (1 << 16) + 4, None) != 0 and not d.takes()
        assert d.use() == 0 and d.takes()
        assert d.lib.ic_decoder_workspace_bytes(d.h, ctypes.byref(d.step())) > before
        assert d.lib.ic_decoder_use_layer_table(d.h, None, None) == 0 and not d.takes()


def _set(path, value, at=1):
    def change(meta, layers, runs):
        o = {"meta": meta, "layer": layers[at], "run": runs[at]}[path[0]]
        for name in path[1:-1]:
            o = getattr(o, name)
        setattr(o, path[-1], value)
    return change


@pytest.mark.parametrize("change", [_set(("meta", "dtype"), 0), _set(("layer", "attention", "window"), 512), _set(("layer", "attention", "shared_kv"), 1), _set(("run", "writes_cache"), 0),
                                    _set(("layer", "attention", "n_kv_heads"), 4), _set(("layer", "ffn", "intermediate"), 3904), _set(("layer", "residual_scale"), 0.3),
                                    _set(("layer", "attention", "rot_dim"), 32), _set(("layer", "attention", "cos"), 768), _set(("layer", "ffn_norm", "eps"), 1e-6),
                                    _set(("run", "k_cache"), (1 << 20) + 6 * 4096), _set(("layer", "attention", "w_o"), (2 << 20) + 4096 + 8)])
def test_layers_that_are_not_alike_have_no_table(change):
    with Decoder(change=change) as d:
        assert d.table() is None and d.use() != 0 and not d.takes()


def test_steps_that_run_kernel_by_kernel():
    with Decoder() as d:
        assert d.use() == 0 and d.takes(4)
        assert not d.takes(9) and not d.takes(4, fixed_decode_splits=2) and not d.takes(4, n_want=3) and not d.takes(4, want_rows_identity=0)
        assert not d.takes(4, decode_rows_identity=0) and not d.takes(4, n_decode_rows=3, n_prefill_tiles=1)


@pytest.mark.parametrize("hidden,heads,kv,inner,units,taken", [(2496, 64, 16, 6144, 304, False), (2496, 64, 16, 6144, 256, True), (1216, 24, 8, 3840, 304, False), (1216, 24, 8, 3840, 256, True),
                                                                  (1536, 24, 8, 3840, 304, True)])
def test_more_sums_of_squares_than_the_head_product_takes(hidden, heads, kv, inner, units, taken):
    """A row has a sum for every block's columns of the stream; the product behind the chain takes 256 of them."""
    blocks = -(-hidden // -(-hidden // units))
    with Decoder(hidden=hidden, heads=heads, kv=kv, inner=inner, units=units) as d:
        assert taken == (blocks <= d.lib.ic_rule_sumsq_parts_max())
        assert (d.use() == 0) == taken and d.takes() == taken


def test_rotary_tables_that_are_not_aligned():
    """The QKV product refuses them in a step of few rows, so the one launch does not take them."""
    def change(meta, layers, runs):
        for l in layers:
            l.attention.sin += 8
    with Decoder(change=change) as d:
        assert d.table() is None and d.use() != 0 and not d.takes()


@pytest.mark.parametrize("page,taken", [(1 << 20, True), ((1 << 22) - 1, True), (1 << 22, False), (1 << 24, False)])
def test_pages_beyond_32_bits(page, taken):
    """8 kv heads of 64 in bfloat16: a page of 2^22 keys has 2^32 bytes."""
    with Decoder(page=page) as d:
        assert (d.use() == 0) == taken and d.takes() == taken


def test_workspaces_that_are_not_aligned():
    """The one launch hands values on in pieces of 8 and 16 bytes; kernel by kernel the attention refuses such a step."""
    with Decoder() as d:
        at = lambda p: bool(d.lib.ic_decoder_takes_chain_at(d.h, ctypes.byref(d.step()), p))
        assert not at(1 << 20) and d.use() == 0
        assert at(1 << 20) and at((1 << 20) + 16) and not at((1 << 20) + 4) and not at((1 << 20) + 8)


@pytest.mark.parametrize("hidden,heads,kv,inner,most", [(1536, 24, 8, 3840, 8), (2048, 32, 16, 4096, 8), (1088, 16, 4, 2176, 8), (2304, 36, 36, 5760, 7), (2112, 64, 32, 6144, 7),
                                                        (3072, 48, 16, 4352, 5), (2304, 64, 16, 6080, 5)])
def test_rows_up_to_which_one_launch_is_faster(hidden, heads, kv, inner, most):
    with Decoder(hidden=hidden, heads=heads, kv=kv, inner=inner) as d:
        assert d.use() == 0
        assert [d.takes(rows, 600) for rows in range(1, 10)] == [rows <= most for rows in range(1, 10)]
