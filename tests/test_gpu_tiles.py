"""The product of many rows in tiles: every tile at its edges, plain and with SwiGLU, and the choice between it and the library."""
import pytest
import torch

from infinicore_infer_amd.kernels import ops

BF16 = torch.bfloat16
TILES = ((64, 32), (64, 64), (64, 96), (128, 64), (64, 128), (96, 128), (128, 128), (192, 128), (128, 192), (160, 192), (256, 128), (128, 256), (160, 256),
         (256, 192), (256, 256))


def _operands(M, N, K, seed, pad=0):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K + pad, generator=g).to(BF16)[:, :K]
    w = (torch.randn(N, K + pad, generator=g) * K ** -0.5).to(BF16)[:, :K]
    return a, w


def _strided(t, pad):
    d = torch.empty(t.shape[0], t.shape[1] + pad, dtype=t.dtype, device="cuda")[:, :t.shape[1]]
    return d.copy_(t)


def _check(a, w, got, swiglu):
    """Element by element: the result's rounding to bfloat16 (2^-8 of it) and float32 sums of K products in any order (each partial sum
    rounds by 2^-24 of at most the sum of the products' magnitudes; K of them, of which the roundings of random sign leave far less than 2^-6)."""
    a, w = a.double(), w.double()
    ref, mag = a @ w.t(), (a.abs() @ w.abs().t()) * a.shape[1] * 2.0 ** -24
    if swiglu:
        n = ref.shape[1] // 2
        g, u, mg, mu = ref[:, :n], ref[:, n:], mag[:, :n], mag[:, n:]
        s = torch.nn.functional.silu(g)
        # |silu'| <= 1.1; exp2 and reciprocal of the hardware: an ulp each
        ref, mag = u * s, 1.1 * mg * (u.abs() + mu) + mu * s.abs() + 2.0 ** -21 * (u * s).abs()
    assert torch.isfinite(got).all()
    err = (got.double().cpu() - ref).abs() - ref.abs() * 2.0 ** -8 - mag
    assert err.max() <= 0, "off by %.3g beyond the bound" % err.max()


def test_tile_rule_cpu():
    """Every choice names a tile; what the kernel cannot take is refused; up to 32 rows other kernels run."""
    from infinicore_infer_amd.kernels.lib import get_lib
    lib = get_lib()
    for m in (1, 33, 64, 65, 871, 4096, 100000):
        for n in (8, 64, 2304, 32768):
            for k in (64, 1536, 16384):
                for mode in (False, True):
                    assert 0 <= ops.gemm_tiles_plan(m, n, k, mode) < len(TILES)
                    assert not (m <= 32 and ops.gemm_tiles_pays(m, n, k, mode))
    sup = lib.ic_gemm_tiles_supported
    assert sup(100, 64, 128, 128, 128, 64, 0) and sup(100, 64, 128, 136, 144, 72, 0) and sup(100, 64, 128, 128, 128, 32, 1)
    assert not sup(100, 64, 96, 96, 96, 64, 0)               # K in whole stages
    assert not sup(100, 68, 128, 128, 128, 72, 0)            # columns in 16-byte pieces
    assert not sup(100, 64, 128, 132, 128, 64, 0) and not sup(100, 64, 128, 128, 132, 64, 0) and not sup(100, 64, 128, 128, 128, 68, 0)
    assert not sup(100, 72, 128, 128, 128, 40, 1)            # gate and up in 16-byte pieces each
    assert not sup(100, 64, 128, 120, 128, 64, 0) and not sup(100, 64, 128, 128, 128, 56, 0) and not sup(0, 64, 128, 128, 128, 64, 0)
    assert not sup((1 << 31) - 1, 64, 64, 64, 64, 64, 0) and not sup(100, (1 << 31) - 8, 64, 64, 64, (1 << 31) - 8, 0)     # sums with a tile's rows stay in range
    assert lib.ic_gemm_tiles_plan(100, 64, 64, 3) == -1 and lib.ic_gemm_tiles_plan(100, 64, 64, -1) == -1 and lib.ic_gemm_tiles_plan(100, 64, 64, 2) >= 0
    assert not lib.ic_gemm_tiles_pays(100, 64, 64, 3) and not lib.ic_gemm_tiles_pays((1 << 31) - 1, 64, 64, 0)
    assert not sup(100, 1 << 16, 1 << 15, 1 << 15, 1 << 15, 1 << 15, 1)     # gate and up rows more than 32 bits of bytes apart


@pytest.mark.parametrize("M,N,K,swiglu,library,own", [
    # microseconds of the library (swiglu: with the activation's kernel) and of the tiles, weights out of memory
    (64, 4096, 14336, False, 40.0, 52.4), (48, 4096, 16384, False, 38.9, 49.2), (48, 2048, 11264, False, 20.2, 35.6), (33, 4096, 14336, False, 34.9, 41.2),
    (48, 2048, 12288, True, 24.3, 38.9), (64, 16384, 8192, True, 56.4, 68.2), (56, 768, 12288, False, 17.5, 39.3), (96, 16384, 6144, True, 54.1, 67.0),
    (160, 4096, 16384, False, 92.9, 67.2), (65, 4096, 16384, False, 50.0, 42.4), (64, 32768, 4096, True, 64.7, 63.0),
    (2048, 6912, 2304, False, 51.4, 58.1), (4096, 7680, 1536, False, 73.3, 79.4), (8192, 4096, 14336, False, 615.5, 704.4), (576, 64, 14784, False, 19.7, 30.9), (3300, 4096, 64, False, 10.9, 15.2), (7000, 2304, 64, False, 12.4, 15.8),
    (1300, 2304, 64, False, 5.7, 4.9),
    (33, 2304, 5760, False, 25.4, 17.4), (64, 2304, 2304, False, 9.9, 7.4), (256, 1536, 3840, False, 14.4, 10.3), (256, 2304, 2304, False, 11.5, 9.1),
    (871, 1536, 1536, False, 12.4, 9.0), (1045, 2560, 1536, False, 16.9, 12.1), (2048, 2304, 2304, False, 28.0, 23.1), (2048, 2304, 5760, False, 62.3, 59.2),
    (48, 7680, 1536, True, 14.3, 8.7), (64, 11520, 2304, True, 20.0, 16.0), (2048, 11520, 2304, True, 130.1, 98.2), (16384, 32768, 4096, True, 3195.3, 3007.4)])
def test_the_faster_side_cpu(M, N, K, swiglu, library, own):
    """The choice between tiles and library where both were measured well apart."""
    assert ops.gemm_tiles_pays(M, N, K, swiglu) == (own < library)


def test_short_walks_take_few_rounds_cpu():
    """A further round of tiles that share a unit costs its launch, first loads and way out however short its walk is: 4,096 x 2,304 x 64 took five
    rounds of 64 x 64 tiles (14.2 us; 9.7 in one round of 256 x 192)."""
    for M, N, K in ((4096, 2304, 64), (1045, 2304, 64), (871, 4096, 128), (2600, 1536, 192), (1024, 6144, 128)):
        bm, bn = TILES[ops.gemm_tiles_plan(M, N, K)]
        assert -(-M // bm) * -(-N // bn) <= 256, (M, N, K, bm, bn)
    assert TILES[ops.gemm_tiles_plan(871, 2304, 64)] == (64, 64)        # one round of them


def test_rules_of_a_partition_cpu():
    """The tiles and the choice against the library follow the units there are: 512 x 1,536 x 1,536 runs as 192 tiles of 64 x 64 on 256 units and as 32
    of 128 x 192 on 32."""
    from infinicore_infer_amd.kernels.lib import get_lib
    lib = get_lib()
    tiles = lambda units, M, N, K: (lambda bm, bn: (bm, bn, -(-M // bm) * -(-N // bn)))(*TILES[lib.ic_gemm_tiles_plan_on(M, N, K, 0, units)])
    for M, N, K in ((512, 1536, 1536), (256, 2048, 2048), (1024, 1024, 4096)):
        whole, part = tiles(256, M, N, K), tiles(32, M, N, K)
        assert whole[2] <= 256 and part[2] <= 32 and part[0] * part[1] > whole[0] * whole[1], (whole, part)
    # what a chip of 256 units does with 256 rounds' worth of work, 32 units do with an eighth of it
    assert not lib.ic_gemm_tiles_pays_on(4096, 4096, 4096, 0, 256) and lib.ic_gemm_tiles_pays_on(512, 4096, 4096, 0, 256)
    assert not lib.ic_gemm_tiles_pays_on(1024, 2048, 4096, 0, 32) and lib.ic_gemm_tiles_pays_on(1024, 2048, 4096, 0, 256)


def test_what_timing_found_cpu():
    """A timed shape's answer holds for it and for row counts within an eighth of it, the nearest timed one first."""
    from infinicore_infer_amd.kernels.lib import get_lib
    note = get_lib().ic_product_timing
    n, k = 5128, 1088                                  # (no test times this matrix)
    assert ops.product_timed(800, n, k) is None
    note(800, n, k, k, k, n, 0)
    note(1000, n, k, k, k, n, 1)
    assert ops.product_timed(800, n, k) is False and ops.product_timed(1000, n, k) is True
    assert ops.product_timed(700, n, k) is False and ops.product_timed(880, n, k) is False and ops.product_timed(920, n, k) is True
    assert ops.product_timed(699, n, k) is None and ops.product_timed(1126, n, k) is None
    assert ops.product_timed(800, n, k, ldc=n + 8) is None and ops.product_timed(800, n + 8, k) is None
    note(800, n, k, k, k, n, 1)
    assert ops.product_timed(700, n, k) is True


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("swiglu", [False, True])
def test_tiles_at_their_edges(tile, swiglu):
    bm, bn = TILES[tile]
    if swiglu and bn == 96:
        pytest.skip("three column tiles a wave: no pairs of gate and up")
    # one row; one tile exactly and one row and column piece more and less; several tiles; one stage of K, fewer and more stages than are loaded ahead
    for M, N, K, pad in ((1, 16, 64, 0), (bm, bn, 128, 0), (bm + 1, bn + 16, 192, 8), (bm - 1, 2 * bn - 16, 320, 0), (2 * bm + 3, 3 * bn + 48, 448, 64)):
        a, w = _operands(M, N, K, 7 * tile + M)
        cols = N // 2 if swiglu else N
        out = torch.full((M + 1, cols + pad), 3.0, dtype=BF16, device="cuda")
        ops.gemm_tiles(_strided(a, pad), _strided(w, pad), out[:M, :cols], swiglu_output=swiglu, tile=tile)
        _check(a, w, out[:M, :cols], swiglu)
        assert (out[M] == 3.0).all() and (out[:, cols:] == 3.0).all()       # nothing beside the result is written


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("swiglu", [False, True])
def test_tiles_over_long_walks(tile, swiglu):
    """41 and 128 stages, an odd and an even number of rounds of every tile's buffers: the products written as assembly (256 x 256) and the compiler's."""
    bm, bn = TILES[tile]
    if swiglu and bn == 96:
        pytest.skip("three column tiles a wave: no pairs of gate and up")
    for M, N, K in ((bm + 5, bn + 16, 2624), (bm, 2 * bn, 8192)):
        a, w = _operands(M, N, K, 100 + tile)
        out = torch.empty(M, N // 2 if swiglu else N, dtype=BF16, device="cuda")
        ops.gemm_tiles(a.cuda(), w.cuda(), out, swiglu_output=swiglu, tile=tile)
        _check(a, w, out, swiglu)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 7680, 1536), (65, 512, 512), (129, 1536, 3840), (871, 2560, 1536), (1045, 1536, 1536), (2049, 2304, 2304)])
def test_chosen_tiles_and_their_replays(M, N, K):
    """ops.product runs the tile that the rule names, and that recorded and replayed with other rows in between."""
    assert ops.gemm_tiles_pays(M, N, K)
    a, w = _operands(M, N, K, M)
    ad, wd, out, chosen = a.cuda(), w.cuda(), *(torch.empty(M, N, dtype=BF16, device="cuda") for _ in range(2))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.product(ad, wd, chosen)
        ops.gemm_tiles(ad, wd, out, tile=ops.gemm_tiles_plan(M, N, K))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            ops.gemm_tiles(ad, wd, out)
    torch.cuda.current_stream().wait_stream(side)
    _check(a, w, chosen, False)
    assert torch.equal(chosen, out)
    for _ in range(3):
        a = a.roll(1, 0)
        ad.copy_(a)
        graph.replay()
        torch.cuda.synchronize()
        _check(a, w, out, False)


@pytest.mark.gpu
def test_infinities_and_nan_stay_where_they_are():
    a, w = _operands(200, 256, 256, 1)
    a[3, 5], a[70, 255], a[199, 0] = float("inf"), float("nan"), -float("inf")
    for tile in range(len(TILES)):
        out = torch.empty(200, 256, dtype=BF16, device="cuda")
        ops.gemm_tiles(a.cuda(), w.cuda(), out, tile=tile)
        bad = ~torch.isfinite(out).all(1).cpu()
        assert bad.nonzero().view(-1).tolist() == [3, 70, 199]
        keep = ~bad
        _check(a[keep], w, out.cpu()[keep], False)


@pytest.mark.gpu
def test_refused_operands_go_to_the_library():
    """What the tiles do not take is an error there and the library's in ops.product."""
    for M, N, K, at in ((100, 200, 96, 0), (100, 250, 128, 0), (100, 200, 128, 1)):
        a, w = _operands(M, N, K, 3)
        room = torch.empty(M * K + 8, dtype=BF16, device="cuda")
        ad = room[at:at + M * K].view(M, K).copy_(a)            # at 1: not 16-byte aligned
        out = torch.empty(M, N, dtype=BF16, device="cuda")
        with pytest.raises(ops.KernelError):
            ops.gemm_tiles(ad, w.cuda(), out)
        ops.product(ad, w.cuda(), out)
        _check(a, w, out, False)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [None] + list(range(len(TILES))))
def test_qkv_with_rotary_and_cache_write(tile):
    """Queries, keys and values against float64: head sizes whose halves are one matrix tile, two and more, tokens without a slot, slots in any
    order, page sizes that are no power of two, heads that begin inside a tile."""
    if tile is not None and TILES[tile] in ((64, 96), (256, 256)):
        pytest.skip("three column tiles a wave: no pairs; 256 accumulators a lane: no registers")
    for M, K, nh, nkv, dh, ps in ((70, 128, 3, 1, 64, 16), (33, 64, 2, 2, 32, 7), (197, 192, 5, 2, 128, 64), (1, 320, 1, 1, 256, 3), (130, 2624, 4, 2, 64, 16)):
        a, w = _operands(M, (nh + 2 * nkv) * dh, K, M + dh)
        g = torch.Generator().manual_seed(M)
        pos = torch.randint(0, 500, (M,), generator=g, dtype=torch.int32)
        pages = (M + ps - 1) // ps + 1
        slots = torch.randperm(pages * ps, generator=g)[:M].to(torch.int32)
        slots[M // 2:M // 2 + 1] = -1
        half = dh // 2
        ang = torch.arange(500).double()[:, None] * 10000.0 ** (-torch.arange(half).double() / half)
        cos, sin = ang.cos().float(), ang.sin().float()
        qkv = torch.full((M, (nh + 2 * nkv) * dh), 3.0, dtype=BF16, device="cuda")
        k = torch.full((pages, nkv, ps, dh), 5.0, dtype=BF16, device="cuda")
        v = torch.full_like(k, 7.0)
        ops.gemm_tiles_rope(a.cuda(), w.cuda(), qkv, pos.cuda(), slots.cuda(), cos.cuda(), sin.cuda(), k, v, nh, nkv, dh, ps, tile=tile)
        ref = (a.double() @ w.double().t()).view(M, nh + 2 * nkv, dh)
        mag = ((a.double().abs() @ w.double().abs().t()) * K * 2.0 ** -24).view(M, nh + 2 * nkv, dh)
        c, s = cos.double()[pos.long()][:, None], sin.double()[pos.long()][:, None]
        rot = nh + nkv
        x, y, mx, my = ref[:, :rot, :half], ref[:, :rot, half:], mag[:, :rot, :half], mag[:, :rot, half:]
        want, bound = ref.clone(), mag.clone()
        want[:, :rot, :half], want[:, :rot, half:] = x * c - y * s, x * s + y * c
        # two products and a sum in float32 beside the sums' own error
        bound[:, :rot] = torch.cat([mx + my, mx + my], -1) + 2.0 ** -22 * torch.cat([x.abs() + y.abs()] * 2, -1)
        bound = bound + want.abs() * 2.0 ** -8
        got = want.clone()
        got[:, :nh] = qkv.cpu().double().view(M, -1, dh)[:, :nh]
        kk, vv = k.cpu().double().transpose(1, 2).reshape(pages * ps, nkv, dh), v.cpu().double().transpose(1, 2).reshape(pages * ps, nkv, dh)
        have = slots >= 0
        at = slots[have].long()
        got[have, nh:rot], got[have, rot:] = kk[at], vv[at]
        assert ((got - want).abs() - bound).max() <= 0, (M, K, nh, nkv, dh, ps)
        untouched = torch.ones(pages * ps, dtype=torch.bool)
        untouched[at] = False
        assert (kk[untouched] == 5.0).all() and (vv[untouched] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [264, 72])
def test_products_follow_what_timing_found(rows):
    """After timing, ops.product runs the kernel that was found the faster one, tiles or the library's kept algorithm, whatever the rule says."""
    from infinicore_infer_amd.kernels.lib import get_lib
    M, N, K = rows, 2560, 4032
    a, w = _operands(M, N, K, 5)
    ad, wd = a.cuda(), w.cuda()
    out, tiles, lib = (torch.empty(M, N, dtype=BF16, device="cuda") for _ in range(3))
    assert ops.product_timed(M, N, K) is None
    flush = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    assert ops.product_tune(ad, wd, out, reps=3, flush=flush) >= 2
    found = ops.product_timed(M, N, K)
    assert found is not None
    ops.gemm_tiles(ad, wd, tiles)
    ops.matmul_library(ad, wd, lib)
    for want in (found, not found):
        get_lib().ic_product_timing(M, N, K, K, K, N, int(want))
        ops.product(ad, wd, out)
        _check(a, w, out, False)
        assert torch.equal(out, tiles if want else lib)
    get_lib().ic_product_timing(M, N, K, K, K, N, int(found))
