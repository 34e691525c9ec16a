"""Float32 products on the bfloat16 matrix cores against 64-bit sums.

The bound of an element is (K + 16) 2^-24 sum |a| |w|: K roundings of a float32 sum in any order, and room for the three products of parts that are left out, under
2^-24 of a product (a second part is at most 2^-8 of its number, a third 2^-17)."""
import ctypes

import pytest
import torch

from infinicore_infer_amd.kernels import ops
from infinicore_infer_amd.kernels.lib import get_lib

# row tiles of 16, column tiles of 64: the order of the kernel's list
SHAPES = [(1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (6, 1), (7, 1), (4, 2), (5, 2), (6, 2), (7, 2), (8, 2), (4, 3), (6, 3), (8, 3)]


def _inputs(M, N, K, pad=0, seed=1):
    g = torch.Generator().manual_seed(seed * 1000003 + M * 7919 + N * 31 + K)
    a = torch.randn(M, K + pad, generator=g) * torch.exp(2.0 * torch.randn(M, 1, generator=g))
    w = torch.randn(N, K + pad, generator=g) * torch.exp(2.0 * torch.randn(N, 1, generator=g))
    return a[:, :K], w[:, :K]


def _check(got, a, w, alpha=1.0):
    A, W = a.double(), w.double()
    bound = (a.shape[1] + 16) * 2.0 ** -24 * abs(alpha) * (A.abs() @ W.abs().t())
    assert bool(((got.double().cpu() - alpha * (A @ W.t())).abs() <= bound).all())


def _check_norm(got, a, w, alpha=1.0):
    """Rows and columns scaled to one size, so that each counts alike: over all elements the error is under (4 + (K / 32)^(1/2)) 2^-24 of the result, a rounding per 32 k
    of a sum that is no larger, of either sign, and a few where the sums meet; a single row's or column's, of few elements, under four times that.  A third part that is
    missing shows by 2^-18.5, a second part's product by 2^-19.5 (rms)."""
    A, W = a.double(), w.double()
    A, W, scale = A / A.norm(dim=1, keepdim=True), W / W.norm(dim=1, keepdim=True), alpha * A.norm(dim=1)[:, None] * W.norm(dim=1)[None] / a.shape[1] ** 0.5
    off = got.double().cpu() / scale - (A @ W.t()) * a.shape[1] ** 0.5
    bound = (4 + (a.shape[1] / 32) ** 0.5) * 2.0 ** -24
    assert float(off.square().mean().sqrt()) < bound
    assert all(float(off.square().mean(dim).sqrt().max()) < 4 * bound for dim in (0, 1))


@pytest.mark.parametrize("units", [256, 64])
def test_plans(units):
    """Every plan names a shape and slices that the kernel takes; up to 32 rows the library's product stays."""
    lib, n = get_lib(), ctypes.c_int()
    for M in (1, 32, 33, 130, 517, 2048, 30000):
        for N, K in ((4, 32), (65, 64), (1536, 1536), (7680, 1536), (1536, 3840), (73440, 4096)):
            assert 0 <= lib.ic_gemm_f32_plan_on(M, N, K, units, n) < len(SHAPES)
            assert 1 <= n.value <= min(4, K // 32) and (n.value == 1 or N % 4 == 0)
            assert not (M <= 32 and lib.ic_gemm_f32_pays_on(M, N, K, units))
    assert lib.ic_gemm_f32_plan_on(0, 64, 64, units, n) == -1 and not lib.ic_gemm_f32_pays_on(100, 0, 64, units)
    sup = lib.ic_gemm_f32_supported
    assert sup(100, 64, 64, 64, 64, 64) and not sup(100, 64, 48, 64, 64, 64) and not sup(100, 64, 64, 66, 64, 64)
    assert not sup(100, 64, 64, 64, 60, 64) and not sup(100, 64, 64, 64, 64, 60) and not sup(0, 64, 64, 64, 64, 64)


def test_the_rule_prices_the_runs_that_a_workspace_makes():
    """A workspace for some of the rows means a split and a product per run of rows, each of which reads all weights again: what pays with room for all rows need not
    with less, never the other way, and none pays with none."""
    lib = get_lib()
    for M, N, K in ((130, 7680, 1536), (517, 1536, 3840), (2048, 4096, 16384), (8192, 4096, 16384)):
        room = [lib.ic_gemm_f32_parts_bytes(rows, K) for rows in (16, 48, 256, M)] + [64 << 20, 1 << 40]
        pays = [lib.ic_gemm_f32_pays_with(M, N, K, n, 256) for n in sorted(room)]
        assert pays == sorted(pays) and pays[0] == 0 and pays[-1] == 1
        assert not lib.ic_gemm_f32_pays_with(M, N, K, 0, 256) and not lib.ic_gemm_f32_pays_with(M, N, K, room[0] - 1, 256)
        assert lib.ic_gemm_f32_pays_on(M, N, K, 256) == lib.ic_gemm_f32_pays_with(M, N, K, lib.ic_gemm_f32_workspace_bytes(M, N, K), 256)


def test_short_rows_and_narrow_matrices_go_to_the_library():
    """Of few k the library's product takes 3.6..8.5 us, less than the split of A and the product of parts (5.5..17), and of narrow matrices whose tiles fill the chip once 12..19
    (17..26); wide and long ones are faster in parts."""
    pays = get_lib().ic_gemm_f32_pays_on
    for M, N, K in ((33, 32, 32), (64, 512, 128), (300, 512, 128), (130, 1536, 512), (2048, 256, 512), (1000, 128, 256), (2048, 128, 64), (517, 1536, 128), (300, 1536, 512),
                    (1500, 512, 768), (1000, 768, 768), (2048, 512, 1024), (1000, 1024, 1024), (700, 1024, 768)):
        assert not pays(M, N, K, 256)
    for M, N, K in ((2048, 4096, 512), (1000, 4096, 512), (130, 7680, 1536), (517, 1536, 3840), (517, 1536, 1536), (517, 2560, 1536), (2048, 7680, 1536),
                    (300, 2560, 1536), (388, 1536, 1536), (76, 7680, 1536), (216, 1536, 3840)):
        assert pays(M, N, K, 256)


@pytest.mark.gpu
def test_a_small_workspace_goes_to_the_library():
    """With scratch memory for 16 rows at a time (129 runs over 32 MB of weights) the product by the rule is the library's."""
    M, N, K = 2064, 2048, 4096
    a, w = _inputs(M, N, K)
    A, W, out, lib = a.cuda(), w.cuda(), torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    parts = torch.empty(int(get_lib().ic_gemm_f32_parts_bytes(16, K)), dtype=torch.uint8, device="cuda")
    ops.product(A, W, out, parts=parts)
    assert torch.equal(out, ops.matmul_library(A, W, lib))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_edges(shape):
    """Rows and columns around a tile's edges, one k-step and odd numbers of them, padded strides, slices; nothing beyond the matrix is written."""
    bm, bn = 16 * SHAPES[shape][0], 64 * SHAPES[shape][1]
    for M, N, K, pad, slices, alpha in ((1, 4, 32, 0, 1, 1.0), (bm, bn, 64, 4, 1, 1.0), (bm + 1, bn + 1, 96, 0, 1, -0.5), (2 * bm - 1, 3 * bn - 1, 288, 8, 1, 1.0),
                                        (bm - 1, bn + 4, 64, 0, 2, 1.0), (3 * bm + 5, bn - 4, 416, 4, 3, 2.0), (17, 2 * bn, 128, 0, 4, 1.0), (bm, 68, 1056, 0, 4, 1.0)):
        a, w = _inputs(M, N, K, pad, shape)
        ldc = (N + 3) // 4 * 4 + 8
        out = torch.full((M + 2, ldc), 7.0, device="cuda")
        A, W = torch.empty(M, K + pad, device="cuda"), torch.empty(N, K + pad, device="cuda")
        A[:, :K], W[:, :K] = a.cuda(), w.cuda()
        ops.gemm_f32(A[:, :K], W[:, :K], out[:M, :N], alpha, shape, slices)
        _check(out[:M, :N], a, w, alpha)
        _check_norm(out[:M, :N], a, w, alpha)
        assert bool((out[M:] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 260, 96), (257, 1536, 1536), (130, 2304, 2304), (517, 512, 3840)])
def test_chosen(M, N, K):
    """The plan it makes itself, the product by the rule, and rows in several runs where the workspace is small."""
    a, w = _inputs(M, N, K)
    A, W, out = a.cuda(), w.cuda(), torch.empty(M, N, device="cuda")
    _check(ops.gemm_f32(A, W, out), a, w)
    _check_norm(out, a, w)
    _check(ops.product(A, W, out, 0.25), a, w, 0.25)
    small = torch.empty(int(get_lib().ic_gemm_f32_parts_bytes(48, K)) + 16, dtype=torch.uint8, device="cuda")
    _check(ops.gemm_f32(A, W, out.zero_(), workspace=small), a, w)
    _check_norm(out, a, w)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [264, 72])
def test_products_follow_what_timing_found(rows):
    """After timing, ops.product runs the kernel that was found the faster one, whatever the rule says, here and with the caller's own scratch memory; bfloat16 products of
    the same shape are not asked about."""
    M, N, K = rows, 2560, 4032
    a, w = _inputs(M, N, K)
    A, W, (out, own, lib) = a.cuda(), w.cuda(), (torch.empty(M, N, device="cuda") for _ in range(3))
    assert ops.product_timed(M, N, K, dtype=torch.float32) is None
    flush = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    assert ops.product_tune(A, W, out, reps=3, flush=flush) >= 2
    found = ops.product_timed(M, N, K, dtype=torch.float32)
    assert found is not None
    ops.gemm_f32(A, W, own)
    ops.matmul_library(A, W, lib)
    assert not torch.equal(own, lib)
    parts = torch.empty(ops.product_parts_bytes(M, N, K), dtype=torch.uint8, device="cuda")
    for want in (found, not found):
        get_lib().ic_product_f32_timing(M, N, K, K, K, N, int(want))
        for mine in (None, parts):
            ops.product(A, W, out.zero_(), parts=mine)
            _check(out, a, w)
            assert torch.equal(out, own if want else lib)
    get_lib().ic_product_f32_timing(M, N, K, K, K, N, int(found))


def test_what_timing_found_cpu():
    """A timed float32 shape says nothing about the bfloat16 one, nor the other way."""
    lib, n, k = get_lib(), 5128, 1120                  # (no other test times this matrix)
    lib.ic_product_f32_timing(800, n, k, k, k, n, 1)
    assert ops.product_timed(700, n, k, dtype=torch.float32) is True and ops.product_timed(800, n, k) is None
    lib.ic_product_timing(800, n, k, k, k, n, 0)
    assert ops.product_timed(800, n, k, dtype=torch.float32) is True and ops.product_timed(800, n, k) is False


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,lda,off", [(300, 2560, 1536, 1538, 0), (300, 2560, 1528, 1528, 0), (300, 2560, 1536, 1540, 1), (300, 2557, 1536, 1536, 0)])
def test_product_of_forms_the_kernel_does_not_take(M, N, K, lda, off):
    """Odd strides, rows that are no whole k-steps, misaligned operands: the product by the rule is right as ever."""
    a, w = _inputs(M, N, K)
    store = torch.zeros(M * lda + 8, device="cuda")
    A = store[off:off + M * lda].view(M, lda)[:, :K]
    A.copy_(a)
    _check(ops.product(A, w.cuda(), torch.empty(M, N, device="cuda")), a, w)


@pytest.mark.gpu
@pytest.mark.parametrize("slices", [1, 3])
def test_values_that_are_not_finite(slices):
    """Infinities, NaN and the largest numbers come out as a float32 sum has them, and touch only their own row or column."""
    M, N, K = 37, 132, 192
    a, w = _inputs(M, N, K)
    w = w.abs() / w.norm(dim=1, keepdim=True)
    a[3, 5], a[4, 7], a[5, 9], a[6, 11] = float("inf"), float("-inf"), float("nan"), 3.4028234e38
    w[8, 100], w[9, 0] = float("inf"), -3.4e38
    a[:, 0] = 0.5                                   # (no sum overflows on its way)
    A, W, out = a.cuda(), w.cuda(), torch.empty(M, N, device="cuda")
    ops.gemm_f32(A, W, out, 1.0, 3, slices)
    want = (a.double() @ w.double().t()).float()
    same = (out.cpu() == want) | (out.cpu().isnan() & want.isnan())
    finite = want.isfinite() & out.cpu().isfinite()
    assert bool((same | finite).all())
    rows = [m for m in range(M) if m not in (3, 4, 5, 6)]
    cols = [n for n in range(N) if n not in (8, 9)]
    _check(out[rows][:, cols], a[rows], w[cols])
    _check(out[[6]][:, cols], a[[6]], w[cols])


@pytest.mark.gpu
def test_smaller_error_than_the_library():
    """Against 64 bits the parts' error is no larger than the library's float32 product has it."""
    for M, N, K in ((40, 1536, 1536), (256, 2560, 1536), (517, 1536, 3840), (130, 512, 32), (517, 1536, 64), (33, 4096, 128), (300, 256, 256), (1000, 512, 512)):
        a, w = _inputs(M, N, K, seed=9)
        A, W, own, lib = a.cuda(), w.cuda(), torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
        ops.gemm_f32(A, W, own)
        ops.matmul_library(A, W, lib)
        want = A.double() @ W.double().t()
        assert (own.double() - want).norm() <= (lib.double() - want).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("slices", [1, 2])
def test_rows_of_one_term(slices):
    """A result that is one product has that product's error only, and of either sign: 2^-24 for its rounding, 2^-24 for the parts left out (2^-8 2^-17 twice) and the
    roundings of the five smaller products, under 2^-28 together.  On average nothing is left out: 65,536 errors of 2^-24.2 at most and any sign are under 2^-29."""
    M, N, K = 256, 256, 256
    a, w = _inputs(M, N, K)
    at = torch.arange(M) * 37 % K                                   # (every k once)
    a = torch.zeros(M, K).scatter_(1, at[:, None], a.gather(1, at[:, None]))
    out = torch.empty(M, N, device="cuda")
    ops.gemm_f32(a.cuda(), w.cuda(), out, 1.0, 7, slices)
    want = a.double() @ w.double().t()
    off = (out.double().cpu() - want) / want
    assert float(off.abs().max()) < 2.0 ** -23 + 2.0 ** -28
    assert abs(float(off.mean())) < 2.0 ** -29


@pytest.mark.gpu
@pytest.mark.parametrize("slices", [1, 2])
@pytest.mark.parametrize("tiny", ["a", "w"])
def test_tiny_numbers(tiny, slices):
    """Rows of one term down to 2^-118, whose third part no bfloat16 number holds: a float32 product's error (2^-24; in parts 2^-23 and the five roundings), and other rows as ever."""
    M, N, K = 60, 132, 128
    a, w = _inputs(M, N, K)
    one, many = (a, w) if tiny == "a" else (w, a)
    n = one.shape[0]
    at = torch.arange(n) * 37 % K
    one = torch.zeros(n, K).scatter_(1, at[:, None], one.gather(1, at[:, None]).sign() * (1.0 + torch.rand(n, 1, generator=torch.Generator().manual_seed(3))))
    one *= torch.exp2(-(torch.arange(n) % 20).double() * 2 - 80).float()[:, None]                 # 2^-80 .. 2^-118
    many = many.sign() * (1.0 + torch.rand(many.shape, generator=torch.Generator().manual_seed(4)))
    one[::3] = torch.randn(one[::3].shape, generator=torch.Generator().manual_seed(5))
    a, w = (one, many) if tiny == "a" else (many, one)
    out = torch.empty(M, N, device="cuda")
    ops.gemm_f32(a.cuda(), w.cuda(), out, 1.0, 7, slices)
    want = a.double() @ w.double().t()
    _check(out, a, w)
    off = (out.double().cpu() / want - 1.0).abs()
    off = off if tiny == "a" else off.t()
    off[::3] = 0.0
    assert float(off.max()) < 2.0 ** -23 + 2.0 ** -28


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 64])
def test_numbers_whose_upper_half_is_small(K):
    """All operands one number whose lower 16 bits are all ones: its upper half leaves 2^-7 of it, and K products of a sign err alike.  Two float32 roundings per 32 k
    and one where the two sums meet, 2^-24 each, and 2^-24 for what is left out."""
    x = torch.tensor(0x3f80ffff, dtype=torch.int32).view(torch.float32).item()
    a, w, out = torch.full((40, K), x), torch.full((64, K), x), torch.empty(40, 64, device="cuda")
    ops.gemm_f32(a.cuda(), w.cuda(), out)
    assert float((out.double().cpu() / (K * float(x) ** 2) - 1.0).abs().max()) < (2 + K / 16) * 2.0 ** -24


def _fastest(call, n=7):
    times = []
    for _ in range(n):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            call()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


@pytest.mark.gpu
@pytest.mark.parametrize("slices", [1, 2])
def test_a_row_that_is_not_finite_costs_others_little(slices):
    """A request whose row holds a NaN shares its step with others: their results keep their bits outside the row's 16, and the product takes at most three times as long
    (with a result summed by one lane, k after k, it took twenty times)."""
    M, N, K = 517, 7680, 1536
    a, w = _inputs(M, N, K)
    A, W, out, want = a.cuda(), w.cuda(), torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    call = lambda: ops.gemm_f32(A, W, out, 1.0, 11, slices)          # noqa: E731
    call()
    clean = _fastest(call)
    want.copy_(out)
    A[300, 7] = float("nan")
    call()
    rows = torch.tensor([m // 16 != 300 // 16 for m in range(M)], device="cuda")
    assert torch.equal(out[rows], want[rows]) and bool(out[300].isnan().all())
    _check(out[[m for m in range(288, 304) if m != 300]], a[[m for m in range(288, 304) if m != 300]], w)
    assert _fastest(call) < 3.0 * clean
