"""GPU: the products of every tile size at the edges of tiles, k-tiles and
ring trips, against fp64.

The bound is elementwise: products of 16-bit operands are exact in fp32, each
of the K fp32 additions rounds by at most 2^-24 of a partial sum no larger
than sum |a||b| (doubled for the order inside an MFMA), and the result rounds
once to its dtype (2^-9 of a bf16 value, 2^-12 of an fp16 one, with fp16's
subnormal spacing as a floor)."""

import ctypes

import pytest
import torch

from eth_amd import _native as nat
from eth_amd import kernels as K
from tests.conftest import announce

pytestmark = pytest.mark.gpu

LAYOUTS = [(True, True), (True, False), (False, False), (False, True)]


def _plan(M, N, Kd, a_k, b_k, dtype, ldc=None):
    """(tile, rows, columns) of the first launch and the tile of the second
    (0: none), as the library plans it."""
    plan = (ctypes.c_int64 * 4)()
    nat.call("eth_gemm_plan", M, N, Kd, int(a_k), int(b_k), ldc or N, nat.dtype_code(dtype), plan)
    return tuple(plan)


def _operands(M, N, Kd, a_k, b_k, dtype, cuda, seed):
    gen = torch.Generator().manual_seed(seed)
    a = torch.randn(M, Kd, generator=gen).to(dtype)
    b = (torch.randn(Kd, N, generator=gen) * 0.1).to(dtype)
    ad = a.to(cuda) if a_k else a.t().contiguous().to(cuda).t()
    bd = b.t().contiguous().to(cuda).t() if b_k else b.to(cuda)
    return a.double(), b.double(), ad, bd


def _check(got, ref, mag, Kd, out_dtype, what):
    unit = {torch.float32: 2.0**-23, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[out_dtype]
    bound = 2 * Kd * 2.0**-24 * mag + unit * ref.abs() + 2.0**-24
    err = (got.cpu().double() - ref).abs()
    assert bool((err <= bound).all()), f"{what}: worst {(err / bound).max().item():.3g} of the bound"


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("M,N,Kd", [
    (8, 8, 8),          # less than a tile in every direction
    (64, 64, 64),       # one 64x64 tile, one k-tile
    (72, 136, 72),      # one past a tile, k-tail of one chunk
    (128, 128, 192),    # three k-tiles: the remainder steps alone
    (120, 248, 264),    # four k-tiles and a tail
    (200, 328, 1000),   # ragged everywhere
    (2048, 1024, 328),  # a whole round and k-tail of one chunk
    (1928, 2056, 520),  # past a whole round, ragged edges
])
def test_products_at_tile_edges(cuda, M, N, Kd, a_k, b_k):
    """64x64 tiles."""
    assert _plan(M, N, Kd, a_k, b_k, torch.float32) == (64, M, N, 0)
    _products(cuda, M, N, Kd, a_k, b_k)


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("M,N,Kd", [
    # ragged edges, 33 to 36 k-tiles (every remainder of a trip round the
    # four stages), the last one short in three of them
    (1928, 1032, 2056), (1928, 1032, 2120), (1928, 1032, 2184), (1928, 1032, 2304),
])
def test_128_tiles(cuda, a_k, b_k, M, N, Kd):
    assert _plan(M, N, Kd, a_k, b_k, torch.float32) == (128, M, N, 0)
    _products(cuda, M, N, Kd, a_k, b_k)


def _products(cuda, M, N, Kd, a_k, b_k):
    announce(f"gemm {M}x{N}x{Kd} a_k={a_k} b_k={b_k}")
    for dtype in (torch.bfloat16, torch.float16):
        a, b, ad, bd = _operands(M, N, Kd, a_k, b_k, dtype, cuda, M + 3 * N + 7 * Kd)
        ref, mag = a @ b, a.abs() @ b.abs()
        bias = torch.linspace(-1, 1, N).to(dtype)
        _check(K.gemm(ad, bd, bias=bias.to(cuda)), ref + bias.double(), mag + bias.double().abs(), Kd, dtype,
               f"{dtype} with bias")
        acc = torch.full((M, N), 0.5, device=cuda)
        K.gemm(ad, bd, out=acc, accumulate=True)
        _check(acc, ref + 0.5, mag + 0.5, Kd, torch.float32, f"{dtype} accumulated")
        once = acc.clone().fill_(0.5)
        K.gemm(ad, bd, out=once, accumulate=True)
        assert torch.equal(acc, once)


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("Kd,dtype", [
    # the last k-tile short: one, two, three, four and six k-tiles
    (8, torch.bfloat16), (72, torch.float16), (184, torch.bfloat16), (200, torch.bfloat16), (328, torch.float16),
    # an odd number of whole k-tiles
    (64, torch.bfloat16), (192, torch.float16),
])
def test_wide_tiles_any_depth(cuda, a_k, b_k, Kd, dtype):
    """128 tiles of 256x256 with ragged edges, every k-tile count the loop
    and its prologue treat apart."""
    M, N = 4088, 2040
    assert _plan(M, N, Kd, a_k, b_k, torch.float32) == _plan(M, N, Kd, a_k, b_k, dtype) == (256, M, N, 0)
    announce(f"gemm wide {M}x{N}x{Kd} a_k={a_k} b_k={b_k}")
    a, b, ad, bd = _operands(M, N, Kd, a_k, b_k, dtype, cuda, Kd)
    ref, mag = a @ b, a.abs() @ b.abs()
    acc = torch.full((M, N), 0.5, device=cuda)
    K.gemm(ad, bd, out=acc, accumulate=True)
    _check(acc, ref + 0.5, mag + 0.5, Kd, torch.float32, "accumulated")
    _check(K.gemm(ad, bd), ref, mag, Kd, dtype, "16-bit")


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
def test_short_k_tile_reads_nothing_past_k(cuda, a_k, b_k):
    """K columns of operands whose rows go on with NaN: what lies past K in
    memory is no part of the product."""
    M, N, Kd = 4088, 2040, 200
    announce(f"gemm wide views {M}x{N}x{Kd} a_k={a_k} b_k={b_k}")
    a, b, _, _ = _operands(M, N, Kd, a_k, b_k, torch.bfloat16, cuda, 3)
    nan = lambda *shape: torch.full(shape, float("nan"), dtype=torch.bfloat16, device=cuda)  # noqa: E731
    wide_a = nan(M, Kd + 56) if a_k else nan(Kd + 56, M)
    wide_b = nan(N, Kd + 56) if b_k else nan(Kd + 56, N)
    ad = wide_a[:, :Kd] if a_k else wide_a[:Kd].t()
    bd = wide_b[:, :Kd].t() if b_k else wide_b[:Kd]
    ad.copy_(a)
    bd.copy_(b)
    _check(K.gemm(ad, bd), a @ b, a.abs() @ b.abs(), Kd, torch.bfloat16, "views")


@pytest.mark.parametrize("a_k,b_k,M,N,Kd,dtype,plan", [
    # 300 wide tiles: 240 and a rest of columns, or of rows
    (False, False, 7680, 2552, 520, torch.bfloat16, (256, 7680, 2048, 128)),
    (False, False, 2552, 7680, 520, torch.bfloat16, (256, 2048, 7680, 128)),
    (True, True, 2304, 8192, 512, torch.float16, (256, 2048, 8192, 64)),
    (True, False, 8200, 2048, 512, torch.bfloat16, (256, 8192, 2048, 64)),  # eight rows past a whole round
    # 792: a last round of 24, deep enough for a smaller promise
    (True, True, 4552, 11224, 1024, torch.bfloat16, (256, 4352, 11224, 128)),
    # a rest of columns (of B's, the bias's and C's rows), in every layout
    (True, True, 8192, 2304, 512, torch.bfloat16, (256, 8192, 2048, 64)),
    (True, False, 8184, 2312, 512, torch.float16, (256, 8184, 2048, 128)),
    (False, False, 8184, 2312, 520, torch.float16, (256, 8184, 2048, 128)),
    (True, True, 8184, 2308, 520, torch.bfloat16, (256, 8184, 2048, 128)),
    (False, True, 8184, 2308, 512, torch.bfloat16, (256, 8184, 2048, 128)),
    # a rest of rows of the same layout
    (False, True, 2552, 7684, 512, torch.float16, (256, 2048, 7684, 128)),
])
def test_products_past_whole_rounds(cuda, a_k, b_k, M, N, Kd, dtype, plan):
    """Grids a little over a whole number of rounds run in two launches."""
    assert _plan(M, N, Kd, a_k, b_k, torch.float32) == _plan(M, N, Kd, a_k, b_k, dtype, N + 8) == plan
    announce(f"gemm rounds {M}x{N}x{Kd} a_k={a_k} b_k={b_k}")
    gen = torch.Generator(device=cuda).manual_seed(M + N)
    a = torch.randn(*((M, Kd) if a_k else (Kd, M)), device=cuda, generator=gen).to(dtype)
    b = torch.randn(*((N, Kd) if b_k else (Kd, N)), device=cuda, generator=gen).to(dtype)
    ad, bd = a if a_k else a.t(), b.t() if b_k else b
    bias = torch.linspace(-1, 1, N, device=cuda).to(dtype)
    ref = (ad.double() @ bd.double()).cpu()
    mag = (ad.double().abs() @ bd.double().abs()).cpu()
    extra = bias.double().cpu()
    wide = torch.full((M, N + 8), 9.0, dtype=dtype, device=cuda)
    K.gemm(ad, bd, out=wide[:, :N], bias=bias)
    _check(wide[:, :N], ref + extra, mag + extra.abs(), Kd, dtype, "strided output with bias")
    assert bool((wide[:, N:] == 9).all())
    acc = torch.full((M, N), 0.5, device=cuda)
    K.gemm(ad, bd, out=acc, accumulate=True)
    _check(acc, ref + 0.5, mag + 0.5, Kd, torch.float32, "accumulated")


@pytest.mark.parametrize("a_k,b_k,Kd,splits", [
    (True, True, 320, 3),     # two whole splits and a short one
    (True, False, 1984, 16),  # 31 k-tiles: two each, the last split one
    (False, False, 200, 16),  # fewer k-tiles than splits, the last one short
    (False, True, 512, 2),
    (True, True, 1000, 5),    # four k-tiles a split, the last split with a short one
    (True, False, 264, 2),    # the last split two k-tiles, one of them of a single chunk
    (False, True, 576, 3),    # three k-tiles a split
    (False, True, 648, 4),    # an odd count and a short k-tile
    (False, True, 640, 4),    # pairs of k-tiles, the last split an odd one
])
def test_splitk_every_output(cuda, a_k, b_k, Kd, splits):
    M, N = 264, 136
    announce(f"gemm split-K {M}x{N}x{Kd}/{splits} a_k={a_k} b_k={b_k}")
    for dtype in (torch.bfloat16, torch.float16):
        a, b, ad, bd = _operands(M, N, Kd, a_k, b_k, dtype, cuda, Kd + splits)
        ref, mag = a @ b, a.abs() @ b.abs()
        bias = torch.linspace(-1, 1, N).to(dtype)
        bd1 = bias.to(cuda)
        lda, ldb = ad.stride(0 if a_k else 1), bd.stride(1 if b_k else 0)
        ws = torch.full((splits * M * N,), float("nan"), device=cuda)
        for out_dtype in (dtype, torch.float32):
            out = torch.full((M, N + 4), 0.5, dtype=out_dtype, device=cuda)
            accumulate = out_dtype == torch.float32
            flags = nat.GEMM_BIAS | (nat.GEMM_ACCUMULATE if accumulate else 0)
            nat.call("eth_gemm_splitk_out", nat.ptr(ad), lda, int(a_k), nat.ptr(bd), ldb, int(b_k), nat.ptr(out),
                     out.stride(0), nat.dtype_code(out_dtype), nat.ptr(bd1), M, N, Kd, nat.dtype_code(dtype),
                     flags, 2.0, splits, nat.ptr(ws), nat.stream_ptr(cuda))
            extra = bias.double() + (0.5 if accumulate else 0.0)
            _check(out[:, :N], 2 * ref + extra, 2 * mag + extra.abs(), Kd, out_dtype, f"{dtype} -> {out_dtype}")
            assert bool((out[:, N:] == 0.5).all())


def test_deep_product_takes_splits(cuda):
    """A 16-bit output of two wide tiles, 16448 deep: split-K, the same bits
    every time, and refused where the plain product is."""
    M, N, Kd = 256, 512, 16448
    announce(f"gemm deep {M}x{N}x{Kd}")
    out = torch.empty(M, N, dtype=torch.bfloat16, device=cuda)
    splits = K._splitk_splits(M, N, Kd, out)
    pays = lambda *args: K._splitk_pays(*args, nat.ETH_BF16)  # noqa: E731
    assert splits == 16 and pays(M, N, Kd, splits, 1, 0) and pays(M, N, Kd + 8, splits, 1, 0)
    assert not pays(M, N, Kd + 4, splits, 1, 0) and not pays(2048, 2048, 2048, 2, 1, 1)
    # half a round of wide tiles splits in two, one tile more does not
    half = torch.empty(2048, 4096, dtype=torch.bfloat16, device=cuda)
    assert K._splitk_splits(2048, 4096, 16384, half) == 2 and pays(2048, 4096, 16384, 2, 1, 1)
    assert K._splitk_splits(2049, 4096, 16384, half) == 1
    a, b, ad, bd = _operands(M, N, Kd, True, False, torch.bfloat16, cuda, 5)
    got = K.gemm(ad, bd)
    _check(got, a @ b, a.abs() @ b.abs(), Kd, torch.bfloat16, "deep")
    assert torch.equal(got, K.gemm(ad, bd))


@pytest.mark.parametrize("M,Kd,N,tile", [(70, 136, 3, 64), (70, 136, 7, 64), (70, 136, 66, 64), (70, 136, 131, 64),
                                         (1928, 2056, 1031, 128)])
def test_products_with_unaligned_output_rows(cuda, M, Kd, N, tile):
    """Output widths and row strides that take no vector stores, 16-bit and
    accumulated."""
    announce(f"gemm {M}x{N}x{Kd} unaligned C")
    for a_k, dtype in ((True, torch.bfloat16), (False, torch.float16)):
        m = M - M % 8 if not a_k else M  # rows of a row-contiguous A are whole 16-byte units
        assert _plan(m, N, Kd, a_k, True, dtype, N + 3) == (tile, m, N, 0)
        a, b, ad, bd = _operands(m, N, Kd, a_k, True, dtype, cuda, N)
        ref, mag = a @ b, a.abs() @ b.abs()
        bias = torch.linspace(-1, 1, N).to(dtype)
        wide = torch.full((m, N + 3), 9.0, dtype=dtype, device=cuda)
        K.gemm(ad, bd, out=wide[:, 1 : N + 1], bias=bias.to(cuda))
        _check(wide[:, 1 : N + 1], ref + bias.double(), mag + bias.double().abs(), Kd, dtype, "strided output")
        assert bool((wide[:, 0] == 9).all()) and bool((wide[:, N + 1 :] == 9).all())
        acc = torch.full((m, N + 3), 0.5, device=cuda)
        K.gemm(ad, bd, out=acc[:, 1 : N + 1], accumulate=True)
        _check(acc[:, 1 : N + 1], ref + 0.5, mag + 0.5, Kd, torch.float32, "accumulated")
        assert bool((acc[:, 0] == 0.5).all()) and bool((acc[:, N + 1 :] == 0.5).all())
