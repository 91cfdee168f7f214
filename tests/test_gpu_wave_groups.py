"""The K-quarter kernel (each wave a quarter of K: 128x96 from K = 1536, 64x64
with at most one tile per CU from K = 704, 776 with a row-major b) where its
schedule can go wrong: K around whole quads and around the rules' lines, ragged
tiles, both output types, an overflow in any quarter."""

import pytest
import torch

import f16acc_amd as f16acc
from f16acc_amd.kernel import mm_bias, mm_flags, mm_tile, tile_config
from oracle import chunk32

pytestmark = pytest.mark.gpu
TILE = "128x96k2"


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


@pytest.mark.parametrize("M, N", [(128, 96), (129, 97), (120, 200)])
@pytest.mark.parametrize("K", [8, 136, 1160, 1528, 1536, 1544, 1640, 1664, 1928, 2040, 2048, 2056, 2568])
def test_quads_per_wave_against_the_oracle(M, N, K):
    a, w = rnd((M, K), 7 + K), rnd((N, K), 8 + K)
    ga, gb = a.cuda(), w.cuda().t()
    ref = chunk32.mm(a, w.t(), torch.float32)
    c32, flags = mm_flags(ga, gb, torch.float32, tile=TILE)
    assert tile_config(ga, gb, TILE)["tile"] == TILE and int(flags.sum()) == 0
    # FP32 reassociation, and chunk partials whose sums fall on either side of
    # a binary16 tie: 2^-11 of a partial, on few of K / 32
    assert chunk32.rel(c32.cpu(), ref) < 1e-3
    assert float((c32.cpu().double() - ref.double()).norm() / ref.double().norm()) < 2e-5
    assert torch.equal(mm_tile(ga, gb, TILE), c32.half())
    full = mm_tile(ga, gb, TILE, torch.float32, chunked=False)
    assert chunk32.rel(full.cpu(), (a.float() @ w.t().float()).double()) < 1e-5


def picks_64(a, b):
    cfg = tile_config(a, b)
    assert cfg["tile"] == "64x64" and cfg["tiles_m"] * cfg["tiles_n"] <= 256


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M, N, K", [(1024, 1024, 512), (1024, 1024, 1024), (1000, 1016, 520), (961, 1024, 648),
                                     (1024, 968, 1160), (1023, 1000, 1544), (1024, 1024, 696),
                                     (1024, 1024, 704), (1000, 1016, 768), (1024, 1000, 776)])
def test_64x64_in_k_quarters_against_one_wave_group(M, N, K, b_t):
    """At most one 64x64 tile per CU runs in wave K groups; 128x128 sums K in
    order.  The same rounded chunks in another FP32 order (sums
    below 2^8 of values of at most 11 bits: at most a few ulps of FP32 apart)."""
    a, w = rnd((M, K), 31).cuda(), rnd((N, K), 32).cuda()
    b = w.t() if b_t else w.t().contiguous()
    picks_64(a, b)
    c, flags = mm_flags(a, b, torch.float32)
    one = mm_tile(a, b, "128x128", torch.float32)
    off = (c - one).abs()
    # an element may also hold a partial that summed to the other side of a tie
    assert int(flags.sum()) == 0 and float((off > 1e-4).float().mean()) < 1e-3 * K / 32 and float(off.max()) < 2 ** -4
    assert torch.equal(f16acc.mm(a, b), c.half()) and torch.equal(mm_tile(a, b, "64x64", torch.float32), c)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("quarter", range(4))
@pytest.mark.parametrize("K", [512, 1024])  # one wave group, four
def test_64x64_redoes_an_overflow_in_any_quarter(K, quarter, b_t):
    """The overflow closed form (chunk sums past 65504 that cancel: exactly 100
    in FP32) in one wave's K range, the other ranges zero there."""
    M = N = 1024
    a, b = rnd((M, K), 33), rnd((K, N), 34)
    r0, c0, k0 = 64 * 5 + 20, 64 * 11 + 40, K // 4 * quarter
    a[r0:r0 + 10, :] = 100.0
    b[:, c0:c0 + 10] = 0.0
    for q, v in enumerate((30.0, -30.0, 30.0, -30.0)):
        b[k0 + 32 * q:k0 + 32 * q + 32, c0:c0 + 10] = v
    b[k0 + 127, c0:c0 + 10] = -29.0
    ga, gb = a.cuda(), b.t().contiguous().cuda().t() if b_t else b.cuda()
    picks_64(ga, gb)
    c, flags = mm_flags(ga, gb, torch.float32)
    assert int(flags.sum()) == 1 and flags[5, 11] == 1
    assert bool((c[r0:r0 + 10, c0:c0 + 10] == 100.0).all())
    # redone whole in FP32: the bits of that mode
    full = mm_tile(ga, gb, "64x64", torch.float32, chunked=False)
    assert torch.equal(c[320:384, 704:768], full[320:384, 704:768])


@pytest.mark.parametrize("quarter", range(4))
def test_128x96_redoes_an_overflow_in_any_quarter(quarter):
    """The same closed form on tile (1, 1) of 128x96 at K = 1536."""
    M, N, K = 300, 250, 1536
    a, w = rnd((M, K), 35), rnd((N, K), 36)
    r0, c0, k0 = 128 + 70, 96 + 60, 384 * quarter + 128
    a[r0:r0 + 10, :] = 100.0
    w[c0:c0 + 10, :] = 0.0
    for q, v in enumerate((30.0, -30.0, 30.0, -30.0)):
        w[c0:c0 + 10, k0 + 32 * q:k0 + 32 * q + 32] = v
    w[c0:c0 + 10, k0 + 127] = -29.0
    ga, gb = a.cuda(), w.cuda().t()
    c, flags = mm_flags(ga, gb, torch.float32, tile=TILE)
    assert int(flags.sum()) == 1 and flags[1, 1] == 1
    assert bool((c[r0:r0 + 10, c0:c0 + 10] == 100.0).all())
    full = mm_tile(ga, gb, TILE, torch.float32, chunked=False)
    assert torch.equal(c[128:256, 96:192], full[128:256, 96:192])


@pytest.mark.parametrize("K", [1280, 1536, 1600, 1672, 1792, 2056, 2560, 3072, 3200, 3584, 4096, 4104])
def test_128x96_redone_tiles_are_the_fp32_modes(K):
    """Every tile overflows (products of U(90, 140), whose FP32 sums round): the
    redo sums in the order of the kernel the FP32 mode runs at this K, two K groups
    or four; tiles of 44 rows (none in the lower half) and 58 columns."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a = (90.0 + 50.0 * torch.rand(300, K, generator=g, device="cuda")).half()
    b = (90.0 + 50.0 * torch.rand(250, K, generator=g, device="cuda")).half().t()
    c, flags = mm_flags(a, b, torch.float32, tile=TILE)
    assert bool((flags == 1).all())
    assert torch.equal(c, mm_tile(a, b, TILE, torch.float32, chunked=False))


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("K", [1536, 2560, 4096])
def test_128x96_redo_with_a_bias(K, out_dtype):
    M, N = 2040, 1530
    a, w, bias = rnd((M, K), 41).cuda(), rnd((N, K), 42).cuda(), rnd((N,), 43).cuda()
    a[256:300, 500:540] = 100.0  # tile rows 2 and 15: with these columns of b, chunks past 65504
    a[2039, 500:540] = 100.0
    w[:, 500:540] = w[:, 500:540].abs() * 0 + 50.0
    assert tile_config(a, w.t())["tile"] == TILE
    want = mm_tile(a, w.t(), TILE, out_dtype, chunked=False)[256:300]
    c = mm_bias(a, w.t(), bias, out_dtype)
    assert torch.equal(c[256:300], want + bias)
    assert torch.equal(c, f16acc.mm(a, w.t(), out_dtype) + bias)
