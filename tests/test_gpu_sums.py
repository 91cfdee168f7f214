"""What every block of a large result holds, each against its own size: in an
overflow stress result the clean blocks their rounded chunks' sums and the redone
ones the plain product, which is 10^6 times larger; and over a ragged-round cut
the sums of the single grid."""

import ctypes

import pytest
import torch

import f16acc_amd as f16acc
from f16acc_amd import _lib
from f16acc_amd.kernel import mm_flags, mm_tile, tile_config

pytestmark = pytest.mark.gpu


def chunk_sums(a, b):
    """Rounded chunk sums and the sum of their magnitudes, in 64 bits."""
    total = torch.zeros(a.shape[0], b.shape[1], dtype=torch.float64, device=a.device)
    mags = torch.zeros_like(total)
    af, bf = a.float(), b.float().contiguous()
    for k in range(0, a.shape[1], 32):
        part = torch.mm(af[:, k:k + 32].contiguous(), bf[k:k + 32].contiguous()).half().double()
        total += part
        mags += part.abs()
    return total, mags


def tiles(x, t=256):
    M, N = x.shape
    return x.reshape(M // t, t, N // t, t).permute(0, 2, 1, 3).reshape(M // t, N // t, t * t)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M, N, K", [
    (4096, 4096, 4096),  # one round: the redo launch
    (4096, 4096, 1024),  # one round, redone in place
    (8192, 4096, 1024),  # two rounds, in place
])
def test_every_tile_of_an_overflow_stress_result(M, N, K, b_t):
    """About 22 % of the 128-wide row and column blocks ~ U(200, 255): tiles that
    hold an intersection are redone, the others hold their chunks' sums, 10^6
    times smaller: each tile against its own norm.  (5e-6 on clean data in
    fp32; a chunk whose partial rounds to the other neighbour moves it by 2^-11.)"""
    g = torch.Generator(device="cuda").manual_seed(11)
    a = torch.randn(M, K, generator=g, device="cuda").half()
    b = torch.randn(K, N, generator=g, device="cuda").half()
    hot = torch.zeros(M // 256, N // 256, dtype=torch.bool, device="cuda")
    rows = torch.randperm(M // 128, generator=g, device="cuda")[:round(0.22 * M / 128)].tolist()
    cols = torch.randperm(N // 128, generator=g, device="cuda")[:round(0.22 * N / 128)].tolist()
    for r in rows:
        a[128 * r:128 * r + 128] = (200.0 + 55.0 * torch.rand(128, K, generator=g, device="cuda")).half()
    for c in cols:
        b[:, 128 * c:128 * c + 128] = (200.0 + 55.0 * torch.rand(K, 128, generator=g, device="cuda")).half()
    for r in rows:
        for c in cols:
            hot[r // 2, c // 2] = True
    b = b.t().contiguous().t() if b_t else b
    assert tile_config(a, b)["tile"] == "256x256"
    got = f16acc.mm(a, b, torch.float32)
    _, flags = mm_flags(a, b, torch.float32)
    assert torch.equal(flags.bool(), hot) and 0 < int(hot.sum()) < hot.numel()
    plain = torch.mm(a.double(), b.double().contiguous())
    sums, _ = chunk_sums(a, b)
    want = torch.where(hot.repeat_interleave(256, 0).repeat_interleave(256, 1), plain, sums)
    off, size = tiles(got.double() - want).norm(dim=2), tiles(want).norm(dim=2)
    assert float((off / size).max()) < 2e-5
    redone = hot.repeat_interleave(256, 0).repeat_interleave(256, 1)
    assert torch.equal(got[redone], f16acc.mm(a, b, torch.float32, chunked=False)[redone])


@pytest.mark.parametrize("rows", [False, True])
def test_a_cut_sums_what_the_single_grid_sums(rows):
    """2048 x 8960 x 1536 with a row-major b (and its transpose) runs as a round of
    256x256 and a second launch.  On data whose FP32 sums round: in FP32 mode,
    where every kernel but the K-group ones adds the chunks one after another, the
    single grid's bits; chunked, where 256x256 adds four at a time, within the
    rounding of that many FP32 additions of the sum of the exact sum of rounded
    chunks."""
    M, N, K = (8960, 2048, 1536) if rows else (2048, 8960, 1536)
    g = torch.Generator(device="cuda").manual_seed(12)

    def scaled(m, n):
        v = torch.randn(m, n, generator=g, device="cuda")
        return (v * torch.exp2(16.0 * torch.rand(m, n, generator=g, device="cuda") - 12.0)).half()

    a, b = scaled(M, K), scaled(K, N)
    cut = ctypes.c_int64()
    _lib.check(_lib.tail_split(M, N, K, K, 1, N, 1, a.data_ptr(), b.data_ptr(), ctypes.byref(cut)))
    assert cut.value == (-8192 if rows else 8192)
    full = f16acc.mm(a, b, torch.float32, chunked=False)
    assert torch.equal(full, mm_tile(a, b, "128x128", torch.float32, chunked=False))
    c = f16acc.mm(a, b, torch.float32)
    sums, mags = chunk_sums(a, b)
    # K / 32 additions, each within half an ulp of a running sum that stays below
    # mags; and partials of the wrong neighbour (an ulp of 2^-10 of the largest
    # chunk) on few elements
    off = (c.double() - sums).abs()
    close = off <= (K // 32) * 2.0 ** -24 * mags
    assert float(close.double().mean()) > 1 - 1e-3 * K / 32
    assert bool((off <= 2.0 ** -10 * mags).all())
