"""256x256 on both sides of the lines between its kernels (chunk quads on four
waves; chunk pairs on eight): K around the chunked rule's (a half-empty last quad up
to 320) and the FP32 mode's, one round of tiles and several, ragged edges, both b
layouts.  Chunked results against the oracle; and c never decides how a and b are
summed: fp16 results are the fp32 ones rounded, on data whose FP32 sums round."""

import pytest
import torch

from f16acc_amd.kernel import mm_flags, mm_tile
from oracle import chunk32

pytestmark = pytest.mark.gpu
TILE = "256x256"


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M, N", [(300, 520), (4352, 4096), (4100, 4136)])
@pytest.mark.parametrize("K", [8, 64, 72, 136, 192, 200, 320, 328])
def test_short_k_matches_oracle(M, N, K, b_t):
    a, w = rnd((M, K), 51 + K), rnd((N, K), 52 + K)
    ga, gb = a.cuda(), w.cuda().t() if b_t else w.cuda().t().contiguous()
    ref = chunk32.chunked_sum(a, w.t().contiguous())
    c, flags = mm_flags(ga, gb, torch.float32, tile=TILE)
    assert int(flags.sum()) == 0
    # N(0, 1) data: the sums are exact, a chunk differs only where its partial,
    # summed in another order, rounds to the other binary16 neighbour
    off = (c.cpu() - ref).abs()
    chunks = -(-K // 32)
    assert float((off > 0).float().mean()) <= 1e-3 * chunks + 2 / off.numel()
    assert float(off.max()) <= 2.0 ** -5 * min(chunks, 2)


def scaled(shape, seed):
    """Values over 2^-12 .. 2^4: chunks of very different sizes, whose sum rounds."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(*shape, generator=g, device="cuda")
    return (v * torch.exp2(16.0 * torch.rand(shape[0], shape[1], generator=g, device="cuda") - 12.0)).half()


@pytest.mark.parametrize("chunked", [True, False])
@pytest.mark.parametrize("M, N, K", [(4096, 4096, 64), (4096, 4096, 320), (4096, 4096, 1024), (8192, 8192, 192),
                                     (8192, 8192, 512), (4090, 8187, 1024), (4093, 4089, 192), (4096, 4096, 2560)])
def test_c_does_not_decide_the_sums(M, N, K, chunked):
    a, b = scaled((M, K), 61), scaled((N, K), 62).t()
    c32 = mm_tile(a, b, TILE, torch.float32, chunked=chunked)
    assert torch.equal(mm_tile(a, b, TILE, torch.float16, chunked=chunked), c32.half())
    if not chunked:  # every element sums its chunks in order, whatever the kernel: 128x128's sums
        assert torch.equal(c32, mm_tile(a, b, "128x128", torch.float32, chunked=False))
