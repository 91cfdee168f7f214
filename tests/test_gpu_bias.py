"""The fused bias on every store: loaded whole tiles at a time at any 2-byte
alignment, element by element at the edge of N; against mm(a, b) + bias."""

import pytest
import torch

import f16acc_amd as f16acc
from f16acc_amd.kernel import mm_bias, tile_config

pytestmark = pytest.mark.gpu
TILE = "128x96k2"


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


@pytest.mark.parametrize("M, N", [(1536, 1536), (1530, 1531)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_bias_equals_the_unfused_sum(M, N, out_dtype):
    K = 136
    a, w = rnd((M, K), 1).cuda(), rnd((N, K), 2).cuda()
    bias = rnd((N + 1,), 3).cuda()[1:]  # 2-byte aligned only
    assert tile_config(a, w.t())["tile"] == TILE
    y = f16acc.mm(a, w.t(), out_dtype)
    assert torch.equal(mm_bias(a, w.t(), bias, out_dtype), y + bias)


@pytest.mark.parametrize("M, N, K, rm", [(128, 256, 256, False), (300, 517, 264, False), (1024, 1000, 512, True),
                                         (512, 384, 8960, True), (2048, 8960, 128, False), (512, 520, 65, False)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_bias_on_the_other_tiles(M, N, K, rm, out_dtype):
    """64x32, 64x64, 128x128 and its K split, 256x288, operands read in place."""
    a, w = rnd((M, K), 4).cuda(), rnd((N, K), 5).cuda()
    b = w.t().contiguous() if rm else w.t()
    bias = rnd((N + 1,), 6).cuda()[1:]
    y = f16acc.mm(a, b, out_dtype)
    assert torch.equal(mm_bias(a, b, bias, out_dtype), y + bias)


@pytest.mark.parametrize("M, N, K, rm", [(512, 384, 8960, True), (1024, 1000, 8192, False), (1000, 1024, 512, True),
                                         (2048, 1536, 136, False), (2048, 1536, 3584, False)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_bias_in_the_fp32_mode(M, N, K, rm, out_dtype):
    """chunked=False: K splits (the bias added by their finishing launch), 64x64,
    128x96."""
    a, w = rnd((M, K), 7).cuda(), rnd((N, K), 8).cuda()
    b = w.t().contiguous() if rm else w.t()
    bias = rnd((N + 1,), 9).cuda()[1:]
    y = f16acc.mm(a, b, out_dtype, chunked=False)
    assert torch.equal(mm_bias(a, b, bias, out_dtype, chunked=False), y + bias)
