"""The 128x96 K-group kernel (each wave a quarter of K) where its schedule can
go wrong: K around whole quads and around one quad per wave, ragged tiles,
both output types and modes."""

import pytest
import torch

from f16acc_amd.kernel import mm_flags, mm_tile, tile_config
from oracle import chunk32

pytestmark = pytest.mark.gpu
TILE = "128x96k2"


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


@pytest.mark.parametrize("M, N", [(128, 96), (129, 97), (120, 200)])
@pytest.mark.parametrize("K", [8, 120, 128, 136, 384, 504, 512, 520, 640, 1032, 1160, 2568])
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
