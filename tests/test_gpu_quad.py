"""The chunk-quad kernel (gemm_quad: chunked 256x256) at its edges: K around
whole quads (128) and chunks, M and N around a wave's sub-tile (128) and the
tile, both b layouts, both output types, strided c; an overflow in every chunk
position of the first, a middle and the last quad; and NaN operands.

Tolerance: every sum of binary16-rounded chunks of N(0, 1) data at these K is
exact in FP32 (11-bit values, running sums within 2^13), so an element differs
from the oracle only where a chunk's FP32 partial, summed in another order, rounds
to the other binary16 neighbour: fewer than 1 in 10^3 chunks, each by at most
an ulp of the partial (2^-6 below 32, 2^-5 above)."""

import pytest
import torch

from f16acc_amd import _lib
from f16acc_amd.kernel import mm_flags, mm_tile, tile_config
from oracle import chunk32

pytestmark = pytest.mark.gpu
TILE = "256x256"


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


def on_gpu(b, b_t):
    return b.t().contiguous().cuda().t() if b_t else b.cuda()


@pytest.mark.parametrize("b_t", [True, False])
@pytest.mark.parametrize("M, N, K", [
    (1, 8, 8), (16, 128, 32), (127, 136, 40), (128, 256, 96), (129, 264, 120), (255, 248, 128), (256, 256, 136),
    (257, 392, 248), (384, 512, 256), (300, 520, 392), (513, 264, 640)])
def test_quad_edges_match_oracle(M, N, K, b_t):
    a, b = rnd((M, K), 11), rnd((K, N), 12)
    ga, gb = a.cuda(), on_gpu(b, b_t)
    ref = chunk32.chunked_sum(a, b)
    c, flags = mm_flags(ga, gb, torch.float32, tile=TILE)
    assert int(flags.sum()) == 0
    off = (c.cpu() - ref).abs()
    chunks = -(-K // 32)
    assert float((off > 0).float().mean()) <= 1e-3 * chunks + 2 / off.numel()
    assert float(off.max()) <= 2.0 ** -5 * min(chunks, 2)
    # fp16: the same sums, rounded
    assert torch.equal(mm_tile(ga, gb, TILE, torch.float16), c.half())


@pytest.mark.parametrize("out_dtype, esize", [(torch.float16, 2), (torch.float32, 4)])
def test_quad_strided_output(out_dtype, esize):
    """c with a row pitch past N (aligned and not), and column-major: the
    contiguous result, and no element around it touched."""
    M, N, K = 300, 520, 160
    a, b = rnd((M, K), 21).cuda(), rnd((K, N), 22).cuda()
    want = mm_tile(a, b, TILE, out_dtype)
    for scm, scn in ((536, 1), (523, 1), (1, 304), (1100, 2)):
        buf = torch.full((M * scm + N * scn + 8,), 7.0, device="cuda", dtype=out_dtype)
        _lib.check(_lib.gemm_tile(a.data_ptr(), b.data_ptr(), buf.data_ptr(), None, M, N, K, K, 1, N, 1, scm, scn,
                                  _lib.OUT_F16 if esize == 2 else _lib.OUT_F32, 1,
                                  torch.cuda.current_stream().cuda_stream, _lib.TILES.index(TILE)))
        view = buf.as_strided((M, N), (scm, scn))
        assert torch.equal(view, want), (scm, scn)
        view.fill_(7.0)
        assert bool((buf == 7.0).all()), (scm, scn)


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("M, N", [(4096, 4096), (4090, 8187)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_quad_column_major_output(out_dtype, M, N, biased):
    """Columns apart are stored from the registers: one round and several, a
    bias, an overflowing element (flagged, redone, stored again), edges; and the
    FP32 mode."""
    K = 520
    a, b = rnd((M, K), 23), rnd((N, K), 24)
    a[M - 3, 64:96] = 100.0
    b[N - 5, 64:96] = 100.0
    a, b = a.cuda(), b.cuda().t()
    assert tile_config(a, b)["tile"] == TILE
    bias = rnd((N,), 25).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    out = _lib.OUT_F32 if out_dtype == torch.float32 else _lib.OUT_F16

    def call(c, scm, scn, chunked):
        flags = torch.zeros(-(-M // 256), -(-N // 256), device="cuda", dtype=torch.uint8)
        args = (flags.data_ptr(), M, N, K, K, 1, 1, K, scm, scn, out, chunked, stream)
        if biased:
            _lib.check(_lib.gemm_bias(a.data_ptr(), b.data_ptr(), bias.data_ptr(), c.data_ptr(), *args))
        else:
            _lib.check(_lib.gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), *args))
        return flags

    for chunked in (1, 0):
        want = torch.empty(M, N, device="cuda", dtype=out_dtype)
        flags = call(want, N, 1, chunked)
        assert int(flags.sum()) == chunked and int(flags[-1, -1]) == chunked
        buf = torch.full((N * M + 8,), 7.0, device="cuda", dtype=out_dtype)
        assert torch.equal(call(buf, 1, M, chunked), flags)
        assert torch.equal(buf[:N * M].view(N, M).t(), want) and bool((buf[N * M:] == 7.0).all())


@pytest.mark.parametrize("b_t", [True, False])
@pytest.mark.parametrize("quad", [0, 1, 2])
@pytest.mark.parametrize("chunk", [0, 1, 2, 3])
def test_quad_overflow_in_every_chunk(quad, chunk, b_t):
    """One chunk of one element past 65504 (32 * 100 * 100 = 320000), in each
    chunk of the first, second and last (partial) quad: its tile, and only it, is
    flagged and equals the FP32-accumulating mode bit for bit."""
    M, N, K = 512, 512, 384 - 8 * (quad == 2)
    k0 = 128 * quad + 32 * chunk
    a, b = rnd((M, K), 31), rnd((K, N), 32)
    for row, col in ((0, 0), (255, 511), (383, 130)):
        aa, bb = a.clone(), b.clone()
        aa[row, k0:k0 + 32] = 100.0
        bb[k0:k0 + 32, col] = 100.0
        ga, gb = aa.cuda(), on_gpu(bb, b_t)
        c, flags = mm_flags(ga, gb, torch.float32, tile=TILE)
        want = torch.zeros(2, 2, dtype=torch.uint8)
        want[row // 256, col // 256] = 1
        if k0 + 32 > K:  # the zero-filled end of the last chunk: 24 products still overflow
            assert 24 * 1e4 > 65504
        assert torch.equal(flags.cpu(), want), (row, col)
        f32 = mm_tile(ga, gb, TILE, torch.float32, chunked=False)
        tm, tn = row // 256 * 256, col // 256 * 256
        assert torch.equal(c[tm:tm + 256, tn:tn + 256], f32[tm:tm + 256, tn:tn + 256])


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_quad_nan_and_fp16_range(out_dtype):
    """A NaN operand flags its tiles; an FP32 sum past the binary16 range whose
    chunks are all in range does not (f16acc/kernel.py:70-71 tests the FP32 sum)."""
    M, N, K = 256, 512, 256
    a, b = rnd((M, K), 41), rnd((K, N), 42)
    a[3, 17] = float("nan")
    c, flags = mm_flags(a.cuda(), b.cuda(), out_dtype, tile=TILE)
    assert flags.cpu().tolist() == [[1, 1]]
    assert bool(torch.isnan(c[3]).all()) and bool(torch.isfinite(torch.cat([c[:3], c[4:]])).all())
    a, b = torch.full((M, K), 16.0).half(), torch.full((K, N), 32.0).half()  # chunks 16384, sums 131072
    c, flags = mm_flags(a.cuda(), b.cuda(), out_dtype, tile=TILE)
    assert flags.cpu().tolist() == [[0, 0]]
    want = torch.full((M, N), 131072.0).to(out_dtype)
    assert torch.equal(c.cpu(), want)
