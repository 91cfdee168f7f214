"""The native call path (csrc/host.cpp) against the general path in kernel.py:
the same bits, type, shape and strides on every kind of operand, and None (the
general path) for the calls it leaves alone."""

import itertools

import pytest
import torch
import torch.nn.functional as F

import f16acc_amd as f16acc
from f16acc_amd import _lib, kernel, patch

pytestmark = pytest.mark.gpu
host = _lib.host


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half().cuda()


def views(rows, cols, seed):
    """[rows, cols] fp16 operands in every layout mm takes."""
    x = rnd(rows + 2, cols + 16, seed=seed)
    yield "contiguous", rnd(rows, cols, seed=seed)
    yield "transposed", rnd(cols, rows, seed=seed).t()
    yield "pitched", x[:rows, :cols]
    yield "offset", x[1:rows + 1, 3:cols + 3]
    yield "strided", rnd(2 * rows, 2 * cols, seed=seed)[::2, ::2]
    yield "broadcast rows", rnd(1, cols, seed=seed).expand(rows, cols)
    yield "broadcast columns", rnd(rows, 1, seed=seed).expand(rows, cols)


@pytest.mark.parametrize("M, N, K", [(1, 1, 1), (1, 8, 16), (130, 72, 64), (33, 257, 129), (256, 256, 1001)])
def test_native_mm_equals_general(M, N, K):
    taken = 0
    for (na, a), (nb, b) in itertools.product(views(M, K, 1), views(K, N, 2)):
        for out, chunked in ((torch.float16, True), (torch.float32, True), (torch.float16, False)):
            c = host.mm(a, b, None, out is torch.float32, chunked)
            want = kernel._mm(a, b, out, chunked)
            if c is not None:
                taken += 1
                assert c.dtype == out and c.shape == want.shape and c.stride() == want.stride()
                assert not c.requires_grad and torch.equal(c, want), (na, nb, out, chunked)
            assert torch.equal(f16acc.mm(a, b, out, chunked), want)
    assert taken > 0


def test_native_bias_and_linear_equal_general():
    f16acc.enable()
    try:
        for shape, N in (((128, 256), 96), ((3, 50, 64), 130), ((2, 2, 64, 200), 72), ((256, 129), 33)):
            x, w, b = rnd(*shape, seed=3), rnd(N, shape[-1], seed=4), rnd(N, seed=5)
            rows = x.numel() // shape[-1]
            x2 = x.reshape(rows, shape[-1])
            for bias in (None, b, rnd(2 * N, seed=6)[::2]):
                native = bias is None or bias.is_contiguous()
                with torch.no_grad():
                    y = F.linear(x, w, bias)
                    assert (host.linear(x, w, bias, patch.MIN_ROWS) is not None) == native
                    want = kernel._mm(x2, w.t(), torch.float16, True) if bias is None else kernel._mm_bias(
                        x2, w.t(), bias, torch.float16, True)
                assert y.shape == (*shape[:-1], N) and y.is_contiguous()
                assert torch.equal(y.view(rows, N), want)
                for out, chunked in ((torch.float32, True), (torch.float16, False), (torch.float32, False)):
                    c = host.mm(x2, w.t(), bias, out is torch.float32, chunked)
                    assert (c is not None) == native
                    if native and bias is not None:
                        want = kernel._mm_bias(x2, w.t(), bias, out, chunked)
                        assert c.dtype == out and torch.equal(c, want)
                        assert torch.equal(f16acc.kernel.mm_bias(x2, w.t(), bias, out, chunked), want)
    finally:
        f16acc.disable()


def test_calls_left_to_the_general_path():
    a, b, w = rnd(160, 64), rnd(64, 32), rnd(32, 64)
    none = [
        host.mm(a.cpu(), b, None, False, True), host.mm(a, b.cpu(), None, False, True),
        host.mm(a.float(), b, None, False, True), host.mm(a, a, None, False, True),
        host.mm(a[0], b, None, False, True), host.mm(a, b, rnd(31), False, True),
        host.mm(a, b, rnd(64)[::2], False, True), host.mm(a[:0], b, None, False, True),
        host.mm(a[:, :0], b[:0], None, False, True), host.mm("a", b, None, False, True), host.mm(a, b),
        host.linear(a, w, None, 161), host.linear(a, b, None, 128),
    ]
    with torch.no_grad():
        none += [host.linear(a, w, None, 161), host.linear(a.float(), w, None, 128), host.linear(a, w.float(), None, 128),
                 host.linear(a, b, None, 128), host.linear(a.view(4, 40, 64).transpose(0, 1), w, None, 128)]
        assert host.linear(a, w, None, 160) is not None
        assert host.linear(torch.nn.Parameter(a), torch.nn.Parameter(w), None, 160) is not None
    assert host.linear(a, w, None, 128) is None  # gradients enabled
    assert all(r is None for r in none)

    class Sub(torch.Tensor):
        pass

    assert host.mm(a.as_subclass(Sub), b, None, False, True) is None

    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Fn(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dp(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Fn(), Dp()):
        with mode:
            assert host.mm(a, b, None, False, True) is None
            assert torch.equal(f16acc.mm(a, b), kernel._mm(a, b, torch.float16, True))
    with pytest.raises(Exception):
        torch.func.vmap(lambda x: f16acc.mm(x, b))(a.view(4, 40, 64))


def test_native_path_on_another_stream_and_in_a_graph():
    x, w = rnd(256, 512, seed=7), rnd(256, 512, seed=8)
    want = kernel._mm(x, w.t(), torch.float16, True)
    # on s, behind work that takes milliseconds and ends by writing x: a launch on
    # another stream would read the zeros
    s = torch.cuda.Stream()
    late = torch.zeros_like(x)
    slow = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for _ in range(20):
            slow = torch.mm(slow, slow).clamp_(-1.0, 1.0)
        late.copy_(x)
        y = host.mm(late, w.t(), None, False, True)
        with torch.no_grad():
            z = host.linear(late, w, None, 128)
    assert not s.query()
    s.synchronize()
    assert torch.equal(y, want) and torch.equal(z, want)
    g = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(g):
        z = patch.linear(x, w)
    for seed in (9, 10, 11):
        x.copy_(rnd(256, 512, seed=seed))
        z.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, kernel._mm(x, w.t(), torch.float16, True))
