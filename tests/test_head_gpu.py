"""The fp16 output head (eet_head_f16, ops.head) against an fp32 product."""
import ctypes

import numpy as np
import pytest
import torch

from eet_amd import ops
from eet_amd._lib import check, lib


def test_argument_errors():
    buf = np.zeros(8192, np.uint8)
    p = buf.ctypes.data + (-buf.ctypes.data) % 16

    def call(x=p, stride=64, M=1, N=16, K=64):
        return lib().eet_head_f16(x, stride, p, p, M, N, K, None)
    assert call(x=None) == -1
    assert call(M=17) == -2 and call(M=0) == -2
    assert call(K=96) == -2 and call(N=24) == -2
    assert call(N=65536, K=8192, stride=8192) == -2          # more than 2^28 weights
    assert call(stride=56) == -1 and call(stride=68) == -1
    assert call(x=p + 2) == -1
    assert call(M=16, stride=1 << 27) == -1                  # rows beyond 32-bit offsets


@pytest.mark.gpu
@pytest.mark.parametrize("M,S,N,K", [(1, 1, 16, 64), (16, 3, 48, 128), (3, 1, 4096, 1024), (15, 2, 4080, 576),
                                     (8, 1, 8000, 1024), (9, 5, 28704, 448), (16, 1, 32000, 4096)])
def test_head(gpu, M, S, N, K):
    """One and several tiles per workgroup, a last workgroup with fewer, fewer k blocks than wavefronts, whole and
    broken rounds of them, the last position of several.  fp32 sums of at most 2^12 products and one rounding to fp16:
    2^-11 of the result plus 2^-12 (K * 2^-24) of the sum of magnitudes."""
    g = torch.Generator(device="cuda").manual_seed(N + K)
    h = torch.randn(M, S, K, generator=g, device=gpu).half()
    w = (torch.randn(N, K, generator=g, device=gpu) * 0.02).half()
    got = ops.head(h, w)
    assert got.shape == (M, 1, N) and got.dtype == torch.float16
    x = h[:, -1].double()
    want, size = x @ w.double().t(), x.abs() @ w.double().abs().t()
    assert ((got[:, 0].double() - want).abs() <= 2 ** -11 * want.abs() + 2 ** -12 * size * K / 2 ** 12 + 2 ** -25).all()


@pytest.mark.gpu
def test_what_stays_with_torch(gpu):
    h = torch.randn(2, 1, 64, device=gpu).half()
    w = torch.randn(32, 64, device=gpu).half()
    wide = torch.randn(17, 1, 64, device=gpu).half()
    assert torch.equal(ops.head(wide, w), torch.nn.functional.linear(wide, w))
    assert ops.head(h, w.clone().requires_grad_()).requires_grad
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert ops.head(h, w).dtype == torch.bfloat16
    odd = torch.randn(33, 64, device=gpu).half()
    assert torch.equal(ops.head(h, odd), torch.nn.functional.linear(h, odd))


@pytest.mark.gpu
def test_sizes_and_calls_that_the_kernel_does_not_have(gpu, monkeypatch):
    """Rows beyond 32-bit offsets, nothing to multiply, another current device, forward-mode and backward autograd of
    the hidden states, a tensor subclass: what torch's linear gives, as it gives it."""
    linear = torch.nn.functional.linear
    w = torch.randn(32, 64, device=gpu).half()
    long = torch.zeros(16, 1 << 21, 64, device=gpu, dtype=torch.float16)      # 16 rows 256 MiB apart
    long[:, -1] = torch.randn(16, 64, device=gpu).half()
    got = ops.head(long, w)
    assert torch.equal(got, linear(long[:, -1:], w)) and got.abs().max() > 0
    del long
    h = torch.randn(2, 3, 64, device=gpu).half()
    want = linear(h[:, -1:], w)
    for empty, weight in ((h[:0], w), (h[:, :0], w), (h, w[:0])):
        assert ops.head(empty, weight).shape == linear(empty[:, -1:], weight).shape
    calls = []
    monkeypatch.setattr(ops.torch.nn.functional, "linear", lambda *a: calls.append(1) or linear(*a))
    with monkeypatch.context() as m:
        m.setattr(ops, "_current_device", lambda: 1)
        assert torch.equal(ops.head(h, w), want) and calls == [1]
    assert ops.head(h.clone().requires_grad_(), w).requires_grad and len(calls) == 2
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(w, torch.ones_like(w))
        tangent = torch.autograd.forward_ad.unpack_dual(ops.head(h, dual)).tangent
        assert torch.equal(tangent, linear(h[:, -1:], torch.ones_like(w))) and len(calls) >= 3

    class Sub(torch.Tensor):
        pass
    assert type(ops.head(h, w.as_subclass(Sub))) is Sub
    calls.clear()
    ops.head(h, torch.nn.Parameter(w, requires_grad=False))
    assert not calls                                                        # a plain call: the kernel


def test_rule_of_the_kernel():
    """Where the product stays with the library: very long rows, the ranges of V in which it measured faster."""
    wins = ops._head_kernel_wins
    assert all(wins(B, V, K) for B in (1, 16) for V, K in ((8000, 1024), (32000, 2048), (32000, 3072), (32000, 4096),
                                                           (10240, 2048), (20480, 4096), (50272, 4096), (100352, 1536)))
    assert not any(wins(B, V, K) for B in (1, 16) for V, K in ((32000, 8192), (10240, 4096), (12288, 3072), (50272, 3072)))
    assert wins(8, 8000, 5120) and not wins(16, 8000, 5120) and wins(16, 32000, 5120)


@pytest.mark.gpu
@pytest.mark.parametrize("M,S,N,K", [(1, 1, 8016, 448),      # two tiles per workgroup, the last workgroup with one
                                     (16, 2, 6144, 1088),    # two, a broken round of k blocks
                                     (5, 1, 10256, 2048),    # four, the last with one
                                     (16, 1, 20480, 3072),   # two, several rounds of workgroups
                                     (2, 1, 18432, 4096)])   # one, several rounds
def test_tiles_per_workgroup(gpu, M, S, N, K):
    assert ops._head_kernel_takes(torch.empty(M, S, K, device=gpu, dtype=torch.float16),
                                  torch.empty(N, K, device=gpu, dtype=torch.float16))
    test_head(gpu, M, S, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,S,N,K", [(16, 1, 40960, 1024),   # one k block per wavefront and tile, less than the ring holds
                                     (5, 1, 20496, 1088),    # one or two; the last turn with one tile
                                     (9, 3, 24624, 3136),    # three or four: tiles end at either slot of the ring
                                     (1, 1, 20480, 1536), (12, 2, 40976, 2560),
                                     (16, 1, 24576, 4096)])  # the most activations that fit
def test_one_workgroup_per_cu(gpu, M, S, N, K):
    test_tiles_per_workgroup(gpu, M, S, N, K)
    h = torch.randn(M, S, K, device=gpu).half()
    w = (torch.randn(N, K, device=gpu) * 0.02).half()
    first = ops.head(h, w)
    assert all(torch.equal(first, ops.head(h, w)) for _ in range(3))


def tiles(M, N, K):
    v = ctypes.c_int(-1)
    check(lib().eet_head_f16_shape(M, N, K, ctypes.byref(v)))
    return v.value


def test_which_kernel():
    """What the sizes of the two tests above run as."""
    assert [tiles(*s) for s in ((1, 8016, 448), (16, 6144, 1088), (5, 10256, 2048))] == [2, 2, 4]
    assert all(tiles(*s) == 0 for s in ((16, 20480, 3072), (2, 18432, 4096), (16, 40960, 1024), (9, 24624, 3136), (1, 20480, 1536),
                                        (12, 40976, 2560), (16, 24576, 4096)))
    assert tiles(5, 20496, 1088) == 2
    v, L = ctypes.c_int(), lib()
    assert [L.eet_head_f16_shape(M, N, K, ctypes.byref(v)) for M, N, K in ((0, 16, 64), (17, 16, 64), (1, 24, 64), (1, 16, 96),
                                                                           (1, 1 << 20, 512))] == [-2] * 5
    assert L.eet_head_f16_shape(1, 16, 64, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("M,S,N,K,form", [(2, 1, 17632, 6144, 1), (1, 1, 20752, 2048, 2), (16, 2, 20480, 5120, 2),
                                          (16, 1, 17632, 512, 4),          # several rounds of workgroups
                                          (9, 1, 16400, 1088, 0),          # one or two k blocks per wavefront and tile, and
                                          (16, 2, 20496, 1088, 0)])        # the last turn with one tile
def test_kernel_by_size(gpu, M, S, N, K, form):
    assert tiles(M, N, K) == form
    test_one_workgroup_per_cu(gpu, M, S, N, K)


@pytest.mark.gpu
def test_parameters_without_gradients(gpu):
    """A matrix that would take gradients stays with the kernel wherever they are off."""
    h = torch.randn(2, 3, 64, device=gpu).half()
    w = torch.nn.Parameter(torch.randn(32, 64, device=gpu).half())
    with torch.no_grad():
        assert ops._head_kernel_takes(h, w)
    assert not ops._head_kernel_takes(h, w) and ops._head_kernel_takes(h, w.detach())
