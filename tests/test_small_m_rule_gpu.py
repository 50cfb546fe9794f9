"""The launch shapes that small_m_us picks at channel counts without an entry of their own: which one, with a workspace and
without, and the product against the fp32 oracle."""
import ctypes

import numpy as np
import pytest
import torch

import eet_amd
from eet_amd._lib import ZEROED_WORKSPACE, check, lib
from oracle import ops as O

from gpu_util import assert_close, stream

pytestmark = pytest.mark.gpu


def shape(M, N, K, epi, rms):
    v = [ctypes.c_int(0) for _ in range(4)]
    check(lib().eet_gemm_w8a16_small_m_shape(M, N, K, epi, rms, *[ctypes.byref(x) for x in v]))
    return tuple(x.value for x in v)


# one k-tile a wavefront and less, a lone n-tile, a ragged last workgroup, wide launches, long k ranges shared by workgroups
@pytest.mark.parametrize("M,N,K,want", [(1, 16, 64, None), (1, 1024, 1024, (1, 8, 2, 1)), (8, 3088, 1024, (1, 8, 2, 1)),
                                        (2, 6144, 2048, (2, 4, 2, 1)), (1, 9216, 3072, (3, 8, 1, 1)),
                                        (9, 16400, 512, None), (32, 2048, 5632, (3, 8, 1, 4)), (16, 3072, 8192, (3, 8, 1, 4)),
                                        (17, 2064, 8256, None), (32, 12288, 1024, None)])
def test_picked_shape(gpu, M, N, K, want):
    got = shape(M, N, K, 1, 0)
    assert want is None or got == want
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn(K, N, generator=g) * 0.02).half()
    u, p, s = eet_amd.quant_weights(w, torch.int8, True)
    x, res = torch.randn(M, K, generator=g).half(), torch.randn(M, N, generator=g).half()
    ref = O.dequant_matmul(x.numpy(), u.numpy(), s.numpy())
    need = lib().eet_gemm_w8a16_zeroed_workspace(M, N, K, 1)
    assert (need > 0) == (got[3] > 1)
    ws = torch.zeros(need + 16, dtype=torch.uint8, device=gpu)
    xd, pd, sd, rd = x.to(gpu), p.to(gpu), s.to(gpu), res.to(gpu)
    for given in ({need, need - 16, 0} if need else {0}):     # a workspace too small is not looked at
        for _ in range(2):                                     # the arrival counters are zero again
            out = torch.full((M + 1, N), 7.25, dtype=torch.float16, device=gpu)
            check(lib().eet_gemm_w8a16_fused(xd.data_ptr(), pd.data_ptr(), sd.data_ptr(), out.data_ptr(), M, N, K, 1,
                                             rd.data_ptr(), None, 0.0, ws.data_ptr() if given else None, given | (ZEROED_WORKSPACE if given else 0),
                                             stream()))
            c = out.cpu()
            assert (c[M] == 7.25).all() and not ws[:32768].any()
            # the product is within 1e-2 / 1e-3 of the oracle; the fp16 sum with the residual adds half an ulp of at most 8
            assert_close(c[:M].numpy(), ref + res.numpy().astype(np.float32), atol=5e-3, what=f"{M} {N} {K} {given}")


# 4 shares, or 2, where the caller vouches for its counters; nothing to be asked for, and nothing touched, where it does not
@pytest.mark.parametrize("M,N,K", [(8, 1024, 8192), (16, 3072, 8192), (32, 2048, 5632), (32, 1040, 2112)])
def test_a_workspace_nobody_vouches_for_is_left_alone(gpu, M, N, K):
    """The caller's buffer for calls of more than 32 rows, say, whose sums lie where the arrival counters would."""
    assert lib().eet_gemm_w8a16_workspace(M, N, K, 1) == 0 and shape(M, N, K, 1, 0)[3] > 1
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn(K, N, generator=g) * 0.02).half()
    u, p, s = eet_amd.quant_weights(w, torch.int8, True)
    x, res = torch.randn(M, K, generator=g).half(), torch.randn(M, N, generator=g).half()
    want = O.dequant_matmul(x.numpy(), u.numpy(), s.numpy()) + res.numpy().astype(np.float32)
    xd, pd, sd, rd = x.to(gpu), p.to(gpu), s.to(gpu), res.to(gpu)
    ws = torch.full((1 << 23,), 1, dtype=torch.uint8, device=gpu)
    for bytes_ in (ws.numel(), (1 << 63) - 1, (1 << 64) - 1):          # a large enough size, however it is put, says nothing
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
        check(lib().eet_gemm_w8a16_fused(xd.data_ptr(), pd.data_ptr(), sd.data_ptr(), out.data_ptr(), M, N, K, 1, rd.data_ptr(),
                                         None, 0.0, ws.data_ptr(), bytes_, stream()))
        assert_close(out.cpu().numpy(), want, atol=5e-3, what=f"{M} {N} {K}")
        assert (ws == 1).all()


def test_an_operator_call_leaves_it_alone_too(gpu):
    M, hidden, d_ff = 32, 2048, 5632
    g = torch.Generator().manual_seed(7)
    w01, w2 = (torch.randint(0, 256, (n,), dtype=torch.uint8, generator=g).to(gpu) for n in (hidden * 2 * d_ff, d_ff * hidden))
    s01, s2 = ((torch.rand(n, generator=g) * 1e-4).half().to(gpu) for n in (2 * d_ff, hidden))
    x, gamma = torch.randn(M, hidden, generator=g).half().to(gpu), torch.ones(hidden, dtype=torch.float16, device=gpu)
    act = torch.empty(M, d_ff, dtype=torch.float16, device=gpu)

    def ffn(ws, nbytes):
        out = torch.full((M, hidden), float("nan"), dtype=torch.float16, device=gpu)
        check(lib().eet_gated_ffn_int8_decode(x.data_ptr(), gamma.data_ptr(), 1e-6, w01.data_ptr(), s01.data_ptr(), w2.data_ptr(),
                                              s2.data_ptr(), act.data_ptr(), out.data_ptr(), M, hidden, d_ff, 1,
                                              ws.data_ptr() if ws is not None else None, nbytes, stream()))
        return out
    dirty = torch.full((1 << 23,), 1, dtype=torch.uint8, device=gpu)
    assert torch.equal(ffn(dirty, dirty.numel()), ffn(None, 0)) and (dirty == 1).all()
    need = lib().eet_gemm_w8a16_zeroed_workspace(M, hidden, d_ff, 1)
    ws = torch.zeros(need, dtype=torch.uint8, device=gpu)
    split = ffn(ws, need | ZEROED_WORKSPACE)
    assert ws[32768:].any() and not ws[:32768].any()                   # it was used, and can be used again
    assert_close(split.cpu().numpy(), ffn(None, 0).float().cpu().numpy(), what="4 shares and one")


@pytest.mark.parametrize("hidden,d_ff", [(2048, 5632), (4096, 11008)])
def test_recorded_first_then_called(gpu, hidden, d_ff):
    """An op whose first call is recorded into a graph, with no eager call ahead, and is called before the first replay: the
    counters of a buffer that the graph alone would zero are not used.  (Split and unsplit products round to neighbouring fp16
    values, 2^-8 apart below 8.)"""
    from eet_amd import ops
    M, g, e = 32, torch.Generator(device=gpu).manual_seed(11), torch.empty(0)
    desc = ops.MetaDesc(dtype=torch.float16, batch_size=M, head_num=hidden // 128, hidden_units=hidden, layer_num=1, max_seq_len=1,
                        max_full_seq_len=8, activation_fn="silu", d_ff=d_ff, cuda_device="cuda:0", is_int8=True)
    mats = [ops.quant_weights_device(torch.randn(k, n, generator=g, device=gpu).half() * 0.02)
            for k, n in ((hidden, d_ff), (hidden, d_ff), (d_ff, hidden))]
    ffn = ops.GatedFeedForwardNetworkInt8(desc, *mats[0], e, *mats[1], e, *mats[2], e,
                                          torch.ones(hidden, dtype=torch.float16, device=gpu), e)
    x = torch.randn(M, 1, hidden, generator=g, device=gpu).half()
    want = ffn.forward(x, True, True).clone()
    other = ffn.forward(x * 2, True, True).clone()
    torch.cuda.synchronize()
    ops.workspaces.clear()
    pool, filler, graph = torch.cuda.graph_pool_handle(), torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(filler, pool=pool):      # memory that another graph of the program has used before
        junk = torch.full((1 << 25,), 77, dtype=torch.int32, device=gpu)
    filler.replay()
    torch.cuda.synchronize()
    del junk
    with torch.cuda.graph(graph, pool=pool):
        recorded = ffn.forward(x, True, True)
    got = ffn.forward(x * 2, True, True)
    assert_close(got.float().cpu().numpy(), other.float().cpu().numpy(), atol=5e-3, what="before the first replay")
    for _ in range(3):
        recorded.fill_(float("nan"))
        graph.replay()
        assert_close(recorded.float().cpu().numpy(), want.float().cpu().numpy(), atol=5e-3, what="replay")
        assert_close(ffn.forward(x * 2, True, True).float().cpu().numpy(), other.float().cpu().numpy(), atol=5e-3, what="eager, between")
    del recorded, got
    ops.workspaces.clear()        # the graph's own memory goes with it
