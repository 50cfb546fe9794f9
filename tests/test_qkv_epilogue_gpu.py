"""eet_gemm_w8a16_qkv: the split of a prompt's fused Q | K | V rows in the epilogue of the large-M product, for every block
shape, against the product and eet_qkv_split as two calls on the same block shape.  The epilogue rounds to fp16 where the
product stores and rotates that value in fp32 as the split kernel does, each result rounded once; to the bit where the
products are exact (test_same_rotation_as_the_split_kernel).  On random weights the bound leaves room for a product that one form rounds by way of
fp32 and the other directly, as the compiler likes: the same but for one in some 2^12 values, and there both inputs of a
rotation and its result are at most one unit of fp16 off, each 2^-10 of the pair's length at most and 2^-11 in the mean of
the numbers between two powers of two: bound 2^-9."""
import pytest
import torch

import eet_amd
from eet_amd._lib import check, lib

from gpu_util import gemm, stream
from test_large_m_blocks_gpu import BLOCKS

pytestmark = pytest.mark.gpu
GUARD = 7.25


def both(gpu, B, S, H, dh, K, T, rope, ws_bytes=0):
    N, M = 3 * H * dh, B * S
    g = torch.Generator().manual_seed(M + N)
    w = (torch.randn(K, N, generator=g) * 0.02).half()
    p, s = (t.to(gpu) for t in eet_amd.quant_weights(w, torch.int8))
    x = torch.randn(M, K, generator=g).half().to(gpu)
    table = eet_amd.ops._rope_table(T, dh, gpu) if rope else None
    ws = torch.zeros(max(ws_bytes, 4) // 4, dtype=torch.float32, device=gpu)

    def buffers():
        return [torch.full(shape, GUARD, dtype=torch.float16, device=gpu) for shape in
                ((B, H, S, dh), (B, H, T, dh), (B, H, T, dh))]
    want, got, qkv = buffers(), buffers(), torch.empty(M, N, dtype=torch.float16, device=gpu)
    rows = gemm(x, p, s, M, N, K)
    check(lib().eet_qkv_split(rows.data_ptr(), *(t.data_ptr() for t in want), B, S, H, dh, int(rope), -1, 0, T, stream()))
    check(lib().eet_gemm_w8a16_qkv(x.data_ptr(), p.data_ptr(), s.data_ptr(), qkv.data_ptr(), *(t.data_ptr() for t in got),
                                   table.data_ptr() if rope else None, B, S, H, dh, K, T, ws.data_ptr() if ws_bytes else None,
                                   ws_bytes, stream()))
    return want, got


@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_every_block(gpu, tuning, block):
    """Heads that end inside a block and inside a wavefront's share, ragged rows over several sequences; cache rows
    behind the prompt keep their value."""
    tm, tn, wm, wn = block
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
    for B, S, H, dh in ((3, 37, 5, 128), (1, 16 * tm * wm + 1, 3, 64), (2, 100, 3, 96), (5, 9, 7, 32)):
        for rope in (True, False):
            want, got = both(gpu, B, S, H, dh, 320, S + 3, rope)
            for name, a, b in zip("qkv", want, got):
                what = f"{block} B {B} S {S} H {H} dh {dh} rope {rope}: {name}"
                d = (a.float() - b.float()).abs()
                assert int((d != 0).sum()) <= 4 + a.numel() // 1000, what
                if rope and name != "v":
                    pair = a.float().unflatten(-1, (2, dh // 2)).norm(dim=-2).repeat(1, 1, 1, 2)
                    assert (d <= pair * 2 ** -9).all(), what
                else:
                    assert (d <= a.float().abs() * 2 ** -10).all(), what


@pytest.mark.parametrize("B,S,H,dh,K", [(1, 20, 4, 128, 512), (1, 45, 2, 128, 4096), (1, 64, 32, 128, 1024), (1, 33, 4, 32, 8192)])
def test_as_the_library_chooses(gpu, B, S, H, dh, K):
    """Few rows, and sizes at which a split of the k range or slabs of rows may be taken: within the rounding of fp32 sums
    in another order (K * 2^-24 of the summed magnitudes, here below 2^-9) and two fp16 roundings of values below 8."""
    N = 3 * H * dh
    for ws in (0, lib().eet_gemm_w8a16_workspace(B * S, N, K, 0)):
        want, got = both(gpu, B, S, H, dh, K, S, True, ws)
        for a, b in zip(want, got):
            assert float(a.float().abs().max()) < 8
            assert float((a.float() - b.float()).abs().max()) <= 2 ** -9 + 3 * 2 ** -9


def test_refused(gpu):
    x = torch.zeros(1 << 16, dtype=torch.float16, device=gpu).data_ptr()
    L = lib()
    assert L.eet_gemm_w8a16_qkv(x, x, x, x, x, x, x, None, 1, 40, 1, 48, 64, 64, None, 0, None) != 0      # head size
    assert L.eet_gemm_w8a16_qkv(x, x, x, x, x, x, x, None, 1, 40, 1, 32, 64, 39, None, 0, None) != 0      # cache rows
    assert L.eet_gemm_w8a16_qkv(x, x, x, x, None, x, x, None, 1, 40, 1, 32, 64, 64, None, 0, None) != 0   # null


@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_same_rotation_as_the_split_kernel(gpu, tuning, block):
    """Where the products are exact (small integers, scales that are powers of two) the rows, rotated or not, are those
    of the split kernel to the bit: each value rounds to fp16 once, straight from the sum of its two products."""
    tm, tn, wm, wn = block
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
    g = torch.Generator().manual_seed(tm * tn)
    for B, S, H, dh, K in ((2, 200, 4, 128, 64), (1, 333, 6, 64, 128), (3, 45, 3, 96, 64), (1, 130, 5, 32, 64)):
        N, M = 3 * H * dh, B * S
        x = torch.randint(-4, 5, (M, K), generator=g).half().to(gpu)
        p = eet_amd.pack_weights(torch.randint(-127, 128, (K, N), generator=g).to(torch.int8)).to(gpu)
        s = torch.full((N,), 2.0 ** -8, dtype=torch.float16, device=gpu)
        table = eet_amd.ops._rope_table(S, dh, gpu)
        for rope in (True, False):
            want, got = ([torch.full((B, H, S, dh), GUARD, dtype=torch.float16, device=gpu) for _ in "qkv"] for _ in range(2))
            rows, qkv = gemm(x, p, s, M, N, K), torch.empty(M, N, dtype=torch.float16, device=gpu)
            check(lib().eet_qkv_split(rows.data_ptr(), *(t.data_ptr() for t in want), B, S, H, dh, int(rope), -1, 0, S, stream()))
            check(lib().eet_gemm_w8a16_qkv(x.data_ptr(), p.data_ptr(), s.data_ptr(), qkv.data_ptr(), *(t.data_ptr() for t in got),
                                           table.data_ptr() if rope else None, B, S, H, dh, K, S, None, 0, stream()))
            for name, a, b in zip("qkv", want, got):
                assert torch.equal(a, b), f"{block} {B}x{S}x{H}x{dh} rope {rope}: {name}, {int((a != b).sum())} of {a.numel()} differ"


@pytest.mark.parametrize("B,S,H,dh,K,off", [(1, 20, 4, 128, 512, 0), (2, 100, 3, 96, 256, 0), (2, 100, 3, 96, 256, 1),
                                            (1, 33, 4, 32, 8192, 0), (1, 45, 2, 256, 4096, 0), (1, 9, 2, 320, 64, 0)])
def test_every_route_turns_by_the_given_table(gpu, B, S, H, dh, K, off):
    """Few rows, the epilogue, a table that is not 16-byte aligned, sizes that run as two launches, and a head too long for
    the split kernel's LDS: rotated by the caller's cosines and sines.  Exact products, and in fp64 the two of a rotation:
    one fp32 rounding of each factor's product and one to fp16 of a result no longer than the pair."""
    N, M = 3 * H * dh, B * S
    g = torch.Generator().manual_seed(S + dh)
    x = torch.randint(-2, 3, (M, K), generator=g).half().to(gpu)
    p = eet_amd.pack_weights(torch.randint(-127, 128, (K, N), generator=g).to(torch.int8)).to(gpu)
    s = torch.full((N,), 2.0 ** -9, dtype=torch.float16, device=gpu)
    angle = torch.arange(S)[:, None] / 500000.0 ** (torch.arange(dh // 2) / (dh // 2)) + 0.5
    store = torch.empty(S * dh + 4, device=gpu)
    table = store[off:off + S * dh].view(S, dh).copy_(torch.cat([angle.cos(), angle.sin()], 1))
    rows = gemm(x, p, s, M, N, K).view(B, S, 3, H, dh).permute(2, 0, 3, 1, 4).double()
    c, sn = (t.double().repeat(1, 2) for t in (table[:, :dh // 2], table[:, dh // 2:]))
    turned = torch.cat([-rows[..., dh // 2:], rows[..., :dh // 2]], -1) * sn + rows * c
    length = (rows ** 2 + torch.cat([rows[..., dh // 2:], rows[..., :dh // 2]], -1) ** 2).sqrt()
    for ws_bytes in (0, lib().eet_gemm_w8a16_workspace(M, N, K, 0)):
        ws = torch.zeros(max(ws_bytes, 4) // 4, dtype=torch.float32, device=gpu)
        got, qkv = [torch.full((B, H, S, dh), GUARD, dtype=torch.float16, device=gpu) for _ in "qkv"], torch.empty(M, N).half().to(gpu)
        check(lib().eet_gemm_w8a16_qkv(x.data_ptr(), p.data_ptr(), s.data_ptr(), qkv.data_ptr(), *(t.data_ptr() for t in got),
                                       table.data_ptr(), B, S, H, dh, K, S, ws.data_ptr() if ws_bytes else None, ws_bytes,
                                       stream()))
        for a, want in zip(got[:2], turned[:2]):
            assert ((a.double() - want).abs() <= length[0 if a is got[0] else 1] * (2 ** -11 + 2 ** -23) + 2 ** -25).all()
        assert torch.equal(got[2].double(), rows[2])
