"""Every block shape of the large-M kernel at the sizes where it can go wrong, through the C ABI against the fp32
oracle: one row, one row less and one row more than a block; channels that end inside a block and inside a
wavefront's share of it; k loops of 1 .. 2 D + 1 k-tiles (D <= 5 stages: prologue longer than the loop, whole turns
of the ring, every length of the tail)."""
import numpy as np
import pytest
import torch

import eet_amd
from eet_amd.ops import interleave_gate_up
from oracle import ops as O

from gpu_util import gemm, gemm_fused

pytestmark = pytest.mark.gpu

# m-tiles, n-tiles of a wavefront, wavefronts down and across a block
BLOCKS = [(2, 1, 1, 4), (2, 2, 1, 4), (4, 1, 1, 4), (4, 2, 1, 4), (4, 3, 1, 4), (4, 4, 1, 4), (6, 1, 1, 4), (6, 2, 1, 4),
          (6, 3, 1, 4), (6, 4, 1, 4), (8, 2, 1, 4), (8, 3, 1, 4), (8, 4, 1, 4), (4, 2, 1, 8), (4, 2, 2, 4), (4, 5, 2, 4),
          (6, 1, 1, 8), (6, 2, 1, 8), (8, 2, 1, 8), (8, 4, 2, 4)]
GUARD = 7.25


def quant(K, N, seed):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(K, N, generator=g) * 0.02).half()
    return eet_amd.quant_weights(w, torch.int8, True)


def bound(x, u, s):
    """|error| of one product: fp32 accumulation in any order (K roundings of partial sums that sum |a w| bounds), one
    fp32 rounding by the scale; the caller adds the fp16 rounding of the result."""
    a, w = np.abs(x.numpy().astype(np.float32)), np.abs(u.numpy().astype(np.float32)) * s.numpy().astype(np.float32)
    mag = a @ w
    return mag * (x.shape[1] + 2) * 2.0 ** -24


def check(got, x, u, s, what):
    ref = x.numpy().astype(np.float64) @ (u.numpy().astype(np.float64) * s.numpy().astype(np.float64))
    tol = bound(x, u, s) + np.abs(ref) * 2.0 ** -11 + 2.0 ** -24
    err = np.abs(got.float().numpy() - ref)
    assert (err <= tol).all(), f"{what}: {int((err > tol).sum())} of {err.size} outside, max err {err.max():.2e}"


@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_block_edges(gpu, tuning, block):
    tm, tn, wm, wn = block
    bm, bn = 16 * tm * wm, 16 * tn * wn
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
    for i, k_tiles in enumerate(range(1, 12)):
        M = max(33, (bm - 1, bm, bm + 1)[i % 3])
        N = (bn, bn + 16, 2 * bn - 16, 16 * max(tn - 1, 1))[i % 4]
        u, p, s = quant(64 * k_tiles, N, i)
        x = torch.randn(M, 64 * k_tiles, generator=torch.Generator().manual_seed(M)).half()
        check(gemm(x.to(gpu), p.to(gpu), s.to(gpu), M, N, 64 * k_tiles).cpu(), x, u, s, f"{block} {M}x{N} k {k_tiles}")


@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_block_epilogues(gpu, tuning, block):
    """Residual, SwiGLU and a k range in uneven shares; nothing is written past the last row (the next rows of the
    buffer keep their value) and a residual of infinities past the last row is not read into the result."""
    tm, tn, wm, wn = block
    bm = 16 * tm * wm
    M, K, F = bm + 1 if bm > 32 else 35, 448, 16 * tn * wn + 48
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).half()
    u, p, s = quant(K, F, 5)
    xd, pd, sd = x.to(gpu), p.to(gpu), s.to(gpu)
    res = torch.full((M + 16, F), float("inf")).half()
    res[:M] = torch.randn(M, F, generator=torch.Generator().manual_seed(4))
    plain = gemm(xd, pd, sd, M, F, K).cpu()
    assert torch.equal(gemm_fused(xd, pd, sd, M, F, K, 1, res.to(gpu)).cpu(), plain + res[:M])
    out = torch.full((M + 16, F), GUARD, dtype=torch.float16, device=gpu)
    eet_amd.ops._gemm(xd, pd, sd, out, M, F, K)
    assert torch.equal(out[:M].cpu(), plain) and (out[M:] == GUARD).all()
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},3,{wm},{wn}")
    check(gemm(xd, pd, sd, M, F, K, ws_min_bytes=3 * M * F * 4).cpu(), x, u, s, f"{block} in three shares")
    if tn % 2:
        return
    tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
    uu, pu, su = quant(K, F, 6)
    w01, s01 = (t.to(gpu) for t in interleave_gate_up(p, s, pu, su))
    out = torch.full((M + 16, F), GUARD, dtype=torch.float16, device=gpu)
    eet_amd.ops._gemm(xd, w01, s01, out, M, 2 * F, K, 2)
    want = O.swiglu(O.dequant_matmul(x.numpy(), u.numpy(), s.numpy()), O.dequant_matmul(x.numpy(), uu.numpy(), su.numpy()))
    got = out[:M].cpu().float().numpy()
    # gate and up are rounded to fp16 (2^-11 of each) before the product: |d(silu)| <= 1.1 |d gate|, plus one rounding
    g = np.abs(O.dequant_matmul(x.numpy(), u.numpy(), s.numpy()).astype(np.float32))
    v = np.abs(O.dequant_matmul(x.numpy(), uu.numpy(), su.numpy()).astype(np.float32))
    eg, eu = bound(x, u, s) + g * 2.0 ** -10, bound(x, uu, su) + v * 2.0 ** -10
    tol = 1.1 * eg * v + g * eu + 1.1 * eg * eu + np.abs(want.astype(np.float32)) * 2.0 ** -10 + 2.0 ** -24
    err = np.abs(got - want.astype(np.float32))
    assert (err <= tol).all(), f"{block}: max err {err.max():.2e}"
    assert (out[M:] == GUARD).all()


@pytest.mark.parametrize("M,K,N", [(33, 3072, 288), (48, 3136, 544), (63, 6144, 1056), (64, 8192, 96)])
def test_slabs_of_32_rows(gpu, M, K, N):
    """The calls of up to 64 rows that run on the small-M kernel: every epilogue, an odd last slab, and a workspace too
    small for a split, whose bytes are not looked at."""
    import ctypes
    from eet_amd._lib import check as ok, lib
    v = [ctypes.c_int() for _ in range(5)]
    for epi in (0, 1, 2):
        ok(lib().eet_gemm_w8a16_large_m_shape(M, N, K, epi, 4096, *[ctypes.byref(x) for x in v]))
        assert v[0].value == 0
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).half()
    u, p, s = quant(K, N, 5)
    xd, pd, sd = x.to(gpu), p.to(gpu), s.to(gpu)
    dirty = torch.full((4096,), 255, dtype=torch.uint8, device=gpu)

    def run(w, scale, n_out, epi, res=None):
        out = torch.full((M + 16, n_out), GUARD, dtype=torch.float16, device=gpu)
        ok(lib().eet_gemm_w8a16_fused(xd.data_ptr(), w.data_ptr(), scale.data_ptr(), out.data_ptr(), M, w.shape[1], K, epi,
                                      res.data_ptr() if res is not None else None, None, 0.0, dirty.data_ptr(), 4096,
                                      torch.cuda.current_stream().cuda_stream))
        assert (out[M:] == GUARD).all() and (dirty == 255).all()
        return out[:M].cpu()
    plain = run(pd, sd, N, 0)
    check(plain, x, u, s, f"{M}x{N} k {K}")
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(4)).half()
    assert torch.equal(run(pd, sd, N, 1, res.to(gpu)), plain + res)
    F = N // 2
    w01, s01 = (t.to(gpu) for t in interleave_gate_up(*quant(K, F, 6)[1:], *quant(K, F, 7)[1:]))
    got = run(w01, s01, F, 2)
    halves = run(w01, s01, N, 0).view(M, F // 16, 2, 16).float()             # gate and up tiles in turn
    gate, up = halves[:, :, 0].reshape(M, F), halves[:, :, 1].reshape(M, F)
    # the launch of this epilogue has a shape of its own and sums in its own order, so its gate and up may be rounded to
    # the neighbouring fp16 value (2^-10 of each): |d(silu)| <= 1.1 |d gate|, then one rounding of the product
    want = up * gate / (1 + torch.exp(-gate))
    tol = 2.0 ** -10 * (1.1 * gate.abs() * up.abs() + 2 * want.abs()) + 2.0 ** -23
    assert ((got.float() - want).abs() <= tol).all()


@pytest.mark.parametrize("shares", [2, 3, 4, 5, 6, 7, 8])
def test_shares_of_the_k_range(gpu, tuning, shares):
    """The reduce kernel at every number of shares, those it is compiled for and the others, with each epilogue."""
    M, K, F = 37, 64 * 17, 112
    tuning("EET_GEMM_LARGE_M_TILE", f"4,2,{shares},1,4")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(shares)).half()
    u, p, s = quant(K, F, 11)
    room = shares * M * 2 * F * 4
    plain = gemm(x.to(gpu), p.to(gpu), s.to(gpu), M, F, K, ws_min_bytes=room).cpu()
    check(plain, x, u, s, f"{shares} shares")
    res = torch.randn(M, F, generator=torch.Generator().manual_seed(1)).half()
    assert torch.equal(gemm_fused(x.to(gpu), p.to(gpu), s.to(gpu), M, F, K, 1, res.to(gpu), ws_min_bytes=room).cpu(), plain + res)
    u2, p2, s2 = quant(K, F, 12)
    w, sc = interleave_gate_up(p.to(gpu), s.to(gpu), p2.to(gpu), s2.to(gpu))
    up = gemm(x.to(gpu), p2.to(gpu), s2.to(gpu), M, F, K, ws_min_bytes=room).cpu().float()
    got = gemm_fused(x.to(gpu), w, sc, M, 2 * F, K, 2, None, ws_min_bytes=room).cpu().float()
    want = up * plain.float() / (1 + torch.exp(-plain.float()))
    # gate, up and the result are each rounded to fp16 once (2^-11), gate and up perhaps to the neighbouring value where
    # one form rounds by way of fp32; gate enters with at most 1 + |gate| < 6 times its error
    assert float(plain.abs().max()) < 5
    assert ((got - want).abs() <= want.abs() * (2 ** -11 + 2 ** -10 + 6 * 2 ** -10) + 2 ** -24).all()


@pytest.mark.parametrize("shares", [1, 3])
def test_swiglu_does_not_depend_on_the_batch(gpu, tuning, shares):
    """A row's SwiGLU is the same number, to the bit, in a batch of 32 rows (small-M kernel) and in a larger one: the
    rounded fp32 quotient in both.  Products of small integers under powers of two, so that every sum is exact."""
    M, K, F = 100, 64 * shares, 4096
    g = torch.Generator().manual_seed(shares)
    x = torch.randint(-4, 5, (M, K), generator=g).half().to(gpu)
    (p, s), (pu, su) = ((eet_amd.pack_weights(torch.randint(-127, 128, (K, F), generator=g).to(torch.int8)).to(gpu),
                         torch.full((F,), 2.0 ** -8, dtype=torch.float16, device=gpu)) for _ in range(2))
    w, sc = interleave_gate_up(p, s, pu, su)
    want = torch.cat([gemm_fused(rows.contiguous(), w, sc, len(rows), 2 * F, K, 2) for rows in x.split(32)])
    for tm, tn, wm, wn in [b for b in BLOCKS if b[1] % 2 == 0]:
        tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},{shares},{wm},{wn}")
        got = gemm_fused(x, w, sc, M, 2 * F, K, 2, None, ws_min_bytes=shares * M * 2 * F * 4)
        assert torch.equal(got, want), f"{tm}x{tn}x{wm}x{wn}: {int((got != want).sum())} of {got.numel()} differ"


def test_products_round_alike_in_every_block(gpu, tuning):
    """A product is rounded to fp32 and then to fp16, whatever the block: with exact sums (integers below 2^24) the rows are
    those of the formula to the bit, at any scale.  SwiGLU takes gate and up rounded at once: the same rows from every
    block."""
    M, K, N = 1000, 64, 8192
    g = torch.Generator().manual_seed(1)
    x = torch.randint(-2047, 2048, (M, K), generator=g).half()
    q = torch.randint(-127, 128, (K, N), generator=g).to(torch.int8)
    s = (torch.rand(N, generator=g) * 0.01 + 1e-3).half()
    want = ((x.float() @ q.float()) * s.float()).half()
    xd, pd, sd, small = x.to(gpu), eet_amd.pack_weights(q).to(gpu), s.to(gpu), (s / 1024).to(gpu)
    wrong, first = {}, None
    for block in BLOCKS:
        tm, tn, wm, wn = block
        tuning("EET_GEMM_LARGE_M_TILE", f"{tm},{tn},1,{wm},{wn}")
        wrong[block] = int((gemm(xd, pd, sd, M, N, K).cpu() != want).sum())
        if tn % 2 == 0:
            got = gemm_fused(xd, pd, small, M, N, K, 2)      # neighbouring tiles of 16 channels as gate and up
            first = got if first is None else first
            wrong[block] += int((got != first).sum())
    assert not any(wrong.values()), {block: n for block, n in wrong.items() if n}
