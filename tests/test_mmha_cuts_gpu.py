"""How a decode-attention launch of few (b, h) pairs is cut: the cut that is estimated to be the fastest where the workspace
allows it, the usual one where it does not; every cut against the fp32 oracle."""
import numpy as np
import pytest
import torch

from eet_amd._lib import lib
from oracle import ops as O

from gpu_util import assert_close, stream

pytestmark = pytest.mark.gpu


def records(B, H, dh, nbytes):
    return nbytes // (B * H * (dh + 2) * 4)


# splits of a short cache, of pairs that do not divide 256, more splits than the usual, none; the shortest steps; head size 32
@pytest.mark.parametrize("B,H,dh,step,usual,best", [(1, 32, 128, 200, 0, 8), (1, 32, 128, 513, 2, 8), (4, 40, 128, 3001, 2, 8),
                                                    (8, 40, 128, 2048, 0, 4), (2, 7, 96, 1030, 4, None), (16, 16, 64, 1000, 0, 0),
                                                    (1, 3, 32, 255, 0, None), (1, 1, 64, 1, 0, 0), (1, 1, 128, 31, 0, 0)])
@pytest.mark.parametrize("padded", [False, True])
def test_cut_by_estimate(gpu, B, H, dh, step, usual, best, padded):
    L, cap = lib(), step + 2
    need = L.eet_mmha_decode_workspace(B, H, dh, step)
    assert best is None or records(B, H, dh, need) == best
    g = torch.Generator().manual_seed(step + B)
    kc, vc = (torch.randn(B, H, cap, dh, generator=g).half() for _ in range(2))
    q, k, v = (torch.randn(B, H, dh, generator=g).half() for _ in range(3))
    # padding that leaves some cuts without a row, a whole sequence of it and none
    pad = torch.tensor([(step, 0, step - 1, step // 3)[b % 4] for b in range(B)]) if padded else None
    kcn, vcn = kc.numpy().copy(), vc.numpy().copy()
    want = O.decode_attention(q.numpy(), k.numpy(), v.numpy(), kcn, vcn, step, pad.numpy() if padded else None, None)
    qd, kd, vd, padd = q.to(gpu), k.to(gpu), v.to(gpu), pad.to(gpu) if padded else None
    least = usual * B * H * (dh + 2) * 4
    ws = torch.full((max(need, least) + 64,), 255, dtype=torch.uint8, device=gpu)

    def run(given):
        ws.fill_(255)
        kcd, vcd = kc.to(gpu), vc.to(gpu)
        ctx = torch.empty(B, H * dh, dtype=torch.float16, device=gpu)
        rc = L.eet_mmha_decode(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), 0, kcd.data_ptr(), vcd.data_ptr(), ctx.data_ptr(),
                               None, padd.data_ptr() if padded else None, B, H, dh, step, cap, None,
                               ws.data_ptr() if given else None, given, stream())
        return rc, ctx.cpu(), kcd.cpu(), vcd.cpu()
    whole = run(need)
    for given in sorted({need, need + 64, max(need - 4, least), least}):
        rc, ctx, kcd, vcd = run(given)
        assert rc == 0
        assert_close(ctx.numpy(), want, what=f"{given} of {need} bytes")
        assert np.array_equal(kcd.numpy(), kcn) and np.array_equal(vcd.numpy(), vcn)
        assert given < need or torch.equal(ctx, whole[1])         # more memory than asked for changes nothing
        assert (ws[given:] == 255).all()
    if least:
        assert run(least - 4)[0] == -4                             # what the usual cut needs is asked for as ever


# the three that a workspace of their own splits although they can do without one
@pytest.mark.parametrize("B,H,dh,step", [(1, 32, 128, 200), (18, 16, 64, 1300), (9, 32, 96, 1000)])
def test_static_array_is_for_calls_that_need_a_workspace(gpu, B, H, dh, step):
    """Two streams may run such calls side by side: a launch that shares the array has the sums of other cuts."""
    L, cap = lib(), step + 2
    assert records(B, H, dh, L.eet_mmha_decode_workspace(B, H, dh, step)) > 1
    g = torch.Generator().manual_seed(step)
    kc, vc = (torch.randn(B, H, cap, dh, generator=g).half().to(gpu) for _ in range(2))
    q, k, v = (torch.randn(B, H, dh, generator=g).half().to(gpu) for _ in range(3))

    def run(fn, *ws):
        ctx = torch.empty(B, H * dh, dtype=torch.float16, device=gpu)
        assert fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), 0, kc.data_ptr(), vc.data_ptr(), ctx.data_ptr(), None, None, B, H, dh,
                  step, cap, None, *ws, stream()) == 0
        return ctx
    own = torch.empty(L.eet_mmha_decode_workspace(B, H, dh, step), dtype=torch.uint8, device=gpu)
    got, alone = run(L.eet_mmha_decode_static), run(L.eet_mmha_decode, None, 0)
    split = run(L.eet_mmha_decode, own.data_ptr(), own.numel())
    assert torch.equal(got, alone) and not torch.equal(got, split)
