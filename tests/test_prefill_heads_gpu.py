"""The prompt attention of head sizes 64 and 96 through the DMA kernel, both launch shapes, at the edges of a query
tile, a key chunk, a wavefront's pair of tiles and a query block, against the fp32 oracle; and the register-staged
kernel that keeps what the DMA cannot address."""
import pytest
import torch

from eet_amd._lib import check, lib
from gpu_util import assert_close, stream
import test_glue_gpu as glue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [1, 2])
@pytest.mark.parametrize("dh", [64, 96])
@pytest.mark.parametrize("S,use_pad,use_alibi", [(1, False, False), (15, True, False), (17, False, False), (64, False, True),
                                                 (65, True, False), (128, True, True), (129, False, False),
                                                 (256, False, True), (258, True, True), (511, True, False)])
def test_launch_shapes(gpu, tuning, shape, dh, S, use_pad, use_alibi):
    tuning("EET_PREFILL_SHAPE", shape)
    glue.test_prefill_attention(gpu, 2, 3, S, dh, use_pad, use_alibi)


@pytest.mark.parametrize("dh", [64, 96])
@pytest.mark.parametrize("S,use_alibi", [(300, False), (131, True), (130, True)])
def test_register_staged_kernel(gpu, tuning, dh, S, use_alibi):
    tuning("EET_PREFILL_LEGACY", 1)
    glue.test_prefill_attention(gpu, 2, 3, S, dh, True, use_alibi)


@pytest.mark.parametrize("B,H,S,dh", [(1, 32, 1537, 64), (8, 8, 1600, 96), (1, 5, 1700, 128)])
def test_rule_beyond_1536_tokens(gpu, B, H, S, dh):
    """One round of wide blocks and less, and nearly two: narrow blocks run."""
    glue.test_prefill_attention(gpu, B, H, S, dh, B > 1 and B <= 2, False)


def run(q, k, v, pad, slopes):
    """(ctx, its float64 value) of a causal prompt, both [B, S, H * dh]; ctx starts as NaN."""
    B, H, S, dh = q.shape
    j = torch.arange(S, device=q.device)
    row = (slopes[:, None] * j.float()).half() if slopes is not None else None
    ctx = torch.full((B, S, H * dh), float("nan"), dtype=torch.float16, device=q.device)
    check(lib().eet_prefill_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), ctx.data_ptr(),
                                      row.data_ptr() if row is not None else None,
                                      pad.data_ptr() if pad is not None else None, B, H, S, dh, S, stream()))
    want = torch.zeros(B, S, H, dh, dtype=torch.float64, device=q.device)
    scale = float(torch.tensor(dh ** -0.5).half())
    for b in range(B):
        p = int(pad[b]) if pad is not None else 0
        for h in range(H):
            s = (q[b, h].double() @ k[b, h].double().t().contiguous()) * scale
            if row is not None:
                s = s + row[h].double()
            s = s.masked_fill((j[None] > j[:, None]) | (j[None] < p), float("-inf"))[p:]
            want[b, p:, h] = torch.softmax(s, -1) @ v[b, h].double()       # rows of the padding: zero
    return ctx, want.view(B, S, H * dh)


def rnd(gpu, seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(*shape, generator=g, device=gpu).half() for _ in range(3)]


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("B,H,S,use_pad,use_alibi", [(2, 32, 2048, False, False), (2, 32, 1999, True, False),
                                                     (3, 21, 1822, True, True), (1, 61, 1794, False, True)])
def test_rule_takes_wide_blocks(gpu, dh, B, H, S, use_pad, use_alibi):
    """Two whole and two nearly whole rounds of 256-query blocks over 1536 tokens, where the rule itself launches them,
    in the grouped order that launches of this size get: ragged last blocks, padding, bias."""
    blocks = B * H * -(-S // 256)
    rounds = -(-blocks // 256)
    assert S > 1536 and rounds >= 2 and blocks * 10 >= rounds * 256 * 9
    pad = torch.tensor([0, 70, 777][:B], device=gpu) if use_pad else None
    slopes = torch.linspace(0.002, 0.3, H, device=gpu) if use_alibi else None
    got, want = run(*rnd(gpu, S, B, H, S, dh), pad, slopes)
    assert_close(got.cpu().numpy(), want.cpu().numpy(), what="wide blocks")


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("group", [-1, 1, 5])
def test_wide_blocks_in_every_order(gpu, tuning, dh, group):
    """Every (pair, query block) is taken once, whatever the order, by blocks of 256 queries as well: seven of them, the
    last one ragged, and pairs that a group does not divide."""
    tuning("EET_PREFILL_SHAPE", 2)
    tuning("EET_PREFILL_GROUP", group)
    got, want = run(*rnd(gpu, dh, 2, 7, 1601, dh), torch.tensor([0, 300], device=gpu), None)
    assert_close(got.cpu().numpy(), want.cpu().numpy(), what=f"group {group}")
