"""The prompt attention of head sizes 64 and 96 through the DMA kernel, both launch shapes, at the edges of a query
tile, a key chunk, a wavefront's pair of tiles and a query block, against the fp32 oracle; and the register-staged
kernel that keeps what the DMA cannot address."""
import pytest

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
    """One round of wide blocks and less (narrow blocks run) and nearly two (wide ones do)."""
    glue.test_prefill_attention(gpu, B, H, S, dh, B > 1 and B <= 2, False)
