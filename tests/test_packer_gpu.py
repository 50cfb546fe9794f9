"""The packer on the GPU (eet_quantize_pack_device) against the known answers recorded from the reference,
the numpy oracle, and the shipped host packer: bit-exact in every case."""
import json
import os

import numpy as np
import pytest
import torch

import eet_amd
from oracle import quant as Q

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
GOLD = json.load(open(os.path.join(HERE, "golden", "quant_known_answers.json")))


def golden_matrix(case, dtype=np.float32):
    K = case["K"]
    w = np.full((K, 64), 0.25, dtype)
    col = np.full(K, case["column"]["fill"], dtype)
    for k, v in case["column"]["set"].items():
        col[int(k)] = v
    w[:, 5] = col
    return w


@pytest.mark.parametrize("case", GOLD["quantize"], ids=lambda c: c["name"])
def test_known_answers(gpu, case):
    w = golden_matrix(case)
    q, p, s = eet_amd.quant_weights_device(torch.from_numpy(w).to(gpu), True)
    q, s = q.cpu().numpy(), s.cpu().numpy()
    assert float(s[5]) == case["scale"]
    if "q_all" in case:
        assert (q[:, 5] == case["q_all"]).all()
    for k, v in case.get("q", {}).items():
        assert int(q[int(k), 5]) == v, k
    assert torch.equal(p.cpu(), eet_amd.pack_weights(torch.from_numpy(q)))


def tricky(K, N, dtype, seed):
    """Random weights plus what a quantiser gets wrong first: an all-zero column, a column whose quotients
    sit exactly on .5 ties, one at the clamp (+absmax -> 128 -> 127, -absmax -> -128), tiny and huge columns."""
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    w[:, 1] = 0.0
    w[:, 2] = (rng.integers(-255, 256, K) * 0.5).astype(np.float32) / 128.0   # scale 1/128 once absmax is 1
    w[0, 2], w[1, 2] = 1.0, -1.0
    w[:, 3] = rng.choice([1.0, -1.0, 0.99609375, 0.00390625], K)
    w[:, 4] *= 1e-4
    w[:, 7] *= 3e3
    return w.astype(dtype)


@pytest.mark.parametrize("K,N", [(64, 16), (64, 144), (192, 400), (1024, 1040), (4096, 4096)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("mode", ["ref128", "sym127"])
def test_matches_host_packer(gpu, K, N, dtype, mode):
    w = torch.from_numpy(tricky(K, N, dtype, K + N))
    uh, ph, sh = eet_amd.quant_weights(w, torch.int8, True, mode=mode)
    ud, pd, sd = eet_amd.quant_weights_device(w.to(gpu), True, mode=mode)
    assert torch.equal(ud.cpu(), uh), "unprocessed int8"
    assert torch.equal(pd.cpu(), ph), "gfx950 layout"
    assert torch.equal(sd.cpu().view(torch.int16 if dtype == np.float16 else torch.int32),
                       sh.view(torch.int16 if dtype == np.float16 else torch.int32)), "scales (bit pattern)"
    p2, s2 = eet_amd.quant_weights_device(w.to(gpu), False, mode=mode)      # without the unprocessed output
    assert torch.equal(p2, pd) and torch.equal(s2, sd)
    if mode == "ref128" and K * N <= 1 << 20:
        qo, so = Q.quantize_ref128(w.numpy())
        assert np.array_equal(ud.cpu().numpy(), qo)


def test_full_size_properties(gpu):
    """LLaMA-7B gate projection (4096 x 11008) generated on the GPU: |q| <= 128, every non-zero column reaches
    127 or -128, dequantised error within half a step, and unpack(packed) == unprocessed."""
    g = torch.Generator(device=gpu).manual_seed(5)
    w = (torch.randn(4096, 11008, generator=g, device=gpu) * 0.02).half()
    q, p, s = eet_amd.quant_weights_device(w, True)
    assert torch.equal(eet_amd.unpack_weights(p.cpu()), q.cpu())
    ext = torch.maximum(q.amax(0), -q.amin(0) - 1)
    assert bool((ext == 127).all())
    s32 = w.float().abs().amax(0) / 128
    err = (q.float() * s32 - w.float()).abs()
    inside = (q > -128) & (q < 127)
    assert float((err[inside] / s32.expand_as(err)[inside]).max()) <= 0.5 + 1e-3


def test_arguments(gpu):
    from eet_amd._lib import lib
    L = lib()
    w = torch.zeros(64, 16, dtype=torch.float16, device=gpu)
    o = torch.zeros(64, 16, dtype=torch.int8, device=gpu)
    s = torch.zeros(16, dtype=torch.float16, device=gpu)
    ws = torch.zeros(16, dtype=torch.int32, device=gpu)
    ok = (w.data_ptr(), 1, 64, 16, 0, None, o.data_ptr(), s.data_ptr(), ws.data_ptr(), 64, None)
    assert L.eet_quantize_pack_device(*ok) == 0
    bad = list(ok); bad[2] = 96
    assert L.eet_quantize_pack_device(*bad) == -2          # K % 64
    bad = list(ok); bad[9] = 8
    assert L.eet_quantize_pack_device(*bad) == -4          # workspace too small
    bad = list(ok); bad[1] = 5
    assert L.eet_quantize_pack_device(*bad) == -1          # dtype
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        eet_amd.quant_weights_device(torch.zeros(64, 16))  # CPU tensor


def test_converter_on_device(gpu):
    """convert_llama_weights(device=...) quantises and packs with the HIP packer: same keys and bits as the
    host conversion, linears left on the GPU."""
    from eet_amd import convert
    hid, ff = 128, 192
    g = torch.Generator().manual_seed(3)
    r = lambda *s: (torch.randn(*s, generator=g) * 0.05).half()
    sd = {"model.embed_tokens.weight": r(50, hid), "model.norm.weight": r(hid), "lm_head.weight": r(50, hid)}
    p = "model.layers.0."
    for n in "qkvo":
        sd[p + f"self_attn.{n}_proj.weight"] = r(hid, hid)
    sd[p + "mlp.gate_proj.weight"], sd[p + "mlp.up_proj.weight"] = r(ff, hid), r(ff, hid)
    sd[p + "mlp.down_proj.weight"] = r(hid, ff)
    sd[p + "input_layernorm.weight"], sd[p + "post_attention_layernorm.weight"] = r(hid), r(hid)
    host = convert.convert_llama_weights(sd)
    dev = convert.convert_llama_weights(sd, device=gpu)
    assert host.keys() == dev.keys()
    for k, v in host.items():
        if isinstance(v, torch.Tensor):
            assert torch.equal(dev[k].cpu(), v), k
            if k.endswith("proj.weight") or k.startswith("layer.0.ffn.") and k.endswith(("weight", "scale")) and "layernorm" not in k:
                assert dev[k].device.type == "cuda", k
        else:
            assert dev[k] == v


@pytest.mark.parametrize("K,N", [(64, 16), (128, 80), (2048, 16), (2112, 48), (1280, 1040), (8256, 112), (32832, 32),
                                 (2624, 16400), (16384, 16), (32768, 16), (20480, 80)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_one_pass_matches_two_passes(gpu, K, N, dtype):
    """The one-pass kernel at the edges of its shares (rows a workgroup holds, one to sixteen workgroups per column
    group, groups cut off by N) and with NaN and infinite weights, against the two-pass kernels, which a call with no
    more than 4 N bytes of workspace takes, and the host packer.  (fp16 2624 x 16400 takes two passes either way; fp16 in the
    8-wavefront form is test_eight_wavefronts_fp16.)  Exact: every step is one correctly rounded operation."""
    from eet_amd._lib import check, lib
    w = tricky(K, N, dtype, K * 3 + N)
    w[K // 2, 8], w[K - 1, 9], w[:, 10], w[5, 11] = np.nan, np.inf, np.nan, np.nan
    uh, ph, sh = eet_amd.quant_weights(torch.from_numpy(w), torch.int8, True)
    wd = torch.from_numpy(w).to(gpu)
    code = 0 if dtype == np.float32 else 1
    for nbytes in (lib().eet_quantize_pack_device_workspace(N), 4 * N):
        ws = torch.full((nbytes // 4 + 1024,), -1, dtype=torch.int32, device=gpu)
        for want_q in (True, False):
            q, p = (torch.zeros(K, N, dtype=torch.int8, device=gpu) for _ in range(2))
            s = torch.zeros(N, dtype=wd.dtype, device=gpu)
            check(lib().eet_quantize_pack_device(wd.data_ptr(), code, K, N, 0, q.data_ptr() if want_q else None, p.data_ptr(),
                                                 s.data_ptr(), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream))
            assert torch.equal(p.cpu(), ph)
            assert not want_q or torch.equal(q.cpu(), uh)
            assert torch.equal(s.cpu().view(torch.int16 if code else torch.int32), sh.view(torch.int16 if code else torch.int32))
            assert (ws[nbytes // 4:] == -1).all()       # nothing behind the workspace


def test_overlapping_calls_do_not_share_a_workspace(gpu, monkeypatch):
    """Calls on two streams may run side by side: each has maxima and arrival counts of its own."""
    from eet_amd import ops
    real, seen = ops.lib(), []

    class Watched:
        def __getattr__(self, name):
            fn = getattr(real, name)
            if name != "eet_quantize_pack_device":
                return fn
            return lambda *a: seen.append((a[8], a[9])) or fn(*a)
    ws = [torch.from_numpy(tricky(512, 256, np.float16, i)).to(gpu) for i in range(2)]
    want = [eet_amd.quant_weights_device(w) for w in ws]
    torch.cuda.synchronize()
    monkeypatch.setattr(ops, "lib", Watched)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for round in range(4):
        got = []
        for w, stream in zip(ws, streams):
            with torch.cuda.stream(stream):
                got.append(eet_amd.quant_weights_device(w))
        (a, size), (b, _) = seen[-2:]
        assert a + size <= b or b + size <= a, "one buffer for both streams"
        torch.cuda.synchronize()
        for pair, other in zip(got, want):
            assert all(torch.equal(x, y) for x, y in zip(pair, other))


@pytest.mark.parametrize("K,N", [(128, 80), (4096, 1040), (1280, 4096), (2048, 16400), (20480, 48)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_columns_without_a_scale(gpu, K, N, dtype):
    """Zero, NaN, infinite, tiny and huge columns between ordinary ones, several of them and of the ordinary ones in every
    lane's share, with a NaN in one part of the rows only: against the host packer, exact."""
    rng = np.random.default_rng(K + N)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    w[:, 1::7] = 0
    w[:, 2::21] = np.nan
    w[K - 3, 9::21] = np.nan
    w[1, 16::21] = -np.nan
    w[K // 2, 3::14] = np.inf
    w[:, 10::14] *= 3e-6 if dtype == np.float16 else 1e-36
    w[:, 4::14] *= 1e6 if dtype == np.float16 else 1e37
    with np.errstate(over="ignore"):
        w = torch.from_numpy(w.astype(dtype))
    uh, ph, sh = eet_amd.quant_weights(w, torch.int8, True)
    ud, pd, sd = eet_amd.quant_weights_device(w.to(gpu), True)
    assert torch.equal(ud.cpu(), uh) and torch.equal(pd.cpu(), ph)
    bits = torch.int16 if dtype == np.float16 else torch.int32
    assert torch.equal(sd.cpu().view(bits), sh.view(bits))


@pytest.mark.parametrize("K,N", [(128, 80), (2048, 96), (4096, 1040), (1280, 4096), (20480, 48), (2048, 16400)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_parts_that_do_not_wait(gpu, tuning, K, N, dtype):
    """Every workgroup gives up its wait at once and reads the other parts' rows itself: the same bits, NaN and infinite
    columns among them."""
    w = tricky(K, N, dtype, K + N)
    w[K // 2, 8::16], w[K - 1, 9], w[:, 10], w[5, 11], w[K - 2, 12] = np.nan, np.inf, np.nan, -np.nan, -np.inf
    w = torch.from_numpy(w)
    uh, ph, sh = eet_amd.quant_weights(w, torch.int8, True)
    tuning("EET_PACK_POLL_LIMIT", 0)
    ud, pd, sd = eet_amd.quant_weights_device(w.to(gpu), True)
    assert torch.equal(ud.cpu(), uh) and torch.equal(pd.cpu(), ph)
    bits = torch.int16 if dtype == np.float16 else torch.int32
    assert torch.equal(sd.cpu().view(bits), sh.view(bits))


@pytest.mark.parametrize("N", [16, 32, 48, 112, 128, 144, 1040, 2064, 4112, 16400])
@pytest.mark.parametrize("K", [64, 320, 2624])
def test_unprocessed_output_at_every_place_in_a_line(gpu, K, N):
    """fp32 with the row-major output, whose workgroups are numbered by cache lines of that output: lines that N cuts off,
    fewer lines than XCDs and more, one part and several."""
    w = torch.from_numpy(tricky(K, max(N, 8), np.float32, K + N)[:, :N])
    uh, ph, sh = eet_amd.quant_weights(w.contiguous(), torch.int8, True)
    ud, pd, sd = eet_amd.quant_weights_device(w.contiguous().to(gpu), True)
    assert torch.equal(ud.cpu(), uh) and torch.equal(pd.cpu(), ph) and torch.equal(sd.cpu().view(torch.int32), sh.view(torch.int32))


@pytest.mark.parametrize("K,N,parts", [(64, 16400, 1), (512, 22016, 1), (1088, 16464, 1), (2048, 16400, 2), (1024, 32000, 1),
                                       (3072, 9232, 3), (5120, 6144, 5), (5120, 13696, 4), (13696, 5120, 11)])
def test_eight_wavefronts_fp16(gpu, K, N, parts):
    """fp16 in the 8-wavefront form, with one part and several, one round of workgroups and more, groups cut off by N and by
    the rows a wavefront holds: the result of the two passes, which a call with 4 N bytes of workspace takes and which the
    other tests hold to the host packer.  With the row-major output too where that takes the form."""
    import ctypes
    from eet_amd._lib import check, lib
    g = torch.Generator(device=gpu).manual_seed(K + N)
    w = torch.randn(K, N, generator=g, device=gpu, dtype=torch.float16) * 0.02
    w[:, 1::67] = 0
    w[K // 2, 8::131], w[K - 1, 9] = float("nan"), float("inf")
    need, form = lib().eet_quantize_pack_device_workspace(N), [ctypes.c_int() for _ in range(2)]

    def run(nbytes, want_q):
        ws = torch.full((nbytes // 4 + 256,), -1, dtype=torch.int32, device=gpu)
        q, p, s = (torch.zeros(*shape, dtype=t, device=gpu) for shape, t in (((K, N), torch.int8), ((K, N), torch.int8),
                                                                             ((N,), torch.float16)))
        check(lib().eet_quantize_pack_device(w.data_ptr(), 1, K, N, 0, q.data_ptr() if want_q else None, p.data_ptr(),
                                             s.data_ptr(), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream))
        assert (ws[nbytes // 4:] == -1).all()
        return q, p, s.view(torch.int16)
    for want_q in (0, 1):
        check(lib().eet_quantize_pack_device_shape(1, K, N, want_q, need, *[ctypes.byref(x) for x in form]))
        assert [x.value for x in form] == [8, parts] or (want_q and form[0].value == 0)
        for one, two in zip(run(need, want_q), run(4 * N, want_q)):
            assert torch.equal(one, two)


@pytest.mark.parametrize("K,N", [(64, 16), (128, 512), (192, 528), (320, 4112), (1088, 8208)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("mode", [0, 1])
def test_two_passes(gpu, K, N, dtype, mode):
    """The two-pass kernels where the second one's order of tiles is ragged (a last chunk of 64 rows, chunks of columns that N
    cuts off, a number of chunks that eight XCDs do not share evenly), with quotients on, beside and away from the halves
    where rounding decides and columns without a usable scale: against the host packer, exact."""
    from eet_amd._lib import check, lib
    w = tricky(K, N, dtype, K * 5 + N)
    w[:, 3::11] = np.arange(K)[:, None] % 255 * 0.5 - 63.5     # all halves of a scale of one, in REF128 mode
    w[K // 2, 3::11] = 128 if mode == 0 else 127
    w[:, 4::11], w[K - 1, 5::11], w[K // 3, 6::11], w[:, 7::11] = 0, np.inf, np.nan, np.nan
    want = eet_amd.quant_weights(torch.from_numpy(w), torch.int8, True, mode=["ref128", "sym127"][mode])
    wd, code = torch.from_numpy(w).to(gpu), 0 if dtype == np.float32 else 1
    ws = torch.full((N,), -1, dtype=torch.int32, device=gpu)
    for want_q in (True, False):
        q, p = (torch.zeros(K, N, dtype=torch.int8, device=gpu) for _ in range(2))
        s = torch.zeros(N, dtype=wd.dtype, device=gpu)
        check(lib().eet_quantize_pack_device(wd.data_ptr(), code, K, N, mode, q.data_ptr() if want_q else None, p.data_ptr(),
                                             s.data_ptr(), ws.data_ptr(), 4 * N, torch.cuda.current_stream().cuda_stream))
        bits = torch.int16 if code else torch.int32
        assert torch.equal(p.cpu(), want[1]) and torch.equal(s.cpu().view(bits), want[2].view(bits))
        assert not want_q or torch.equal(q.cpu(), want[0])


def test_idle_cus_take_two_passes():
    """fp16 columns whose shared groups would leave over a sixth of the workgroup slots empty, or a few workgroups to a second
    round, with 11 M weights and more."""
    import ctypes
    from eet_amd._lib import check, lib

    def waves(K, N, code=1, q=0):
        w, p = ctypes.c_int(), ctypes.c_int()
        check(lib().eet_quantize_pack_device_shape(code, K, N, q, lib().eet_quantize_pack_device_workspace(N),
                                                   ctypes.byref(w), ctypes.byref(p)))
        return w.value
    assert all(waves(K, N, 1, q) == 0 for q in (0, 1) for K, N in ((2048, 5632), (3072, 6144), (4096, 5632), (2048, 6656), (2560, 11008), (3072, 11008)))
    assert waves(1920, 5632) == 16                                       # under 11 M weights
    assert waves(2048, 7168) == 16 and waves(2048, 8192) == 16           # 224 workgroups, 256
    assert waves(2560, 10240) == 8 and waves(5120, 13696) == 8           # 480 of 512; several rounds
    assert waves(1024, 11008) == 16                                      # no group is shared
    assert waves(2048, 5632, 0) == 16                                    # fp32


def test_idle_cus_that_do_not_matter():
    """Sizes inside the range of the two-pass rule that measure faster, or no slower, in one: fewer than two units to a wavefront, three
    workgroups to a group and under 16 M weights, 82 % of the slots taken.  And the other side of each line."""
    import ctypes
    from eet_amd._lib import check, lib

    def waves(K, N):
        w, p = ctypes.c_int(), ctypes.c_int()
        check(lib().eet_quantize_pack_device_shape(1, K, N, 0, lib().eet_quantize_pack_device_workspace(N), ctypes.byref(w), ctypes.byref(p)))
        return w.value
    assert waves(1856, 6208) == 16 and waves(1984, 6144) == 16 and waves(2048, 6144) == 0
    assert waves(2752, 4224) == 16 and waves(3712, 4160) == 16 and waves(4032, 4160) == 0
    assert waves(2560, 8960) == 8 and waves(3136, 6784) == 16 and waves(2944, 6656) == 0 and waves(5120, 6656) == 0
