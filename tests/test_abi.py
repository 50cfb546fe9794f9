"""The C-ABI library: loads without a GPU, exports exactly what include/eet_hip.h
declares, and validates arguments before touching the device."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from eet_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "eet_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(eet_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    syms = declared_symbols()
    assert len(syms) >= 14
    assert sorted(_lib.SIGNATURES) == syms


def test_library_exports_every_declared_symbol():
    handle = ctypes.CDLL(_lib.LIB_PATH)
    for s in declared_symbols():
        assert hasattr(handle, s), s


def test_layout_version_and_last_error():
    L = _lib.lib()
    assert L.eet_packed_layout_version() == 1
    rc = L.eet_pack_gfx950(None, 64, 16, None)
    assert rc == -1 and b"null pointer" in L.eet_last_error()


def test_quantize_argument_errors():
    L = _lib.lib()
    w = np.zeros((4, 4), np.float32)
    q = np.zeros((4, 4), np.int8)
    s = np.zeros(4, np.float32)
    assert L.eet_quantize_int8(w.ctypes.data, 7, 4, 4, 0, q.ctypes.data, s.ctypes.data) == -1
    assert L.eet_quantize_int8(w.ctypes.data, 0, 4, 4, 9, q.ctypes.data, s.ctypes.data) == -1
    assert L.eet_quantize_int8(None, 0, 4, 4, 0, q.ctypes.data, s.ctypes.data) == -1
    assert L.eet_quantize_int8(w.ctypes.data, 0, 4, 4, 0, q.ctypes.data, s.ctypes.data) == 0


def test_device_entry_points_validate_before_launch():
    """Bad arguments are refused on the host: no GPU is needed to see the error."""
    L = _lib.lib()
    buf = np.zeros(4096, np.uint8)
    p = buf.ctypes.data
    assert L.eet_gemm_w8a16(None, p, p, p, 1, 16, 64, None, 0, None) == -1
    assert L.eet_gemm_w8a16(p, p, p, p, 1, 16, 100, None, 0, None) == -2      # K % 64
    assert L.eet_gemm_w8a16(p, p, p, p, 1, 24, 64, None, 0, None) == -2       # N % 16
    assert b"K % 64" in L.eet_last_error()
    assert L.eet_gemm_w8a16(p, p, p, p, 0, 16, 64, None, 0, None) == 0        # empty batch: nothing to do
    # split-k workspace: none once the tiles fill the chip, ksplit x M x N fp32 for M in the tens to hundreds;
    # the small-M kernel's k split: counters + exchange slots for N = 4096 / 5120 at the rows that split
    assert L.eet_gemm_w8a16_workspace(8, 4096, 4096, 0) == 0 and L.eet_gemm_w8a16_workspace(8, 12288, 4096, 0) == 0
    assert L.eet_gemm_w8a16_workspace(32, 4096, 4096, 1) == 32768 + 128 * 2 * 2 * 2 * 1024     # counters + NT 2, 2 shares, 2 m-tiles
    assert L.eet_gemm_w8a16_workspace(16, 4096, 11008, 1) == 32768 + 64 * 4 * 4 * 1 * 1024      # NT 4, 4 shares
    assert L.eet_gemm_w8a16_workspace(8, 5120, 13696, 1) == 32768 + 64 * 4 * 5 * 1 * 1024       # NT 5, 4 shares
    assert L.eet_gemm_w8a16_workspace(32, 4096, 4096, 2) == 0                                     # not with SwiGLU
    for M, N, K in ((8, 1024, 8192), (16, 3072, 8192), (32, 2048, 5632)):   # other channel counts: where the caller vouches for it
        assert L.eet_gemm_w8a16_workspace(M, N, K, 1) == 0 and L.eet_gemm_w8a16_zeroed_workspace(M, N, K, 1) > 32768
        assert L.eet_gemm_w8a16_zeroed_workspace(M, N, K, 2) == 0
    assert L.eet_gemm_w8a16_zeroed_workspace(32, 4096, 4096, 1) == L.eet_gemm_w8a16_workspace(32, 4096, 4096, 1)
    assert L.eet_gemm_w8a16_zeroed_workspace(40, 2048, 5632, 1) == 0 and L.eet_gemm_w8a16_zeroed_workspace(8, 2048, 5600, 1) == 0
    zeroed = 1 << 20 | _lib.ZEROED_WORKSPACE
    assert L.eet_gemm_w8a16(p, p, p, p, 33, 16, 64, p, zeroed, None) == -1    # more rows would write over its counters
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 33, 16, 64, 0, None, None, 0.0, p, zeroed, None) == -1
    assert L.eet_gemm_w8a16_residual_norm(p, p, p, p, 33, 16, 64, p, p, 1e-6, p, p, zeroed, None) == -1
    assert L.eet_gemm_w8a16_qkv(p, p, p, p, p, p, p, None, 1, 33, 1, 32, 64, 40, p, zeroed, None) == -1
    assert L.eet_gemm_w8a16_workspace(2048, 4096, 4096, 0) == 0
    need = L.eet_gemm_w8a16_workspace(64, 4096, 11008, 0)
    assert need >= 2 * 64 * 4096 * 4 and need % (64 * 4096 * 4) == 0
    assert L.eet_gemm_w8a16_workspace(64, 4100, 11008, 0) == 0                # not a shape the GEMM accepts
    assert L.eet_mmha_decode(p, None, None, 0, p, p, p, None, None, 1, 1, 128, 9, 8, None, None, 0, None) == -1  # step > cap
    assert L.eet_mmha_decode(p, None, None, 0, p, p, p, None, None, 1, 1, 80, 1, 8, None, None, 0, None) == -2   # head size
    assert L.eet_mmha_decode(p, p, None, 0, p, p, p, None, None, 1, 1, 128, 1, 8, None, None, 0, None) == -1     # k without v
    assert L.eet_mmha_decode(p, None, None, 0, p, p, p, None, None, 1, 1, 128, 1, 8, p, None, 0, None) == -1  # rotary without k
    assert L.eet_mmha_decode_workspace(8, 32, 128, 1100) == 0     # one workgroup per (b, h): no partial results
    need = L.eet_mmha_decode_workspace(1, 8, 128, 1100)           # fewer heads than CUs: the time axis is split
    assert need > 0
    assert L.eet_mmha_decode(p, None, None, 0, p, p, p, None, None, 1, 8, 128, 1100, 1153, None, None, 0, None) == -4
    # operator-level decode calls: argument checks happen before any launch
    assert L.eet_mmha_int8_decode(None, p, 1e-6, p, p, p, p, p, p, None, None, None, p, p, p, 1, 1, 128, 128, 1, 8,
                                  None, 0, None, 0, None) == -1
    assert L.eet_mmha_int8_decode(p, p, 1e-6, p, p, p, p, p, p, None, None, None, p, p, p, 33, 1, 128, 128, 1, 8,
                                  None, 0, None, 0, None) == -2              # more than 32 rows
    assert L.eet_mmha_int8_decode(p, p, 1e-6, p, p, p, p, p, p, None, None, None, p, p, p, 1, 1, 128, 128, 1, 8,
                                  None, 0, None, 0, None) == -1              # out aliases x
    assert L.eet_gated_ffn_int8_decode(p, p, 1e-6, p, p, p, p, p, None, 1, 128, 256, 1, None, 0, None) == -1
    assert L.eet_gated_ffn_int8_decode(p, p, 1e-6, p, p, p, p, p, p, 40, 128, 256, 1, None, 0, None) == -2
    assert L.eet_mmha_int8_decode_workspace(8, 32, 128, 1100) == L.eet_mmha_decode_workspace(8, 32, 128, 1100)
    assert L.eet_rope_table(None, 4, 128, None) == -1
    assert L.eet_rmsnorm(p, p, p, 1, 20000, 1e-6, None) == -2
    assert L.eet_qkv_split(p, p, p, p, 1, 4, 1, 128, 1, -1, 6, 8, None) == -1  # rows past the cache end
    assert L.eet_swiglu(p, p, 1, 12, None) == -2
    assert L.eet_residual_add(p, None, 1, 16, None) == -1
    assert L.eet_prefill_attention(p, p, p, p, None, None, 1, 1, 4096, 80, 4096, None) == -2


def test_python_api_errors():
    import eet_amd
    with pytest.raises(RuntimeError, match="contiguous"):
        eet_amd.quant_weights(torch.zeros(64, 32).t(), torch.int8)
    with pytest.raises(RuntimeError, match="dim"):
        eet_amd.quant_weights(torch.zeros(64), torch.int8)
    with pytest.raises(RuntimeError, match="FP16 or FP32"):
        eet_amd.quant_weights(torch.zeros(64, 16, dtype=torch.float64), torch.int8)
    with pytest.raises(RuntimeError, match="empty"):
        eet_amd.quant_weights(torch.zeros(0, 16), torch.int8)
    with pytest.raises(RuntimeError, match="int4 or int8"):
        eet_amd.quant_weights(torch.zeros(64, 16), torch.int32)
    with pytest.raises(NotImplementedError):
        eet_amd.quant_weights(torch.zeros(64, 16), torch.quint4x2)
    p, s = eet_amd.quant_weights(torch.ones(64, 16), torch.int8)
    assert p.dtype == torch.int8 and p.shape == (64, 16) and s.dtype == torch.float32 and s.shape == (16,)
    u, p, s = eet_amd.quant_weights(torch.ones(2, 64, 16).half(), torch.int8, True)
    assert u.shape == (2, 64, 16) and s.shape == (2, 16) and s.dtype == torch.float16
    with pytest.raises(NotImplementedError):
        eet_amd.MultiHeadAttention()
    import EET
    for name in ("MetaDesc", "LlamaMmha", "BaichuanMmha", "GatedFeedForwardNetworkInt8", "GatedFeedForwardNetwork",
                 "Embedding", "preprocess_weights", "quant_weights", "FeedForwardNetwork", "MultiHeadAttention",
                 "CrossMultiHeadAttention", "MaskedMultiHeadAttention", "LayerNorm"):
        assert hasattr(EET, name)
    d = EET.MetaDesc(torch.float16, 8, 32, 4096, 32, 1024, 1153, "silu", 0, 11008, "cuda:0", False, 1e-6, True)
    assert d.max_full_seq_len == 1153 and d.d_ff == 11008 and d.is_int8
    with pytest.raises(NotImplementedError):
        EET.LlamaMmha(EET.MetaDesc(torch.float32, 1, 1, 64, 1, 8), *[torch.empty(0)] * 10)


def test_alibi_caller_matches_oracle():
    from eet_amd import decoder
    from oracle import ops as O
    assert np.allclose(decoder.alibi_slopes(40), O.alibi_slopes(40))
    m = decoder.alibi_mask(8, 6).numpy()
    assert np.array_equal(np.nan_to_num(m, neginf=-1), np.nan_to_num(O.alibi_mask(8, 6), neginf=-1))


def test_fused_argument_errors():
    from eet_amd._lib import lib
    buf = np.zeros(4096, np.uint8)
    p = buf.ctypes.data
    L = _lib.lib()
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 1, 32, 64, 7, None, None, 0.0, None, 0, None) == -1          # unknown epilogue
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 1, 32, 64, 1, None, None, 0.0, None, 0, None) == -1          # residual missing
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 1, 32, 64, 0, p, None, 0.0, None, 0, None) == -1             # residual without the epilogue
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 1, 48, 64, 2, None, None, 0.0, None, 0, None) == -2          # odd tile count
    assert L.eet_gemm_w8a16_fused(p, p, p, p, 64, 32, 64, 0, None, p, 1e-6, None, 0, None) == -2       # RMSnorm prologue, M > 32


def test_tuning_keys():
    """Every documented tuning key is accepted and cleared (host state only, no GPU); malformed values and
    unknown keys are refused with a message."""
    L = _lib.lib()
    for name, value in [("EET_GEMM_SMALL_M_CONFIG", "2,8,1"), ("EET_GEMM_SMALL_M_CONFIG", "2,8,1,2"),
                        ("EET_CHAIN_SPIN_LIMIT", "0"), ("EET_CHAIN_SLEEP", "4"), ("EET_GEMM_LARGE_M_TILE", "4,4"),
                        ("EET_GEMM_LARGE_M_TILE", "2,2,4"), ("EET_MMHA_NSPLIT", "2"), ("EET_MMHA_THREADS", "256"),
                        ("EET_MMHA_UNROLL", "4"), ("EET_PREFILL_LEGACY", "1"), ("EET_PREFILL_SHAPE", "2"),
                        ("EET_PREFILL_GROUP", "4"), ("EET_PREFILL_GROUP", "-1")]:
        assert L.eet_set_tuning(name.encode(), value.encode()) == 0, L.eet_last_error()
        assert L.eet_set_tuning(name.encode(), None) == 0
    assert L.eet_set_tuning(b"EET_GEMM_SMALL_M_CONFIG", b"2,8") != 0
    assert b"nt,waves,u" in L.eet_last_error()
    assert L.eet_set_tuning(b"EET_NO_SUCH_KEY", b"1") != 0
    assert b"unknown key" in L.eet_last_error()


def test_every_table_answer_has_a_kernel():
    """The small-M launch-shape table (formula, measured shapes, k split) only answers with shapes the library
    holds a kernel for -- plain, without the workspace and chained: the query decides this on the host, for
    every row count and a wide range of channel counts, with every prologue / epilogue."""
    L = _lib.lib()
    q = [ctypes.c_int() for _ in range(4)]
    widths = sorted(set(list(range(16, 2049, 16)) + [n * 16 for n in (160, 192, 200, 230, 240, 255, 256, 257, 300, 320, 344, 384,
                                                                         428, 480, 512, 640, 688, 768, 856, 960, 1024, 1376,
                                                                         1712, 2000, 2048, 2752, 4096)]))
    for K in (64, 4096, 5120, 11008, 13696):
        for N in widths:
            for M in (1, 2, 3, 4, 7, 8, 9, 16, 17, 24, 32):
                for epi, rms in ((0, 0), (1, 0), (0, 1), (1, 1), (2, 1), (2, 0)):
                    if epi == 2 and N % 32:
                        continue
                    rc = L.eet_gemm_w8a16_small_m_shape(M, N, K, epi, rms, *[ctypes.byref(x) for x in q])
                    assert rc == 0, L.eet_last_error().decode()


def large_m_shape(M, N, K, epi, ws=0):
    v = [ctypes.c_int() for _ in range(5)]
    rc = _lib.lib().eet_gemm_w8a16_large_m_shape(M, N, K, epi, ws, *[ctypes.byref(x) for x in v])
    assert rc == 0, _lib.lib().eet_last_error().decode()
    return tuple(x.value for x in v)


SLABS = (0, 0, 0, 0, 1)


@pytest.mark.parametrize("M,N,K,epi,slabs", [
    (33, 1024, 8192, 0, True), (64, 1024, 8192, 1, True), (48, 4096, 11008, 1, True), (33, 4096, 4096, 0, True),
    (64, 4096, 11008, 1, False), (56, 3072, 8192, 1, False),          # equal or behind from 56 rows on
    (33, 1024, 1024, 0, False), (48, 4096, 2048, 1, False),           # short k ranges
    (33, 5120, 5120, 1, False), (48, 12288, 4096, 0, False),          # blocks enough
    (64, 4096, 4096, 2, True), (48, 7168, 4096, 2, True), (64, 7168, 4096, 2, False), (33, 9216, 4096, 2, False),
    (65, 1024, 8192, 0, False)])
def test_calls_without_a_workspace_keep_their_faster_path(M, N, K, epi, slabs):
    """33 to 64 rows and few channels: the small-M kernel in slabs of 32 rows, unless the caller hands over the
    workspace of a split or asks for a block shape."""
    L = _lib.lib()
    assert (large_m_shape(M, N, K, epi) == SLABS) == slabs
    need = L.eet_gemm_w8a16_workspace(M, N, K, epi)
    if slabs:
        assert need > 0 and large_m_shape(M, N, K, epi, need)[4] > 1
        assert large_m_shape(M, N, K, epi, need - 16) == SLABS
    assert L.eet_set_tuning(b"EET_GEMM_LARGE_M_TILE", b"4,2") == 0
    try:
        assert large_m_shape(M, N, K, epi)[:2] == (4, 2)
    finally:
        assert L.eet_set_tuning(b"EET_GEMM_LARGE_M_TILE", None) == 0
    v = [ctypes.byref(ctypes.c_int()) for _ in range(5)]
    for bad in ((32, N, K, 0, 0), (40, 8, 64, 0, 0), (40, 16, 32, 0, 0), (40, 48, 64, 2, 0), (40, 16, 64, 3, 0)):
        assert L.eet_gemm_w8a16_large_m_shape(*bad, *v) == -2


@pytest.mark.parametrize("M,N,K", [(406, 3072, 8192), (406, 1536, 6144), (150, 5120, 13696)])
def test_shares_are_counted_per_xcd(M, N, K):
    """A launch whose workgroups fit the 256 CUs has none left over on an XCD: its blocks go to the XCDs in eight equal
    ranges, 32 CUs each."""
    ws = _lib.lib().eet_gemm_w8a16_workspace(M, N, K, 1)
    tm, tn, wm, wn, ks = large_m_shape(M, N, K, 1, ws)
    blocks = -(-M // (16 * tm * wm)) * -(-N // (16 * tn * wn))
    assert ks > 1 and blocks * ks <= 256 and -(-blocks // 8) * ks <= 32


def pack_shape(w_dtype, K, N, ws=None, unprocessed=0):
    L, v = _lib.lib(), [ctypes.c_int() for _ in range(2)]
    ws = L.eet_quantize_pack_device_workspace(N) if ws is None else ws
    assert L.eet_quantize_pack_device_shape(w_dtype, K, N, unprocessed, ws, *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


def test_packer_grids_and_workspace():
    """Every launch the one-pass packer plans: at most 16 parts, rows that its wavefronts hold, fewer threads than the 32
    bits they are counted in, and counts and maxima within the workspace.  fp32 N = 2^28 once had a grid of 2^32 threads."""
    for K in (64, 128, 192, 320, 1024, 4096, 20480, 20544, 28672, 32768, 65536):
        for N in (16, 48, 1040, 4096, 16400, 151936, 1 << 22, (1 << 22) + 16, 1 << 26, 1 << 27, 1 << 28, 1 << 29, 1 << 30,
                  (1 << 31) - 16, 1 << 31, 1 << 33):
            for w_dtype, columns, unprocessed in ((0, 32, 0), (0, 32, 1), (1, 64, 0), (1, 64, 1)):
                waves, parts = pack_shape(w_dtype, K, N, None, unprocessed)
                assert pack_shape(w_dtype, K, N, 4 * N) == (0, 0)
                if not waves:
                    continue
                groups = -(-N // columns)
                per_part = -(-(K // 64) // parts) * 2            # units of 32 rows, whole k-tiles
                assert parts <= 16 and waves * {16: 4, 8: 5}[waves] >= per_part, (K, N, w_dtype)
                lines = 128 // columns
                grid = max(groups * parts, -(-(-(-groups // lines) * parts) // 8) * 8 * lines)
                assert grid * waves * 64 < 1 << 32 and N < 1 << 31, (K, N, w_dtype)
                words = groups * 32 + groups * parts * columns
                assert words * 4 <= _lib.lib().eet_quantize_pack_device_workspace(N), (K, N, w_dtype)
    L, v = _lib.lib(), [ctypes.byref(ctypes.c_int()) for _ in range(2)]
    for bad in ((5, 64, 16, 0, 64), (0, 96, 16, 0, 64), (0, 64, 24, 1, 64), (1, 0, 16, 1, 64)):
        assert L.eet_quantize_pack_device_shape(*bad, *v) < 0
    assert L.eet_quantize_pack_device_shape(0, 64, 16, 0, 64, None, v[1]) == -1


@pytest.mark.parametrize("w_dtype,K,N,unprocessed,waves", [
    (1, 4096, 4096, 0, 16), (1, 1024, 32000, 0, 8), (1, 11008, 4096, 0, 0), (1, 5120, 15360, 0, 8), (1, 28672, 256, 0, 0),
    (1, 28672, 1024, 0, 16), (1, 4096, 4096, 1, 16), (1, 2560, 12288, 1, 0), (1, 512, 22016, 1, 8), (1, 5120, 15360, 1, 0),
    (1, 64, 64000, 0, 8), (1, 64, 128256, 0, 0), (0, 64, 128256, 0, 0), (0, 256, 128256, 0, 8), (0, 28672, 256, 0, 16),
    (0, 14336, 11008, 1, 8), (0, 28672, 4096, 0, 0)])
def test_packer_takes_the_faster_way(w_dtype, K, N, unprocessed, waves):
    """Either side of every line of the rule."""
    assert pack_shape(w_dtype, K, N, None, unprocessed)[0] == waves


def test_cuts_of_replayed_attention():
    """A launch that is replayed keeps its cut at every step up to step_max: a split that long caches gain by and short ones
    lose by is for the calls that are cut anew at each step."""
    L = _lib.lib()

    def records(fn, B, H, dh, step):
        return fn(B, H, dh, step) // (B * H * (dh + 2) * 4)
    for size, once, replayed in (((8, 40, 128, 1024), 4, 0), ((8, 40, 128, 4096), 4, 0), ((12, 32, 96, 2048), 4, 0),
                                 ((1, 32, 128, 256), 8, 0),
                                 # more than eight splits are merged one after another: no more than the usual nine, or eight
                                 ((1, 12, 128, 2393), 9, 9), ((1, 16, 64, 2048), 8, 8),
                                 ((4, 40, 128, 2048), 8, 6), ((1, 32, 128, 1024), 8, 8), ((4, 40, 128, 1024), 3, 3),
                                 ((8, 32, 128, 4096), 0, 0), ((1, 32, 128, 1), 0, 0)):
        assert records(L.eet_mmha_decode_workspace, *size) == once, size
        assert records(L.eet_mmha_decode_replayable_workspace, *size) == replayed, size


def test_small_m_shapes_of_a_few_rows():
    """A launch of one to seven rows is not shaped as one of eight: with few activations a split costs more than it saves."""
    v = [ctypes.c_int() for _ in range(4)]

    def shape(M, N, K):
        assert _lib.lib().eet_gemm_w8a16_small_m_shape(M, N, K, 1, 0, *[ctypes.byref(x) for x in v]) == 0
        return tuple(x.value for x in v)
    for M, N, K, want in ((1, 3072, 8192, (1, 8, 2, 1)), (2, 3072, 8192, (1, 8, 2, 1)), (1, 4080, 11008, (1, 16, 1, 1)),
                          (2, 2560, 6912, (1, 16, 1, 1)), (17, 1024, 2816, (1, 16, 1, 1)), (32, 3072, 8192, (3, 8, 1, 4)),
                          (16, 3072, 8192, (3, 8, 1, 4)), (8, 4096, 16384, (1, 8, 2, 1)), (1, 4096, 11008, (1, 16, 1, 1))):
        assert shape(M, N, K) == want, (M, N, K, shape(M, N, K))
