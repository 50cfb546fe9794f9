// Operator-level entry points for the incremental (one token per sequence) call:
// everything LlamaMmha::forward_inc / BaichuanMmha::forward_inc
// (csrc/op/llama_mmha.cpp:202-266, csrc/op/baichuan_mmha.cpp:166-216) and
// GatedFeedForwardNetworkInt8::forward (csrc/op/gated_ffn_int8.cpp:98-132)
// launch, issued from one call each, as the reference's C++ operators do.  At
// decode sizes a token step is ~160 short kernels; driving each through its own
// foreign-function call costs more host time than the kernels take on the GPU
// once the batch is small.
//
// Host code only: the kernels are reached through the library's own C entry
// points, so every argument check and dispatch decision is theirs.
#include <cstddef>
#include <cstdint>

#include "common.h"

namespace {
// do the byte ranges [a, a + an) and [b, b + bn) share a byte?
bool overlaps(const void *a, size_t an, const void *b, size_t bn)
{
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + bn && y < x + an;
}
}  // namespace

extern "C" size_t eet_mmha_int8_decode_workspace(int B, int H, int dh, int step)
{
    return eet_mmha_decode_workspace(B, H, dh, step);
}

static int mmha_int8_decode(const char *fn, const void *x, const void *rms_gamma, float rms_eps, const void *qkv_w,
                                    const void *qkv_scale, const void *o_w, const void *o_scale, void *k_cache,
                                    void *v_cache, const void *alibi, const int64_t *pad, const float *rope_cos_sin,
                                    void *qkv_buf, void *ctx_buf, void *out, int B, int H, int dh, int hidden,
                                    int step, int T_cap, void *workspace, size_t workspace_bytes, void *gemm_workspace,
                                    size_t gemm_workspace_bytes, const int32_t *beam_rows_in, int32_t *beam_rows_out,
                            const int64_t *reorder_index, void *stream)
{
    EET_REQUIRE(x && rms_gamma && qkv_buf && ctx_buf && out, EET_ERR_INVALID_ARGUMENT,
                "%s: null pointer", fn);
    EET_REQUIRE(B > 0 && B <= 32 && H > 0 && dh > 0 && hidden > 0, EET_ERR_UNSUPPORTED_SHAPE,
                "%s: B=%d must be 1..32 (one token per sequence), H=%d dh=%d hidden=%d", fn, B, H, dh, hidden);
    const int inner = H * dh;
    {
        // x is read by the first launch and again, as the residual, by the last; every
        // buffer written in between must stay clear of it and of what the launch that
        // writes it reads
        const size_t xb = (size_t)B * hidden * 2, qb = (size_t)B * 3 * inner * 2, cb = (size_t)B * inner * 2;
        EET_REQUIRE(!overlaps(out, xb, x, xb) && !overlaps(qkv_buf, qb, x, xb) && !overlaps(ctx_buf, cb, x, xb),
                    EET_ERR_INVALID_ARGUMENT,
                    "%s: out, qkv_buf and ctx_buf must not overlap x (x is the residual of the last launch)", fn);
        EET_REQUIRE(!overlaps(ctx_buf, cb, qkv_buf, qb) && !overlaps(out, xb, ctx_buf, cb), EET_ERR_INVALID_ARGUMENT,
                    "%s: ctx_buf must not overlap qkv_buf, nor out ctx_buf", fn);
    }
    // RMSnorm + QKV projection (llama_mmha.cpp:222-227)
    if (int rc = eet_gemm_w8a16_fused(x, qkv_w, qkv_scale, qkv_buf, B, 3 * inner, hidden, EET_EPILOGUE_NONE, nullptr,
                                      rms_gamma, rms_eps, nullptr, 0, stream))
        return rc;
    // rotary (when a table row is given) + cache append + attention (:229-258): q, k, v are rows of qkv_buf
    const _Float16 *base = static_cast<const _Float16 *>(qkv_buf);
    const int rc = beam_rows_out != nullptr
                       ? eet_mmha_decode_beams(base, base + inner, base + 2 * inner, 3L * inner, k_cache, v_cache, ctx_buf,
                                               alibi, pad, B, H, dh, step, T_cap, rope_cos_sin, beam_rows_in,
                                               beam_rows_out, reorder_index, workspace, workspace_bytes, stream)
                       : eet_mmha_decode(base, base + inner, base + 2 * inner, 3L * inner, k_cache, v_cache, ctx_buf,
                                         alibi, pad, B, H, dh, step, T_cap, rope_cos_sin, workspace, workspace_bytes,
                                         stream);
    if (rc != EET_OK)
        return rc;
    // output projection + residual (:260-262, 428-462)
    return eet_gemm_w8a16_fused(ctx_buf, o_w, o_scale, out, B, hidden, inner, EET_EPILOGUE_RESIDUAL, x, nullptr, 0.f,
                                gemm_workspace, gemm_workspace_bytes, stream);
}

extern "C" int eet_mmha_int8_decode(const void *x, const void *rms_gamma, float rms_eps, const void *qkv_w,
                                    const void *qkv_scale, const void *o_w, const void *o_scale, void *k_cache,
                                    void *v_cache, const void *alibi, const int64_t *pad, const float *rope_cos_sin,
                                    void *qkv_buf, void *ctx_buf, void *out, int B, int H, int dh, int hidden,
                                    int step, int T_cap, void *workspace, size_t workspace_bytes, void *gemm_workspace,
                                    size_t gemm_workspace_bytes, void *stream)
{
    return mmha_int8_decode("eet_mmha_int8_decode", x, rms_gamma, rms_eps, qkv_w, qkv_scale, o_w, o_scale, k_cache,
                            v_cache, alibi, pad, rope_cos_sin, qkv_buf, ctx_buf, out, B, H, dh, hidden, step, T_cap,
                            workspace, workspace_bytes, gemm_workspace, gemm_workspace_bytes, nullptr, nullptr, nullptr,
                            stream);
}

extern "C" int eet_mmha_int8_decode_beams(const void *x, const void *rms_gamma, float rms_eps, const void *qkv_w,
                                          const void *qkv_scale, const void *o_w, const void *o_scale, void *k_cache,
                                          void *v_cache, const void *alibi, const int64_t *pad,
                                          const float *rope_cos_sin, void *qkv_buf, void *ctx_buf, void *out, int B,
                                          int H, int dh, int hidden, int step, int T_cap, const int32_t *beam_rows_in,
                                          int32_t *beam_rows_out, const int64_t *reorder_index, void *workspace,
                                          size_t workspace_bytes, void *gemm_workspace, size_t gemm_workspace_bytes,
                                          void *stream)
{
    EET_REQUIRE(beam_rows_out != nullptr, EET_ERR_INVALID_ARGUMENT, "eet_mmha_int8_decode_beams: null pointer");
    return mmha_int8_decode("eet_mmha_int8_decode_beams", x, rms_gamma, rms_eps, qkv_w, qkv_scale, o_w, o_scale, k_cache,
                            v_cache, alibi, pad, rope_cos_sin, qkv_buf, ctx_buf, out, B, H, dh, hidden, step, T_cap,
                            workspace, workspace_bytes, gemm_workspace, gemm_workspace_bytes, beam_rows_in,
                            beam_rows_out, reorder_index, stream);
}

extern "C" int eet_gated_ffn_int8_decode(const void *x, const void *rms_gamma, float rms_eps, const void *w01,
                                         const void *scale01, const void *w2, const void *scale2, void *act_buf,
                                         void *out, int B, int hidden, int d_ff, int add_residual,
                                         void *gemm_workspace, size_t gemm_workspace_bytes, void *stream)
{
    EET_REQUIRE(x && rms_gamma && act_buf && out, EET_ERR_INVALID_ARGUMENT, "eet_gated_ffn_int8_decode: null pointer");
    EET_REQUIRE(B > 0 && B <= 32 && hidden > 0 && d_ff > 0, EET_ERR_UNSUPPORTED_SHAPE,
                "eet_gated_ffn_int8_decode: B=%d must be 1..32 (one token per sequence), hidden=%d d_ff=%d", B, hidden,
                d_ff);
    {
        const size_t xb = (size_t)B * hidden * 2, ab = (size_t)B * d_ff * 2;
        EET_REQUIRE(!overlaps(out, xb, x, xb) && !overlaps(act_buf, ab, x, xb) && !overlaps(out, xb, act_buf, ab),
                    EET_ERR_INVALID_ARGUMENT, "eet_gated_ffn_int8_decode: x, act_buf and out must not overlap");
    }
    // RMSnorm + gate and up projections + SwiGLU (gated_ffn_int8.cpp:112-120): w01 holds gate and up
    // interleaved by 16-channel tile
    if (int rc = eet_gemm_w8a16_fused(x, w01, scale01, act_buf, B, 2 * d_ff, hidden, EET_EPILOGUE_SWIGLU, nullptr,
                                      rms_gamma, rms_eps, nullptr, 0, stream))
        return rc;
    // down projection + residual (:122-128, 303-357)
    return eet_gemm_w8a16_fused(act_buf, w2, scale2, out, B, hidden, d_ff,
                                add_residual ? EET_EPILOGUE_RESIDUAL : EET_EPILOGUE_NONE, add_residual ? x : nullptr,
                                nullptr, 0.f, gemm_workspace, gemm_workspace_bytes, stream);
}

// The layers of a decoder one after another: what the two calls above launch for each, from one foreign-function call.
extern "C" int eet_decoder_int8_decode(const eet_decoder_layer *layers, int num_layers, const void *x, const void *alibi,
                                       const int64_t *pad, const float *rope_cos_sin, void *qkv_buf, void *ctx_buf,
                                       void *attn_out, void *act_buf, void *out, int B, int H, int dh, int hidden, int d_ff,
                                       float rms_eps, int step, int T_cap, void *workspace, size_t workspace_bytes,
                                       void *o_workspace, size_t o_workspace_bytes, void *down_workspace,
                                       size_t down_workspace_bytes, void *stream)
{
    EET_REQUIRE(layers && num_layers > 0, EET_ERR_INVALID_ARGUMENT, "eet_decoder_int8_decode: no layers");
    for (int i = 0; i < num_layers; ++i) {
        const eet_decoder_layer &l = layers[i];
        if (int rc = mmha_int8_decode("eet_decoder_int8_decode", x, l.attn_gamma, rms_eps, l.qkv_w, l.qkv_scale, l.o_w,
                                      l.o_scale, l.k_cache, l.v_cache, alibi, pad, rope_cos_sin, qkv_buf, ctx_buf, attn_out,
                                      B, H, dh, hidden, step, T_cap, workspace, workspace_bytes, o_workspace,
                                      o_workspace_bytes, nullptr, nullptr, nullptr, stream))
            return rc;
        if (int rc = eet_gated_ffn_int8_decode(attn_out, l.ffn_gamma, rms_eps, l.w01, l.scale01, l.w2, l.scale2, act_buf, out,
                                               B, hidden, d_ff, 1, down_workspace, down_workspace_bytes, stream))
            return rc;
        x = out;
    }
    return EET_OK;
}

// The same incremental call in its replayable form (see eet_mmha_decode_replayable): recorded once
// into a HIP graph, it serves every later token.
extern "C" int eet_mmha_int8_decode_replayable(const void *x, const void *rms_gamma, float rms_eps, const void *qkv_w,
                                               const void *qkv_scale, const void *o_w, const void *o_scale,
                                               void *k_cache, void *v_cache, const void *alibi, int alibi_ld,
                                               const int64_t *pad, const float *rope_table, void *qkv_buf,
                                               void *ctx_buf, void *out, int B, int H, int dh, int hidden,
                                               const int *step_dev, int step_max, int T_cap, void *workspace,
                                               size_t workspace_bytes, void *gemm_workspace,
                                               size_t gemm_workspace_bytes, void *stream)
{
    EET_REQUIRE(x && rms_gamma && qkv_buf && ctx_buf && out, EET_ERR_INVALID_ARGUMENT,
                "eet_mmha_int8_decode_replayable: null pointer");
    EET_REQUIRE(B > 0 && B <= 32 && H > 0 && dh > 0 && hidden > 0, EET_ERR_UNSUPPORTED_SHAPE,
                "eet_mmha_int8_decode_replayable: B=%d must be 1..32 (one token per sequence), H=%d dh=%d hidden=%d", B,
                H, dh, hidden);
    const int inner = H * dh;
    {
        const size_t xb = (size_t)B * hidden * 2, qb = (size_t)B * 3 * inner * 2, cb = (size_t)B * inner * 2;
        EET_REQUIRE(!overlaps(out, xb, x, xb) && !overlaps(qkv_buf, qb, x, xb) && !overlaps(ctx_buf, cb, x, xb) &&
                        !overlaps(ctx_buf, cb, qkv_buf, qb) && !overlaps(out, xb, ctx_buf, cb),
                    EET_ERR_INVALID_ARGUMENT, "eet_mmha_int8_decode_replayable: x, qkv_buf, ctx_buf and out must not overlap");
    }
    if (int rc = eet_gemm_w8a16_fused(x, qkv_w, qkv_scale, qkv_buf, B, 3 * inner, hidden, EET_EPILOGUE_NONE, nullptr,
                                      rms_gamma, rms_eps, nullptr, 0, stream))
        return rc;
    const _Float16 *base = static_cast<const _Float16 *>(qkv_buf);
    if (int rc = eet_mmha_decode_replayable(base, base + inner, base + 2 * inner, 3L * inner, k_cache, v_cache, ctx_buf,
                                            alibi, alibi_ld, pad, B, H, dh, step_dev, step_max, T_cap, rope_table,
                                            workspace, workspace_bytes, stream))
        return rc;
    return eet_gemm_w8a16_fused(ctx_buf, o_w, o_scale, out, B, hidden, inner, EET_EPILOGUE_RESIDUAL, x, nullptr, 0.f,
                                gemm_workspace, gemm_workspace_bytes, stream);
}
