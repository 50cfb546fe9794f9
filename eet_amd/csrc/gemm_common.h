// Pieces shared by the small-M (HBM-bound) and large-M (MFMA-bound) dequant-GEMM
// kernels: vector types, the exact int8 -> fp16 widening, epilogue codes and the
// argument block the dispatcher hands to the launchers.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"

namespace eet {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 4 biased bytes -> 4 fp16 values (q = u8 - 128), exact.
__device__ __forceinline__ void widen4(uint32_t x, half2v &lo, half2v &hi)
{
    const half2v magic = {(_Float16)1152.0f, (_Float16)1152.0f};
    uint32_t a = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);  // {0x64, b1, 0x64, b0}
    uint32_t b = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);  // {0x64, b3, 0x64, b2}
    lo = __builtin_bit_cast(half2v, a) - magic;
    hi = __builtin_bit_cast(half2v, b) - magic;
}

__device__ __forceinline__ half8 widen8(uint32_t x0, uint32_t x1)
{
    half2v a, b, c, d;
    widen4(x0, a, b);
    widen4(x1, c, d);
    half8 r = {a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
    return r;
}

// Epilogues: plain; + residual[M][N] (fp16 add); SwiGLU over (gate, up) n-tile
// pairs of an interleaved weight, output [M][N/2].
constexpr int kEpiNone = 0, kEpiResidual = 1, kEpiSwiglu = 2;
// The fused Q | K | V rows of a prompt, split on their way out (large-M kernel, its own entry point).
constexpr int kEpiQkv = 3;

// Row m = b * S + s, channel (part * H + h) * dh + d goes to q[b][h][s][d] of [B][H][S][dh] or to k / v[b][h][s][d] of
// [B][H][T][dh]; with a table (cos | sin of position s) the pairs (d, d + dh / 2) of q and k are rotated.
struct QkvOut {
    _Float16 *q, *k, *v;
    const float *rope;   // [>= S][dh] or null
    int S, H, dh, T;
};

struct GemmArgs {
    const _Float16 *A;
    const u32x4 *Wp;
    const _Float16 *scale;
    _Float16 *C;
    int M, N, K;
    const _Float16 *residual;
    int epi;
    const _Float16 *rms_gamma;  // non-null: RMSnorm prologue (small-M kernel only)
    float rms_eps;
    void *ws;  // optional fp32 workspace (split-k partial results)
    size_t ws_bytes;
    hipStream_t st;
    QkvOut qkv = {};  // kEpiQkv
    bool ws_zeroed = false;  // the caller vouches for the small-M kernel's counters in ws (EET_ZEROED_WORKSPACE)
    int chain = 0;  // kChainOff / kChainFirst / kChainNext (chain.h; small-M kernel only)
    // RMSnorm of the finished rows, beside them (large-M kernel only): norm_out = RMSnorm(C) * norm_gamma, or null
    const _Float16 *norm_gamma = nullptr;
    _Float16 *norm_out = nullptr;
};

// gemm_w8a16_large.hip: the MFMA-tile kernel for M > 32, and the workspace it can use.  kTakesSlabs, with nothing
// launched, for a call that 32-row slabs of the small-M kernel run faster.
constexpr int kTakesSlabs = 1;
// kEpiQkv only: nothing launched, a plain launch and a split kernel are faster.
constexpr int kSplitApart = 2;
// With norm_out: C has been launched, norm_out has not.
constexpr int kNormApart = 3;
int run_large_m(const GemmArgs &a);
size_t large_m_workspace(int M, int N, int K, int epi);

}  // namespace eet
