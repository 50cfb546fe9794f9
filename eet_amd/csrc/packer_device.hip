// The offline packer on the GPU: fp16 / fp32 [K][N] weights already resident in
// HBM -> per-output-channel int8 + scales -> gfx950 tile layout.
//
// Same results, bit for bit, as eet_quantize_int8 followed by eet_pack_gfx950
// (packer.cc), i.e. as the reference's symmetric_quantize
// (3rdparty/cutlass_kernels/cutlass_preprocessors.cc:581-678) in
// EET_QUANT_REF128 mode: every step is a single correctly rounded IEEE fp32
// operation (|x| and max, one multiply or divide for the scale, the quotient, an
// exact round-half-away), so host and device cannot differ; a product with the
// reciprocal stands for the quotient only where both provably round to the same
// integer.  The reference has no device quantiser; converting a checkpoint on the
// host costs seconds per billion weights, here the time of reading it from HBM.
//
// HBM-bound.  Most matrices go in one pass that holds them in the registers of
// the chip (quant_group_kernel; one_pass_wins has the rule and the times).  The
// others take two: pass 1 reads the matrix once (column absmax, one 32-bit
// atomic max per column and 128-row chunk); pass 2 reads it again (from the
// Infinity Cache when it fits) and writes one byte per weight in the packed
// layout, plus one more in row-major order when the caller wants the
// unprocessed matrix.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "tuning.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kColsPerThread = 8;   // pass 1: 16 bytes of fp16 per load
constexpr int kMaxRows = 128;       // rows per workgroup in pass 1 (32 per wavefront)
constexpr int kMaxPolls = 1 << 14;   // one pass: waiting for the other parts of a column group
constexpr int kMaxParts = 16;
constexpr int kCountStride = 32;    // words: a line for every count
constexpr int kChunkCols = 64 * kColsPerThread;
constexpr int kTileCols = 128;      // pass 2: one k-tile x 8 n-tiles per workgroup
constexpr unsigned kMostTurns = 1 << 15;   // pass 2: rows of a grid

// x / s + 128 by way of the reciprocal, below: the scales it is used for, and how near to a half it decides nothing
constexpr float kLeastScale = 0x1p-100f, kLargestScale = 0x1p100f, kNear = 0x1p-15f;

template <typename T>
__device__ __forceinline__ float to_f32(T x)
{
    return static_cast<float>(x);
}

__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t *p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        p[i] = 0u;
}

// amax[c] = max over rows of |w[r][c]|, as the bit pattern of a non-negative
// float (which orders like the unsigned integer).  NaN weights are ignored, as
// on the host (the comparison is false).  The four wavefronts of a workgroup
// share 512 columns and take every fourth row, eight loads in flight each; they
// meet in LDS, so one atomic per column leaves the workgroup.
template <typename T>
__global__ __launch_bounds__(256) void colmax_kernel(const T *__restrict__ w, size_t K, size_t N,
                                                     uint32_t *__restrict__ amax)
{
    __shared__ float part[4][64 * kColsPerThread];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t c0 = ((size_t)blockIdx.x * 64 + lane) * kColsPerThread;
    const size_t r0 = (size_t)blockIdx.y * kMaxRows;
    const size_t r1 = r0 + kMaxRows < K ? r0 + kMaxRows : K;
    float m[kColsPerThread];
#pragma unroll
    for (int i = 0; i < kColsPerThread; ++i)
        m[i] = 0.f;
    if (c0 < N) {   // N % 16 == 0: the 8 columns are in range together
        for (size_t r = r0 + wave; r < r1; r += 32) {
            T v[8][kColsPerThread];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t rr = r + 4 * u < r1 ? r + 4 * u : r;   // past the end: the row again
                __builtin_memcpy(v[u], w + rr * N + c0, sizeof(v[u]));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int i = 0; i < kColsPerThread; ++i) {
                    const float a = __builtin_fabsf(to_f32(v[u][i]));
                    m[i] = (m[i] < a) ? a : m[i];
                }
        }
    }
#pragma unroll
    for (int i = 0; i < kColsPerThread; ++i)
        part[wave][lane * kColsPerThread + i] = m[i];
    __syncthreads();
    for (int c = threadIdx.x; c < 64 * kColsPerThread; c += 256) {
        const size_t col = (size_t)blockIdx.x * 64 * kColsPerThread + c;
        if (col < N) {
            float a = part[0][c];
            a = a < part[1][c] ? part[1][c] : a;
            a = a < part[2][c] ? part[2][c] : a;
            a = a < part[3][c] ? part[3][c] : a;
            atomicMax(amax + col, __float_as_uint(a));
        }
    }
}

// round-half-away-from-zero of x / s clamped to [lo, 127]; see quant_row in
// packer.cc for why this equals clamp(round(x / s)).
__device__ __forceinline__ int quant_one(float x, float s, float nan_to, int lo)
{
    float v = __fdiv_rn(x, s);
    v = (v == v) ? v : nan_to;
    v = (v < 200.f) ? v : 200.f;
    v = (v > -200.f) ? v : -200.f;
    int t = static_cast<int>(v);
    const float d = v - static_cast<float>(t);
    t += (d >= 0.5f) ? 1 : 0;
    t -= (d <= -0.5f) ? 1 : 0;
    t = (t < 127) ? t : 127;
    t = (t > lo) ? t : lo;
    return t;
}

// One k-tile (64 rows) x 128 columns per workgroup: rows are read in 256-byte
// (fp16) pieces and quantised; the tile is kept column-major in LDS (a thread
// owns 4 consecutive rows of its 8 columns, i.e. 8 whole 32-bit words), so that
// the 16 bytes lane (g, i) of a packed tile holds -- q[64*kt + 16*g + b][16*nt
// + i] ^ 0x80 for b = 0 .. 15, the layout of eet_pack_gfx950 -- are four
// consecutive words, and the tile leaves as eight whole 1 KiB packed tiles.
//
// What is left to bound it is memory.  It was the vector ALU, with 15 instructions a weight and two divisions a thread
// and column; now a weight takes 4.5 (the product with the reciprocal through the byte conversion, as the one-pass kernel
// below has it with its bounds; what lies near a half or has no usable reciprocal is divided, weight by weight), a column's scale is
// found once per workgroup, under the weights' latency, and the tiles are taken in the reverse of pass 1's order on the XCDs
// that read them there, whose L2s hold the last of them.  Both passes, us, before / now: fp16 2048 x 5632 19.8 / 16.4,
// 11008 x 4096 42.8 / 40.2, 16384 x 16384 266 / 249; fp32 8192 x 11008 166 / 151; with the row-major output, fp16,
// 4096 x 11008 51.5 / 48.6.
template <typename T>
__global__ __launch_bounds__(256) void quant_pack_kernel(const T *__restrict__ w, size_t K, size_t N, int ref128,
                                                         const uint32_t *__restrict__ amax, int8_t *__restrict__ q_out,
                                                         uint8_t *__restrict__ packed, T *__restrict__ scale)
{
    __shared__ uint32_t lq[kTileCols][17];   // [column][4-row word], one word of padding per column
    __shared__ __attribute__((aligned(16))) float s_all[kTileCols], inv_all[kTileCols];
    const size_t ktiles = K / 64;
    // Pass 1's workgroups, last one first, each on the XCD that it ran on, and each as the tiles of its 512 x 128 weights
    const unsigned wide = (unsigned)((N + kChunkCols - 1) / kChunkCols), chunks = wide * (unsigned)((K + kMaxRows - 1) / kMaxRows);
    const unsigned turns = (chunks + 7) / 8, done = blockIdx.z * gridDim.y + blockIdx.y;
    const unsigned chunk = (turns - 1 - done) * 8 + blockIdx.x % 8, sub = blockIdx.x / 8, chunk_row = chunk / wide;
    const size_t kt = (size_t)chunk_row * (kMaxRows / 64) + sub / (kChunkCols / kTileCols);
    const size_t col0 = (size_t)(chunk - chunk_row * wide) * kChunkCols + sub % (kChunkCols / kTileCols) * kTileCols;
    if (done >= turns || chunk >= chunks || kt >= ktiles || col0 >= N)
        return;
    const int tid = threadIdx.x;
    const int c8 = (tid & 15) * 8, rw = tid >> 4;   // columns c8 .. c8+7, rows 4*rw .. 4*rw+3
    const size_t col = col0 + c8;
    const float nan_to = ref128 ? 1000.f : 0.f;
    const int lo = ref128 ? -128 : -127;

    // (columns past N read the last ones: no branch in front of the waits)
    constexpr int kWords = 2 * (int)sizeof(T);
    uint32_t raw[4][kWords];
#pragma unroll
    for (int it = 0; it < 4; ++it)
        __builtin_memcpy(raw[it], w + (kt * 64 + 4 * rw + it) * N + (col < N ? col : N - 8), sizeof(raw[it]));
    if (tid < kTileCols && col0 + tid < N) {
        const float a = __uint_as_float(amax[col0 + tid]);
        const float s = ref128 ? a * (1.f / 128.f) : __fdiv_rn(a, 127.f);
        s_all[tid] = s;
        // (NaN: every weight of the column is divided)
        inv_all[tid] = s > kLeastScale && s < kLargestScale ? __fdiv_rn(1.f, s) : __builtin_nanf("");
        if (kt == 0)
            scale[col0 + tid] = static_cast<T>(s);
    }
    __syncthreads();
    if (col < N) {   // N % 16 == 0: the 8 columns are in range together
        T v[4][8];
#pragma unroll
        for (int it = 0; it < 4; ++it) {
#pragma unroll
            for (int d = 0; d < kWords; ++d)
                asm volatile("" : "+v"(raw[it][d]));   // the weights are waited for here, behind the column's scale
            __builtin_memcpy(v[it], raw[it], sizeof(v[it]));
        }
        float inv_s[8];
        __builtin_memcpy(inv_s, inv_all + c8, sizeof(inv_s));
        uint32_t word[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        float near = 1.f;
#pragma unroll
        for (int it = 0; it < 4; ++it)
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                const float f0 = __builtin_fmaf(to_f32(v[it][i]), inv_s[i], 128.f);
                const float f1 = __builtin_fmaf(to_f32(v[it][i + 1]), inv_s[i + 1], 128.f);
                word[i] = __builtin_amdgcn_cvt_pk_u8_f32(f0, it, word[i]);
                word[i + 1] = __builtin_amdgcn_cvt_pk_u8_f32(f1, it, word[i + 1]);
                asm("v_minimum3_f32 %0, %0, abs(%1), abs(%2)"   // NaN where one of them is
                    : "+v"(near)
                    : "v"(__builtin_amdgcn_fractf(f0) - 0.5f), "v"(__builtin_amdgcn_fractf(f1) - 0.5f));
            }
        if (!(near >= kNear)) {
#pragma unroll
            for (int it = 0; it < 4; ++it)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = to_f32(v[it][i]), f = __builtin_fmaf(x, inv_s[i], 128.f);
                    if (!(__builtin_fabsf(__builtin_amdgcn_fractf(f) - 0.5f) >= kNear))
                        word[i] = (word[i] & ~(0xffu << (8 * it))) |
                                  (uint32_t)(quant_one(x, s_all[c8 + i], nan_to, lo) + 128) << (8 * it);
                }
        }
        if (q_out != nullptr) {
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                u32x2 o = {0, 0};
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    o[i / 4] |= (word[i] >> (8 * it) & 0xffu) << (8 * (i % 4));
                *reinterpret_cast<u32x2 *>(q_out + (kt * 64 + 4 * rw + it) * N + col) = o ^ 0x80808080u;
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            lq[c8 + i][rw] = word[i];
    }
    __syncthreads();
    // 8 tiles x 64 lanes = 512 pieces of 16 bytes, two per thread
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int piece = it * 256 + tid;
        const int n8 = piece >> 6, lane = piece & 63;
        const int g = lane >> 4, i = lane & 15;
        const size_t nt = col0 / 16 + n8;
        if (nt * 16 >= N)
            continue;
        const uint32_t *src = &lq[n8 * 16 + i][4 * g];
        const u32x4 o = {src[0], src[1], src[2], src[3]};
        *reinterpret_cast<u32x4 *>(packed + (nt * ktiles + kt) * 1024 + lane * 16) = o;
    }
}


// ---- one pass: the matrix stays in registers between the maxima and the weights ----
//
// A group of columns one cache line wide (64 of fp16, 32 of fp32; half a line doubles what the L1 fetches, and stripes of
// 16 fp16 columns that need no exchange took 65-77 us for 11008 x 4096) is shared by `parts` workgroups, each with a
// contiguous range of its k-tiles in registers.  They exchange their column maxima through memory -- a slot per part,
// then a count of the parts that are through, on a line of its own (counts side by side: 62 us instead of 46 at eight
// parts) -- and then each quantises and packs what it holds.  The wait is bounded: parts of a group are neighbours in
// the grid and so run together, but where one is kept off the chip the others read its rows themselves.  A wavefront takes
// units of 32 rows round-robin; a lane holds 4 consecutive rows of the columns that one 16-byte load brings, so that
// its bytes of a column are whole words of the packed tile.
constexpr int kUnit = 32;

template <typename T>
struct GroupShape {
    static constexpr int kCols = 16 / (int)sizeof(T);   // columns of a lane
    static constexpr int kGroup = 8 * kCols;            // columns of a group: 128 bytes of a row
    static constexpr int kLine = 128 / kGroup;          // groups that share a cache line of int8
};

// largest of |x| over the register's values as unsigned integers, which order like them (NaN above everything)
template <typename T>
__device__ __forceinline__ uint32_t max_abs(uint32_t m, uint32_t x)
{
    if constexpr (sizeof(T) == 2) {
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, m),
                                                                     __builtin_bit_cast(u16x2, x & 0x7fff7fffu)));
    } else {
        return m > (x & 0x7fffffffu) ? m : x & 0x7fffffffu;
    }
}

// x without the values that are NaN (0 in their place)
template <typename T>
__device__ __forceinline__ uint32_t drop_nan(uint32_t x)
{
    if constexpr (sizeof(T) == 2)
        return ((x & 0x7fffu) > 0x7c00u ? 0u : x & 0xffffu) | ((x & 0x7fff0000u) > 0x7c000000u ? 0u : x & 0xffff0000u);
    else
        return (x & 0x7fffffffu) > 0x7f800000u ? 0u : x;
}

template <typename T>
__device__ __forceinline__ float value_at(const u32x4 &v, int i)
{
    if constexpr (sizeof(T) == 2) {
        typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
        return (float)__builtin_bit_cast(f16x8, v)[i];
    } else {
        return __uint_as_float(v[i]);
    }
}

template <typename T, int WAVES, int UNITS, bool QOUT>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4))) void quant_group_kernel(
    const T *__restrict__ w, int K, int N, int parts, int ref128, int max_polls, uint32_t *maxima, uint32_t *arrived,
    int8_t *__restrict__ q_out, uint8_t *__restrict__ packed, T *__restrict__ scale)
{
    using S = GroupShape<T>;
    __shared__ uint32_t part[WAVES][S::kGroup];
    __shared__ float s_all[S::kGroup], inv_all[S::kGroup];
    __shared__ int flags[3];    // NaN among the weights; a column without a usable scale; the other parts did not arrive
    __shared__ uint32_t lq[WAVES][S::kGroup][9];   // [column][4-row word] of a unit, one word of padding per column
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int group = blockIdx.x / parts, mine = blockIdx.x % parts;
    if constexpr (QOUT && S::kLine > 2) {
        // From fp32 a row of a group is a quarter of a cache line of q: the groups of a line follow one another on one XCD,
        // whose L2 puts the line together.  (us, two passes / scattered over the XCDs / now: 14336 x 11008 297 / 333 / 296,
        // 11008 x 4096 87 / 90 / 82, 14336 x 14336 380 / 352 / 323.  Halves of a line, from fp16, gain nothing.)
        const int xcd = blockIdx.x % 8, turn = blockIdx.x / 8, id = turn / S::kLine * 8 + xcd;
        group = id / parts * S::kLine + turn % S::kLine;
        mine = id % parts;
        if (group * S::kGroup >= N)
            return;
    }
    const int ktiles = K / 64, kt0 = (int)((long)mine * ktiles / parts), kt1 = (int)((long)(mine + 1) * ktiles / parts);
    const int col0 = group * S::kGroup, quad = lane >> 3, c0 = (lane & 7) * S::kCols;
    const bool cols_in = col0 + c0 < N;    // N % 16 == 0: a lane's columns are in range together
    const T *base = w + (cols_in ? col0 + c0 : N - S::kCols);
    const float nan_to = ref128 ? 1000.f : 0.f;
    const int lo = ref128 ? -128 : -127;

    // The wavefront's units: unit0 + wave, + WAVES, ... below unit1, at most UNITS of them.
    const int unit0 = 2 * kt0, unit1 = 2 * kt1;
    u32x4 v[UNITS][4];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int unit = unit0 + wave + WAVES * u;
        if (unit < unit1) {
            const T *p = base + (size_t)(unit * kUnit + 4 * quad) * N;
#pragma unroll
            for (int it = 0; it < 4; ++it)
                v[u][it] = *reinterpret_cast<const u32x4 *>(p + (size_t)it * N);
        }
    }
    if (threadIdx.x < 3)
        flags[threadIdx.x] = 0;

    // lane maxima to column maxima: thread t < kGroup returns that of column t
    auto column_max = [&](uint32_t (&m)[4]) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
#pragma unroll
            for (int x = 8; x < 64; x *= 2)
                m[d] = max_abs<T>(m[d], (uint32_t)__shfl_xor((int)m[d], x));
        }
        if (quad == 0) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                if constexpr (sizeof(T) == 2) {
                    part[wave][c0 + 2 * d] = m[d] & 0xffffu;
                    part[wave][c0 + 2 * d + 1] = m[d] >> 16;
                } else {
                    part[wave][c0 + d] = m[d];
                }
            }
        }
        __syncthreads();
        uint32_t a = 0;
        if (threadIdx.x < S::kGroup) {
#pragma unroll
            for (int k = 0; k < WAVES; ++k)
                a = a > part[k][threadIdx.x] ? a : part[k][threadIdx.x];
        }
        return a;
    };
    // the same from memory, all units, without the weights that are NaN
    auto column_max_again = [&]() {
        uint32_t m[4] = {0, 0, 0, 0};
        for (int unit = wave; unit < 2 * ktiles; unit += WAVES) {
            const T *p = base + (size_t)(unit * kUnit + 4 * quad) * N;
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const u32x4 x = *reinterpret_cast<const u32x4 *>(p + (size_t)it * N);
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    m[d] = max_abs<T>(m[d], drop_nan<T>(x[d]));
            }
        }
        return column_max(m);
    };

    uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
        if (unit0 + wave + WAVES * u < unit1) {
#pragma unroll
            for (int it = 0; it < 4; ++it)
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    m[d] = max_abs<T>(m[d], v[u][it][d]);
        }
    constexpr uint32_t kInf = sizeof(T) == 2 ? 0x7c00u : 0x7f800000u;
    uint32_t a = column_max(m);
    const bool has_nan = a > kInf;
    if (has_nan)
        flags[0] = 1;
    __syncthreads();
    if (flags[0]) {   // NaN weights are ignored, as on the host
#pragma unroll
        for (int d = 0; d < 4; ++d)
            m[d] = 0;
#pragma unroll
        for (int u = 0; u < UNITS; ++u)
            if (unit0 + wave + WAVES * u < unit1) {
#pragma unroll
                for (int it = 0; it < 4; ++it)
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        m[d] = max_abs<T>(m[d], drop_nan<T>(v[u][it][d]));
            }
        a = column_max(m);
    }
    if (parts > 1) {
        // the first wavefront holds every column's maximum: exchange, count up, wait for the other parts
        if (wave == 0) {
            uint32_t *count = arrived + (size_t)group * kCountStride;
            uint32_t *slots = maxima + (size_t)group * parts * S::kGroup + lane;
            if (lane < S::kGroup)
                __hip_atomic_store(slots + mine * S::kGroup, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the maxima are in memory
            if (lane == 0)
                __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool all = false;
            for (int poll = 0; poll < max_polls && !all; ++poll) {
                all = __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= (uint32_t)parts;
                if (!all)
                    __builtin_amdgcn_s_sleep(8);
            }
            asm volatile("" ::: "memory");
            if (!all)
                flags[2] = 1;
            else if (lane < S::kGroup) {
                uint32_t o[kMaxParts];
#pragma unroll
                for (int p = 0; p < kMaxParts; ++p)
                    o[p] = __hip_atomic_load(slots + min(p, parts - 1) * S::kGroup, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int p = 0; p < kMaxParts; ++p)
                    a = a > o[p] ? a : o[p];
            }
        }
        __syncthreads();
        if (flags[2])   // a part is kept off the chip: its rows are read here
            a = column_max_again();
    }
    if (threadIdx.x < S::kGroup) {
        float m;
        if constexpr (sizeof(T) == 2)
            m = (float)__builtin_bit_cast(_Float16, (uint16_t)a);
        else
            m = __uint_as_float(a);
        const float s = ref128 ? m * (1.f / 128.f) : __fdiv_rn(m, 127.f);
        s_all[threadIdx.x] = s;
        if (mine == 0 && col0 + (int)threadIdx.x < N)
            scale[col0 + threadIdx.x] = static_cast<T>(s);
        const bool usable = !has_nan && s > kLeastScale && s < kLargestScale;
        inv_all[threadIdx.x] = usable ? __fdiv_rn(1.f, s) : 0.f;
        if (!usable)
            flags[1] = 1;
    }
    __syncthreads();

    float inv[S::kCols];
#pragma unroll
    for (int i = 0; i < S::kCols; ++i)
        inv[i] = inv_all[c0 + i];
    // The lane's columns without a usable scale (zero, tiny, huge, not finite, or with a NaN among these rows), and those
    // that are such a column in any lane: their weights are divided one by one from the registers, and no others pay for
    // that.  (us, two passes / the whole group read again and divided for one such column / now, a zero column in 32: 4096 x
    // 4096 fp16 26.9 / 32.4 / 24.0, 5120 x 15360 82 / 114 / 81, 4096 x 11008 fp32 78 / 92 / 69.)
    unsigned bare = 0, bare_any = 0;
    if (flags[1] != 0) {
#pragma unroll
        for (int i = 0; i < S::kCols; ++i) {
            bare |= (inv[i] == 0.f ? 1u : 0u) << i;
            bare_any |= (__any(inv[i] == 0.f) ? 1u : 0u) << i;
        }
    }
    auto divide_bare = [&](const u32x4 (&x)[4], uint32_t (&word)[S::kCols]) {
        for (unsigned rest = bare_any; rest != 0; rest &= rest - 1) {
            const int i = __builtin_ctz(rest), d = i * (int)sizeof(T) / 4;
            const float s = s_all[c0 + i];
            uint32_t o = 0;
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                uint32_t r = x[it][0];
#pragma unroll
                for (int k = 1; k < 4; ++k)
                    r = d == k ? x[it][k] : r;
                float xi;
                if constexpr (sizeof(T) == 2)
                    xi = (float)__builtin_bit_cast(_Float16, (uint16_t)(r >> (i % 2 * 16)));
                else
                    xi = __uint_as_float(r);
                o |= (uint32_t)(quant_one(xi, s, nan_to, lo) + 128) << (8 * it);
                __builtin_amdgcn_sched_barrier(0);   // one division at a time: four do not fit beside the matrix
            }
#pragma unroll
            for (int k = 0; k < S::kCols; ++k)
                word[k] = k == i && (bare >> k & 1) ? o : word[k];
        }
    };

    // the unit's words -- four rows of a column, q + 128 -- leave
    auto store = [&](const uint32_t (&word)[S::kCols], int unit) {
        if constexpr (QOUT) {
            if (cols_in) {
                // words of four rows to words of four columns
                uint32_t o[4][S::kCols / 4];
#pragma unroll
                for (int h = 0; h < S::kCols / 4; ++h) {
                    const uint32_t *c = word + 4 * h;
                    const uint32_t t0 = __builtin_amdgcn_perm(c[1], c[0], 0x05010400u);
                    const uint32_t t1 = __builtin_amdgcn_perm(c[1], c[0], 0x07030602u);
                    const uint32_t t2 = __builtin_amdgcn_perm(c[3], c[2], 0x05010400u);
                    const uint32_t t3 = __builtin_amdgcn_perm(c[3], c[2], 0x07030602u);
                    o[0][h] = __builtin_amdgcn_perm(t2, t0, 0x05040100u) ^ 0x80808080u;
                    o[1][h] = __builtin_amdgcn_perm(t2, t0, 0x07060302u) ^ 0x80808080u;
                    o[2][h] = __builtin_amdgcn_perm(t3, t1, 0x05040100u) ^ 0x80808080u;
                    o[3][h] = __builtin_amdgcn_perm(t3, t1, 0x07060302u) ^ 0x80808080u;
                }
                int8_t *q = q_out + (size_t)(unit * kUnit + 4 * quad) * N + col0 + c0;
#pragma unroll
                for (int it = 0; it < 4; ++it)
                    __builtin_memcpy(__builtin_assume_aligned(q + (size_t)it * N, S::kCols < 8 ? S::kCols : 8), o[it],
                                     S::kCols);
            }
        }
        // Into packed order through a slab of the wavefront's own: no barrier.  A unit is the g = 0, 1 or the g = 2, 3
        // half of a k-tile, 512 bytes of each of the group's n-tiles.
#pragma unroll
        for (int i = 0; i < S::kCols; ++i)
            lq[wave][c0 + i][quad] = word[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int p = 0; p < S::kGroup / 32; ++p) {
            const int piece = p * 64 + lane, n16 = piece >> 5, g = (piece >> 4) & 1, i = piece & 15;
            const int nt = col0 / 16 + n16;
            const uint32_t *src = &lq[wave][n16 * 16 + i][4 * g];
            const u32x4 o = {src[0], src[1], src[2], src[3]};
            if (nt * 16 < N)
                *reinterpret_cast<u32x4 *>(packed + ((size_t)nt * ktiles + (unit >> 1)) * 1024 + (unit & 1) * 512 +
                                           (g * 16 + i) * 16) = o;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    // v = x / s + 128 to within 2^-16 (x times the rounded reciprocal: 2^-17 at |x / s| <= 128; the sum, below 256:
    // 2^-17), and the correctly rounded quotient of the host is within 2^-17 of the exact one: unless v lies within
    // 2^-15 of a half, both round to the same integer.  The conversion rounds to nearest and clamps to 0 .. 255, i.e. +128
    // to 127.  Units with a weight near a half (one in eight of random weights) are left to the second loop, which reads
    // them again and divides.  (A bare column's value is 128 or NaN here: not near, and the minimum skips a NaN.)
    unsigned again = 0;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int unit = unit0 + wave + WAVES * u;
        if (unit >= unit1)
            continue;
        uint32_t word[S::kCols];
#pragma unroll
        for (int i = 0; i < S::kCols; ++i)
            word[i] = 0;
        float near = 1.f;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
#pragma unroll
            for (int i = 0; i < S::kCols; i += 2) {
                const float f0 = __builtin_fmaf(value_at<T>(v[u][it], i), inv[i], 128.f);
                const float f1 = __builtin_fmaf(value_at<T>(v[u][it], i + 1), inv[i + 1], 128.f);
                word[i] = __builtin_amdgcn_cvt_pk_u8_f32(f0, it, word[i]);
                word[i + 1] = __builtin_amdgcn_cvt_pk_u8_f32(f1, it, word[i + 1]);
                // (the compiler's minimum of two magnitudes is four instructions)
                asm("v_min3_f32 %0, %0, abs(%1), abs(%2)"
                    : "+v"(near)
                    : "v"(__builtin_amdgcn_fractf(f0) - 0.5f), "v"(__builtin_amdgcn_fractf(f1) - 0.5f));
            }
        }
#pragma unroll
        for (int i = 0; i < S::kCols; ++i)
            asm volatile("" : "+v"(word[i]));   // not after the branch, with all 32 quotients in registers
        if (__any(near < kNear)) {
            again |= 1u << u;
            continue;
        }
        if (bare_any != 0)
            divide_bare(v[u], word);
        store(word, unit);
    }
    while (again != 0) {
        const int u = __builtin_ctz(again), unit = unit0 + wave + WAVES * u;
        again &= again - 1;
        uint32_t word[S::kCols];
#pragma unroll
        for (int i = 0; i < S::kCols; ++i)
            word[i] = 0;
        const T *p = base + (size_t)(unit * kUnit + 4 * quad) * N;
        u32x4 x[4];
#pragma unroll
        for (int it = 0; it < 4; ++it)
            x[it] = *reinterpret_cast<const u32x4 *>(p + (size_t)it * N);
#pragma unroll
        for (int it = 0; it < 4; ++it) {
#pragma unroll
            for (int i = 0; i < S::kCols; ++i) {
                const float xi = value_at<T>(x[it], i), f = __builtin_fmaf(xi, inv[i], 128.f);
                word[i] = __builtin_amdgcn_cvt_pk_u8_f32(f, it, word[i]);
                if (__builtin_fabsf(__builtin_amdgcn_fractf(f) - 0.5f) < kNear) {
                    const int t = quant_one(xi, s_all[c0 + i], nan_to, lo) + 128;
                    word[i] = (word[i] & ~(0xffu << (8 * it))) | (uint32_t)t << (8 * it);
                }
            }
        }
        if (bare_any != 0)
            divide_bare(x, word);
        store(word, unit);
    }
}

template <typename T, int WAVES, int UNITS>
int launch_groups(const void *w, size_t K, size_t N, int parts, int ref128, int8_t *q, int8_t *packed, void *scale,
                  uint32_t *counts, hipStream_t st)
{
    const size_t groups = (N + GroupShape<T>::kGroup - 1) / GroupShape<T>::kGroup, n = groups * kCountStride;
    if (parts > 1) {
        hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, counts, n);
        EET_HIP_CHECK(hipGetLastError());
    }
    const int limit = eet::tuning().pack_poll_limit;
    const auto kernel = q != nullptr ? quant_group_kernel<T, WAVES, UNITS, true> : quant_group_kernel<T, WAVES, UNITS, false>;
    constexpr size_t kLine = GroupShape<T>::kLine;
    const size_t grid = q != nullptr && kLine > 2 ? ((groups + kLine - 1) / kLine * parts + 7) / 8 * 8 * kLine : groups * parts;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * WAVES), 0, st, static_cast<const T *>(w), (int)K, (int)N, parts,
                       ref128, limit >= 0 ? limit : kMaxPolls, counts + n, counts, q, reinterpret_cast<uint8_t *>(packed),
                       static_cast<T *>(scale));
    EET_HIP_CHECK(hipGetLastError());
    return EET_OK;
}

// One pass or two, measured at some 700 sizes (K 64 .. 32768, N 16 .. 262144, up to 450 M weights, from HBM) with the second
// pass as it was when it divided per thread and column (3-15 % slower than now); us, two passes as they are / one.
// fp32: one (4096 x 4096 28.7 / 23.1, 5120 x 13696 114.5 / 85.4, 16384 x 16384 437 / 280).
// fp16 has twice the weights to a byte, so that the quantising of a workgroup's share, which nothing overlaps where the grid
// fits the chip once, weighs more.  Up to 36 M weights one pass wins by its two launches less (1024 x 1024 11.9 / 10.5, 4096
// x 4096 20.8 / 20.2, 16384 x 1024 21.0 / 19.8), where its workgroups fill the chip (plan_pack); from there the registers of the
// chip no longer hold every matrix in one round, while the second pass of the other way is read from the Infinity Cache; with
// more rounds, and what does not fit that cache, one pass is ahead again (5120 x 13696 67.6 / 62.2, 5120 x 15360 75.2 / 74.3,
// 8192 x 16384 129 / 110).
// fp16 with the row-major output, whose stores are half lines of rows: only where the whole matrix is in the 16-wavefront
// form (4096 x 4096 28.6 / 25.0) or small (512 x 22016 23.9 / 16.9); above, it is anything from 0.82 (8192 x 32000) to 1.22
// (2560 x 12288 43 / 53; 20480 x 4096 100 / 122, 4096 x 32768 162 / 186).
// Either type: rows for less than a unit per wavefront leave the workgroups nearly empty, which counts once there are many
// of them (K = 64: N 50272 0.74-0.81, 98304 0.99-1.09, 262144 1.40; K = 128: 151936 0.86, 262144 1.05; K = 256 never).
// fp16 with more than 20480 rows and few columns: the parts of a group end at 16 (28672 x 128 1.13, 32768 x 256 1.19, x 640
// 0.95; 20480 x 256 1.00).
template <typename T>
bool one_pass_wins(size_t K, size_t N, bool unprocessed, bool wide)
{
    const size_t n = K * N, units = K / kUnit, groups = (N + GroupShape<T>::kGroup - 1) / GroupShape<T>::kGroup;
    if (units < 8 && groups > 800 * units)
        return false;
    if (sizeof(T) == 4)
        return true;
    if (units > 640 && groups <= 8)
        return false;
    return unprocessed ? n <= (wide ? 24000000 : 15000000) : n <= 36000000 || n >= 70000000;
}

// How many workgroups share a column group: as many as its rows need, and as many as the chip still takes in one round.
int parts_of(size_t units, size_t groups, int waves, int held, size_t slots)
{
    const size_t need = (units + waves * held - 1) / (waves * held), most = units / waves;
    size_t parts = slots / groups < (size_t)kMaxParts ? slots / groups : (size_t)kMaxParts;
    parts = parts < most ? parts : most;
    return (int)(parts > need ? parts : need);
}

// What a call runs as: wavefronts of a workgroup and workgroups of a column group, or no wavefronts for two passes.
struct PackPlan {
    int waves, parts;
};

template <typename T>
PackPlan plan_pack(size_t K, size_t N, bool unprocessed, size_t ws_bytes)
{
    const size_t units = K / kUnit, groups = (N + GroupShape<T>::kGroup - 1) / GroupShape<T>::kGroup;
    const int wide = parts_of(units, groups, 16, 4, 256), narrow = parts_of(units, groups, 8, 5, 512);
    const bool fits = wide <= kMaxParts && groups * wide <= 256;
    // Groups of fp16 columns shared by workgroups that leave more than 18 % of the slots empty, or that are three and more
    // to a group and a few too many for one round: the two passes, which have neither, are ahead where a workgroup's
    // wavefronts hold two units and more (2048 rows) and the matrix has 11 M weights, 16 M with three workgroups to a group.  Measured
    // at 158 sizes of 11-36 M weights, two passes / one, by the share of the slots: up to 0.75 0.84 .. 1.04 (0.95 in the mean:
    // 2560 x 11008 32.6 / 36.8 us, 4096 x 5632 28.5 / 32.9), to 0.82 0.81 .. 1.04 (0.95: 2432 x 12800 35.2 / 43.8, 5120 x
    // 6656 38.3 / 42.9), to 0.84 0.98 .. 1.05, above 0.93 .. 1.12 (1.03), 1.01 .. 1.1 0.78 .. 0.89 (3072 x 11008 38.3 / 42.9).
    // Left with one pass by the other lines: 1856 x 6208 (0.76) 20.9 / 18.9, 1728 x 6400 (0.78) 19.6 / 18.1, 2752 x 4224
    // (0.77, three) 19.8 / 19.2.  Groups with a workgroup each need no exchange and stay (1216 x 12288, 0.75: 17.9 / 15.4).
    const size_t slots = fits ? 256 : 512, parts = fits ? wide : narrow, total = groups * parts;
    const bool idle = sizeof(T) == 2 && parts > 1 && units >= 64 && K * N > (parts > 2 ? 16000000 : 11000000) &&
                      (total * 100 < slots * 82 || (total > slots && total * 10 <= slots * 11 && parts > 2));
    // (threads of a grid are counted in 32 bits, and the kernel's column indices are int; a row of workgroups to spare)
    if (ws_bytes < eet_quantize_pack_device_workspace(N) || idle || !one_pass_wins<T>(K, N, unprocessed, fits) ||
        (!fits && (narrow > kMaxParts || groups * narrow >= ((size_t)1 << 32) / (64 * 8) - 64)))
        return {0, 0};
    return fits ? PackPlan{16, wide} : PackPlan{8, narrow};
}

template <typename T>
int run(const void *w, size_t K, size_t N, int mode, int8_t *q, int8_t *packed, void *scale, uint32_t *ws, size_t ws_bytes,
        hipStream_t st)
{
    const int ref128 = mode == EET_QUANT_REF128 ? 1 : 0;
    const PackPlan plan = plan_pack<T>(K, N, q != nullptr, ws_bytes);
    if (plan.waves == 16)
        return launch_groups<T, 16, 4>(w, K, N, plan.parts, ref128, q, packed, scale, ws, st);
    if (plan.waves == 8)
        return launch_groups<T, 8, 5>(w, K, N, plan.parts, ref128, q, packed, scale, ws, st);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st, ws, N);
    EET_HIP_CHECK(hipGetLastError());
    const dim3 g1((unsigned)((N + 64 * kColsPerThread - 1) / (64 * kColsPerThread)),
                  (unsigned)((K + kMaxRows - 1) / kMaxRows));
    hipLaunchKernelGGL(colmax_kernel<T>, g1, dim3(256), 0, st, static_cast<const T *>(w), K, N, ws);
    EET_HIP_CHECK(hipGetLastError());
    const size_t turns = ((size_t)g1.x * g1.y + 7) / 8, rows = turns < kMostTurns ? turns : kMostTurns;
    const dim3 g2(8 * (kMaxRows / 64) * (kChunkCols / kTileCols), (unsigned)rows, (unsigned)((turns + rows - 1) / rows));
    hipLaunchKernelGGL(quant_pack_kernel<T>, g2, dim3(256), 0, st, static_cast<const T *>(w), K, N, ref128, ws, q,
                       reinterpret_cast<uint8_t *>(packed), static_cast<T *>(scale));
    EET_HIP_CHECK(hipGetLastError());
    return EET_OK;
}

}  // namespace

// A count per group of columns (32 columns or more) and, in whole groups (64 columns or fewer), the column maxima of each
// part; the two passes use N words of it.
extern "C" size_t eet_quantize_pack_device_workspace(size_t N)
{
    return ((N + 31) / 32 * kCountStride + (N + 63) / 64 * 64 * kMaxParts) * sizeof(uint32_t);
}

static int check_pack_args(const char *fn, int w_dtype, size_t K, size_t N)
{
    EET_REQUIRE(w_dtype == EET_DTYPE_F32 || w_dtype == EET_DTYPE_F16, EET_ERR_INVALID_ARGUMENT,
                "%s: w_dtype must be EET_DTYPE_F32 or EET_DTYPE_F16, got %d", fn, w_dtype);
    EET_REQUIRE(K > 0 && N > 0 && K % 64 == 0 && N % 16 == 0, EET_ERR_UNSUPPORTED_SHAPE,
                "%s: need K %% 64 == 0 and N %% 16 == 0, got K=%zu N=%zu", fn, K, N);
    EET_REQUIRE(K / 64 <= 65535 && (K + kMaxRows - 1) / kMaxRows <= 65535, EET_ERR_UNSUPPORTED_SHAPE,
                "%s: K = %zu exceeds the grid limit", fn, K);
    return EET_OK;
}

extern "C" int eet_quantize_pack_device_shape(int w_dtype, size_t K, size_t N, int unprocessed, size_t workspace_bytes,
                                              int *waves, int *parts)
{
    const char *fn = "eet_quantize_pack_device_shape";
    EET_REQUIRE(waves && parts, EET_ERR_INVALID_ARGUMENT, "%s: null pointer", fn);
    if (int rc = check_pack_args(fn, w_dtype, K, N))
        return rc;
    const PackPlan plan = w_dtype == EET_DTYPE_F32 ? plan_pack<float>(K, N, unprocessed != 0, workspace_bytes)
                                                   : plan_pack<_Float16>(K, N, unprocessed != 0, workspace_bytes);
    *waves = plan.waves, *parts = plan.parts;
    return EET_OK;
}

extern "C" int eet_quantize_pack_device(const void *w, int w_dtype, size_t K, size_t N, int mode, int8_t *q,
                                        int8_t *packed, void *scale, void *workspace, size_t workspace_bytes,
                                        void *stream)
{
    EET_REQUIRE(w && packed && scale, EET_ERR_INVALID_ARGUMENT, "eet_quantize_pack_device: null pointer");
    if (int rc = check_pack_args("eet_quantize_pack_device", w_dtype, K, N))
        return rc;
    EET_REQUIRE(mode == EET_QUANT_REF128 || mode == EET_QUANT_SYM127, EET_ERR_INVALID_ARGUMENT,
                "eet_quantize_pack_device: unknown mode %d", mode);
    EET_REQUIRE((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(packed)) % 16 == 0 &&
                    (q == nullptr || reinterpret_cast<uintptr_t>(q) % 8 == 0),
                EET_ERR_INVALID_ARGUMENT, "eet_quantize_pack_device: w and packed need 16-byte, q 8-byte alignment");
    EET_REQUIRE(workspace != nullptr && workspace_bytes >= N * sizeof(uint32_t) &&
                    reinterpret_cast<uintptr_t>(workspace) % 4 == 0,
                EET_ERR_WORKSPACE, "eet_quantize_pack_device: workspace of %zu bytes needed, %zu given",
                N * sizeof(uint32_t), workspace_bytes);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (w_dtype == EET_DTYPE_F32)
        return run<float>(w, K, N, mode, q, packed, scale, static_cast<uint32_t *>(workspace), workspace_bytes, st);
    return run<_Float16>(w, K, N, mode, q, packed, scale, static_cast<uint32_t *>(workspace), workspace_bytes, st);
}
