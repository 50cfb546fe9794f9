// The output head of a decode step: out[M][N] = x[M][K] * w[N][K]^T in fp16 with fp32 sums, M <= 16 rows (one per
// sequence), w the row-major fp16 matrix of the checkpoint.
//
// HBM-bound: 2*N*K weight bytes, each read once.  A workgroup owns NT tiles of 16 output columns over the whole k
// range; its wavefronts take blocks of 64 k (one 128-byte line per row) in turn, so that together they stream NT * 16
// adjacent rows.  Weights and activations are loaded as the operands of v_mfma_f32_16x16x32_f16 (lane (g, i): row i,
// 16 bytes at 16 g) into a ring of U register slots, a slot being refilled as soon as it is consumed; nothing goes
// through LDS before the wavefronts' fp32 sums meet there.  Requests past the last k block have the top offset bit
// set: they return zeros and touch no memory, which keeps the loop free of branches around loads.  The two halves of
// a line are two requests: with the non-temporal bit the second one missed again (M = 1, 64000 <- 5120: 138 us
// against 108).
// Three things set NT: the tiles of the CU with the most workgroups (whole rounds of 256, 16 K weights each), the
// activations that every workgroup reads whole from L2 (at 16 rows as many bytes as a tile, at 0.4 of the cost), and
// the start and the meeting of its wavefronts (as long as 1024 k of a tile).  head_tiles takes the smallest sum; over
// 832 sizes (K 512 .. 8192, N 1024 .. 256000, M 1 .. 16; graph replays, weights from HBM) it is 0.6 % behind the best of
// the three NT on average, 18 % at most.  us, NT = 1 / 2 / 4, M = 1 and 16: 4096 <- 4096 8.3 / 11.2 / 17.7, 10.2 / 13.5 /
// 21.0; 8000 <- 1024 5.9 / 5.5 / 6.7, 7.0 / 5.9 / 7.5; 10240 <- 4096 19.5 / 23.6 / 19.4, 25.5 / 26.6 / 22.6; 20480 <- 4096
// 31.2 / 36.5 / 42.5, 42.5 / 41.4 / 45.6; 32000 <- 2048 26.3 / 25.0 / 26.9, 35.1 / 30.6 / 28.5; 32000 <- 4096 46.1 / 48.0 /
// 48.4, 65.1 / 55.1 / 51.3.  (Thresholds on the number of tiles, from four matrices: 5 % behind on average, 53 % at most.)
// 64000 <- 5120 at M = 16 took 127 us against the library's 110: matrices that large are refused here (a limit of this
// kernel's speed, not of its addressing) and left to it.
// Large matrices are streamed by head_resident_kernel instead, one workgroup per CU; see there.
#include <hip/hip_runtime.h>

#include "common.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// NT: tiles of 16 columns per workgroup.
template <int NT, int WAVES, int U>
__global__ __launch_bounds__(64 * WAVES) void head_kernel(const _Float16 *__restrict__ x, long x_stride,
                                                          const _Float16 *__restrict__ w, _Float16 *__restrict__ out,
                                                          int M, int N, int K)
{
    __shared__ float part[WAVES][NT][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (NT * 16);
    const int blocks = K / 64;
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#if defined(__HIP_DEVICE_COMPILE__)  // buffer-resource builtins exist in the device pass only
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16 *>(w + (size_t)n0 * K), 0, (unsigned)min(NT * 16, N - n0) * (unsigned)K * 2u, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16 *>(x), 0, ((unsigned)(M - 1) * (unsigned)x_stride + (unsigned)K) * 2u, 0x00020000);
    const unsigned wlane = (unsigned)i * (unsigned)K * 2u + (unsigned)g * 16u;
    const unsigned xlane = i < M ? (unsigned)i * (unsigned)x_stride * 2u + (unsigned)g * 16u : 0x80000000u;
    u32x4 wv[U][NT][2], xv[U][2];
    auto request = [&](int u, int kb) {
        const unsigned off = kb < blocks ? (unsigned)kb * 128u : 0x80000000u;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                wv[u][t][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    wr, (wlane + (unsigned)t * 16u * (unsigned)K * 2u + h * 64u + off) | (off & 0x80000000u), 0, 0));
#pragma unroll
        for (int h = 0; h < 2; ++h)
            xv[u][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                xr, (xlane + h * 64u + off) | ((off | xlane) & 0x80000000u), 0, 0));
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
        request(u, wave + u * WAVES);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int kb = wave; kb < blocks; kb += U * WAVES) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, xv[u][h]),
                                                                    __builtin_bit_cast(half8, wv[u][t][h]), acc[t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            request(u, kb + (u + U) * WAVES);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#endif
    // lane (g, i) of a tile holds rows 4 g + r of column i
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            part[wave][t][r][lane] = acc[t][r];
    __syncthreads();
    for (int e = threadIdx.x; e < NT * 256; e += 64 * WAVES) {
        const int l = e & 63, r = (e >> 6) & 3, t = e >> 8;
        const int row = (l >> 4) * 4 + r, col = n0 + t * 16 + (l & 15);
        if (row >= M || col >= N)
            continue;
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v)
            s += part[v][t][r][l];
        out[(size_t)row * N + col] = (_Float16)s;
    }
}

// The same with one workgroup of 16 wavefronts per CU, which keeps the activations in LDS and walks over the tiles
// blockIdx.x, + gridDim.x, ...: they are read from L2 once per CU instead of once per NT tiles, and nothing starts, meets
// or drains between two tiles.  Each wavefront has a contiguous part of the k range; the ring of requests runs on from one
// tile into the next.  At a tile's end the wavefronts' fp32 sums go to one of two LDS buffers, one barrier, and one
// wavefront (in turn) adds and stores them while the others are at the next tile; the buffer is written again behind the next
// barrier but one, which that wavefront reaches after its reads.
// HBM-bound: 32000 <- 4096 is 5.9 TB/s at M = 1, where a kernel that only reads so many bytes takes 42-43 us (6.2).  us,
// head_kernel / this, M = 1, 8, 16: 32000 <- 4096 48.6 / 43.6, 50.9 / 45.9, 51.0 / 48.6; 20480 <- 4096 31.1 / 29.2,
// 35.6 / 30.8, 41.3 / 32.6; 50272 <- 4096 85 / 69, 91 / 72, 97 / 76; 32000 <- 2048 26.5 / 26.3, 27.8 / 28.3, 28.1 / 29.1.
// Rings of 3, 4, 6 and 8 slots: equal to 6 % slower.  Behind the last layer of a decoder, 32000 <- 4096, the gain is smaller
// (the head of M = 16 beams 52.3 / 50.4, of 8 sequences 45.9 / 45.8).
constexpr int kResidentWaves = 16, kResidentRing = 2, kResidentHalves = 65536;   // the most activations: 128 KiB

__global__ __launch_bounds__(64 * kResidentWaves) void head_resident_kernel(const _Float16 *__restrict__ x, long x_stride,
                                                                            const _Float16 *__restrict__ w,
                                                                            _Float16 *__restrict__ out, int M, int N, int K)
{
    constexpr int W = kResidentWaves, U = kResidentRing;
    __shared__ f32x4 part[2][W][64];
    __shared__ u32x4 xs[kResidentHalves / 8];   // [M][K / 8] pieces of 16 bytes, XORed with the row against bank conflicts
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int blocks = K / 64, pieces = K / 8, tiles = N / 16;
    const int kb0 = blocks * wave / W, nb = blocks * (wave + 1) / W - kb0;   // at least one: 16 blocks and more
    const int mine = (tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
#if defined(__HIP_DEVICE_COMPILE__)  // buffer-resource builtins exist in the device pass only
    const unsigned tile_bytes = 32u * (unsigned)K;
    const __amdgpu_buffer_rsrc_t wr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(w), 0, (unsigned)tiles * tile_bytes, 0x00020000);
    const unsigned wlane = (unsigned)i * (unsigned)K * 2u + (unsigned)g * 16u;
    u32x4 wv[U][2];
    int turn = 0, kb = 0;   // the next request
    auto request = [&](int u) {
        const bool in = turn < mine;   // past the last tile the top offset bit is set: zeros, no memory touched
        const unsigned at = in ? (blockIdx.x + (unsigned)turn * gridDim.x) * tile_bytes + (unsigned)(kb0 + kb) * 128u : 0u;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            wv[u][h] = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, (in ? wlane : 0x80000000u) + h * 64u, at, 0));
        if (++kb == nb)
            kb = 0, ++turn;
    };
    const int total = M * pieces;
    constexpr int kAtOnce = 8;
    for (int p0 = 0; p0 < total; p0 += 64 * W * kAtOnce) {
        u32x4 v[kAtOnce];
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int p = min(p0 + q * 64 * W + tid, total - 1), row = p / pieces;
            v[q] = *reinterpret_cast<const u32x4 *>(x + (size_t)row * x_stride + (p - row * pieces) * 8);
        }
        if (p0 == 0) {   // the first weights behind the first activations
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                request(u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int p = p0 + q * 64 * W + tid, row = p / pieces;
            if (p < total)
                xs[row * pieces + ((p - row * pieces) ^ (row & 7))] = v[q];
        }
    }
    __syncthreads();
    const int xrow = min(i, M - 1);   // rows past M repeat the last: their results are not stored
    const u32x4 *xl = xs + xrow * pieces;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int t = 0, b = 0;
    while (t < mine) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u32x4 xv = xl[((kb0 + b) * 8 + h * 4 + g) ^ (xrow & 7)];
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, xv),
                                                             __builtin_bit_cast(half8, wv[u][h]), acc, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            request(u);
            __builtin_amdgcn_sched_barrier(0);
            ++b;
            if (b == nb && t < mine) {
                part[t & 1][wave][lane] = acc;
                acc = f32x4{0.f, 0.f, 0.f, 0.f};
                // (not __syncthreads(), which would wait for the requests as well)
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (wave == t % W) {
                    f32x4 s = part[t & 1][0][lane];
#pragma unroll
                    for (int v = 1; v < W; ++v)
                        s += part[t & 1][v][lane];
                    const size_t col = (size_t)(blockIdx.x + (unsigned)t * gridDim.x) * 16 + i;
#pragma unroll
                    for (int r = 0; r < 4; ++r)   // lane (g, i) of a tile holds rows 4 g + r of column i
                        if (4 * g + r < M)
                            out[(size_t)(4 * g + r) * N + col] = (_Float16)s[r];
                }
                ++t;
            }
            if (b == nb)
                b = 0;
        }
    }
#endif
}

// Tiles per workgroup, see above; 0: head_resident_kernel.  That one costs a tile and 210 k of start per turn, the
// activations once, and its own start, more where its wavefronts have unequal parts; rows a multiple of 8 KiB apart take
// head_kernel a quarter longer than the sum says (K = 8192, outside the fit, alike: 24576 rows M = 8 83.1 / 77.5 us, 32000 107.1
// / 98.6, and this one ahead at all of ten sizes), rows 4 KiB apart take this one 15 % longer (12 KiB apart, outside the
// fit, it would be ahead by 1 to 12 %).  Fewer than five turns are left to head_kernel (4096 <- 1024 3.3 / 4.8 us).  Over
// 656 sizes (K 1024 .. 5120, N 4096 .. 128256, M 1 .. 16; weights from HBM) the two take 0.956 of head_kernel's time, 0.71 at
// best, 1.03 at worst.
int head_tiles(int tiles, int M, int K)
{
    int best = 1;
    float least = 0.f;
    for (int nt : {1, 2, 4}) {
        const int workgroups = (tiles + nt - 1) / nt, rounds = (workgroups + 255) / 256;
        const float cost = (float)rounds * ((float)nt + 0.4f * (float)M / 16.f + 1024.f / (float)K);
        if (nt == 1 || cost < least)
            best = nt, least = cost;
    }
    if (tiles > 1024 && K >= 64 * kResidentWaves && M * K <= kResidentHalves) {
        const float turns = (float)((tiles + 255) / 256), uneven = (float)((K / 64 + kResidentWaves - 1) / kResidentWaves * 1024) / K;
        const float cost = (turns * (1.f + 210.f / (float)K) + 0.42f * (float)M / 16.f + 0.63f) * (0.75f + 0.25f * uneven);
        if (cost * (K % 4096 == 2048 ? 1.15f : 1.f) < least * (K % 4096 == 0 ? 1.25f : 1.f))
            return 0;
    }
    return best;
}

}  // namespace

static int check_head_sizes(const char *fn, int M, int N, int K)
{
    EET_REQUIRE(M > 0 && M <= 16 && N > 0 && K > 0 && K % 64 == 0 && N % 16 == 0, EET_ERR_UNSUPPORTED_SHAPE,
                "%s: need 1 <= M <= 16, K %% 64 == 0 and N %% 16 == 0, got M=%d N=%d K=%d", fn, M, N, K);
    EET_REQUIRE((size_t)N * K <= ((size_t)1 << 28), EET_ERR_UNSUPPORTED_SHAPE,
                "%s: a matrix of %d x %d is larger than 2^28 elements", fn, N, K);
    return EET_OK;
}

extern "C" int eet_head_f16_shape(int M, int N, int K, int *tiles)
{
    EET_REQUIRE(tiles, EET_ERR_INVALID_ARGUMENT, "eet_head_f16_shape: null pointer");
    if (int rc = check_head_sizes("eet_head_f16_shape", M, N, K))
        return rc;
    *tiles = head_tiles(N / 16, M, K);
    return EET_OK;
}

extern "C" int eet_head_f16(const void *x, long x_stride, const void *w, void *out, int M, int N, int K, void *stream)
{
    EET_REQUIRE(x && w && out, EET_ERR_INVALID_ARGUMENT, "eet_head_f16: null pointer");
    if (int rc = check_head_sizes("eet_head_f16", M, N, K))
        return rc;
    EET_REQUIRE(x_stride >= K && x_stride % 8 == 0 && ((size_t)(M - 1) * x_stride + K) * 2 <= ((size_t)1 << 31),
                EET_ERR_INVALID_ARGUMENT, "eet_head_f16: x_stride %ld must be a multiple of 8, at least K", x_stride);
    EET_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0, EET_ERR_INVALID_ARGUMENT,
                "eet_head_f16: x and w need 16-byte alignment");
    const int tiles = N / 16, nt = head_tiles(tiles, M, K);
    if (nt == 0) {
        hipLaunchKernelGGL(head_resident_kernel, dim3(tiles < 256 ? tiles : 256), dim3(64 * kResidentWaves), 0,
                           static_cast<hipStream_t>(stream), static_cast<const _Float16 *>(x), x_stride,
                           static_cast<const _Float16 *>(w), static_cast<_Float16 *>(out), M, N, K);
        EET_HIP_CHECK(hipGetLastError());
        return EET_OK;
    }
    auto kern = nt == 4 ? head_kernel<4, 8, 1> : nt == 2 ? head_kernel<2, 8, 2> : head_kernel<1, 8, 2>;
    hipLaunchKernelGGL(kern, dim3((tiles + nt - 1) / nt), dim3(512), 0, static_cast<hipStream_t>(stream),
                       static_cast<const _Float16 *>(x), x_stride, static_cast<const _Float16 *>(w),
                       static_cast<_Float16 *>(out), M, N, K);
    EET_HIP_CHECK(hipGetLastError());
    return EET_OK;
}
