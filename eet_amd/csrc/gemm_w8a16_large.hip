// Large-M fused dequant-GEMM (M > 32: prompts, and decode steps of more than 32 sequences; see slabs_win for the calls
// of up to 64 rows that stay with the small-M kernel).
//
// Replaces the tensor-core side of fastertransformer::gemm_fp16_int_bias_act<uint8_t>
// (3rdparty/cutlass_kernels/fpA_intB_gemm/fpA_intB_gemm_template.h:48-177).
//
// A workgroup of WM x WN wavefronts owns a block of WM*TM*16 rows x WN*TN*16 channels; each wavefront owns
// TM x TN tiles of v_mfma_f32_16x16x32_f16 (TM*TN*4 fp32 accumulator registers).  Both operands of a 64-wide
// k-tile are copied global -> LDS by the memory pipeline itself (buffer_load_dwordx4 ... lds: no staging
// registers, no ds_write) into a ring of D stages:
//   weights      the packed 1 KiB tiles as they are: lane l of a wavefront reads its 16 bytes back with one
//                conflict-free ds_read_b128, already in operand order, and widens them (one vector
//                instruction per weight) while the matrix cores work on the step before;
//   activations  16 "super-rows" of 256 B per pair of m-tiles (2u, 2u + 1), super-row j holding row j of both:
//                the 16-byte piece 2g + h of row j of m-tile 2u + e sits at slot (4 * (2e + h) + g) ^ j, which
//                lets a ds_read_b128 of the whole wavefront run at the full 256 B/clk of the LDS (128-byte rows
//                with any XOR of the row index reach 150 B/clk); the lanes of one copy fetch whole 128-byte lines.
//
// What bounds it.  At thousands of rows the power the matrix cores draw (1.25-1.35 PFLOP/s at the clock that is
// left), below that the way the k-loop is fed: an XCD's L2 hands a CU 118 KB/us when everything hits, but with
// misses among the requests the two times add (60 KB/us at one miss in five), so what counts is few bytes per
// flop, i.e. large blocks, on all 256 CUs at once.  The earlier form of this kernel kept the weights in registers,
// two k-tiles ahead, and had to wait for all but the copies of the current step before each barrier (a copy whose
// rows are all past M completes at once, ahead of older ones, and makes a deeper counted wait unsafe); a workgroup
// alone on its CU then took 0.26-0.33 us per k-tile whatever its size.  Here
//   * every copy touches memory (rows past M re-read row M - 1, a k-tile past the end re-reads the last one), so
//     completion is in order, the wait before the hand-over counts the copies of D - 2 whole k-tiles, and the ring
//     is really D deep;
//   * the hand-over (wait, s_barrier) sits inside the stream of matrix instructions of the second-to-last of the
//     TN steps of a k-tile, the operands of the next k-tile are read under those of the last step, and the widening
//     is interleaved with them one vector instruction per matrix instruction: neither the barrier nor the LDS
//     latency is exposed even with one wavefront per SIMD;
//   * the block shape follows the problem (kTiles below): 20 shapes from 32 x 64 to 256 x 256.
// Measured against that earlier kernel (us, QKV / O / gate-up / down of a 4096-wide layer, weights from HBM; both with
// the stores straight from the accumulators that are described, with what replaced them, at the epilogue below):
//   M = 64    12288 <- 4096  20.7 -> 17.8   4096 <- 4096  12.9 -> 10.8   22016 <- 4096  31.6 -> 25.7   4096 <- 11008  22.1 -> 17.7
//   M = 406                  50.0 -> 54.2                 25.7 -> 24.7                  91.6 -> 80.8                  50.1 -> 50.9
//   M = 1024                103.3 -> 88.3                 37.9 -> 40.2                   156 -> 155                   91.8 -> 88.7
//   M = 2048                  163 -> 164                  69.1 -> 70.2                   293 -> 298                    174 -> 154
//   M = 8192                  631 -> 624                   217 -> 220                   1097 -> 1106                   544 -> 547
// Over 649 problems (26 matrices of decoders 1024 .. 8192 wide, 33 .. 8192 rows) the time is 0.92 of what it was in the
// geometric mean: 0.85 up to 200 rows, 0.91 up to 800, 0.96 to 0.97 beyond.  32 of them are more than 5 % slower, 13 % at
// most: matrices with 1024 or 2048 columns at 900 rows and more (2048 <- 2048 at 2048 rows 22.2 -> 24.4: its blocks fit
// the CUs once, and those of the earlier kernel shared a CU in twos), and launches a little over one round.
// 32x32x16 matrix instructions (operands free by addressing, the weights being in LDS) were 8-12 % slower, wavefront
// tiles of 128 x 128 with one wavefront per SIMD 20-30 %.
#include "gemm_common.h"
#include "tuning.h"

#include <type_traits>

using namespace eet;

namespace {

template <int TM, int TN, int WM, int WN, int D>
struct TileShape {
    static constexpr int kWaves = WM * WN;
    static constexpr int kBM = WM * TM * 16, kBN = WN * TN * 16;
    static constexpr int kAUnits = WM * TM * 2, kWUnits = WN * TN;      // 1 KiB copies per k-tile
    static constexpr int kAVec = kAUnits * 64, kWVec = kWUnits * 64;    // u32x4 per stage
    static constexpr int kA = (kAUnits + kWaves - 1) / kWaves, kW = (kWUnits + kWaves - 1) / kWaves;   // ... per wavefront
    static_assert(TM % 2 == 0, "a stage block holds a pair of m-tiles");
    static_assert(D >= 2 && D <= 5 && D * (kAVec + kWVec) * 16 <= 163840, "the stage ring must fit the LDS");
    static_assert((D - 1) * (kA + kW) <= 63, "the copies in flight must fit the wait counter");
};

// (a0 * b0 + c0, a1 * b1 + c1), each rounded once, to fp16.  Left to itself the compiler rounds some of a block's values by
// way of fp32.
__device__ __forceinline__ uint32_t fma_f16x2(float a0, float b0, float c0, float a1, float b1, float c1)
{
    uint32_t o;
    asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(o) : "v"(a0), "v"(b0), "v"(c0));
    asm("v_fma_mixhi_f16 %0, %1, %2, %3" : "+v"(o) : "v"(a1), "v"(b1), "v"(c1));
    return o;
}

template <int TM, int TN, int WM, int WN, int D, bool QKV>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2))) void w8a16_large_m_kernel(
    const _Float16 *__restrict__ A, const u32x4 *__restrict__ Wp, const _Float16 *__restrict__ scale,
    _Float16 *__restrict__ C, int M, int N, int K, int m_blocks, int n_blocks,
    const _Float16 *__restrict__ residual, int epi, int ksplit, float *__restrict__ partial, QkvOut out)
{
#if defined(__HIP_DEVICE_COMPILE__)  // buffer-resource builtins exist in the device pass only
    using S = TileShape<TM, TN, WM, WN, D>;
    __shared__ u32x4 lds[D][S::kAVec + S::kWVec];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: feeds scalar offsets and M0
    const int wm = wave / WN, wn = wave % WN;
    const int g = lane >> 4, j = lane & 15;
    const int ktiles = K >> 6, ntiles = N >> 4;
    // With ksplit > 1 (grid.y) the workgroup covers k-tiles [kbeg, kbeg + nk) only and
    // leaves its raw fp32 sums in partial[split][M][N] for the reduce kernel.
    const int split = blockIdx.y;
    const int kbeg = (int)((long)split * ktiles / ksplit);
    const int nk = (int)((long)(split + 1) * ktiles / ksplit) - kbeg;

    // Workgroups are numbered so that the ones resident on an XCD at one time (workgroup i lands on XCD i % 8)
    // cover a compact block of rows x columns and share both operands in its L2: bands of kBand column blocks
    // across all row blocks, the column block running fastest inside a band, a contiguous range of that order per
    // XCD (with one column block after the other, 64 row blocks shared one weight block and each fetched activation
    // rows of its own from the fabric: M = 8192, 4096 -> 12288 went from 1.18 to 1.28 PFLOP/s with the bands).
    const int total = m_blocks * n_blocks;
    const int per_xcd = (total + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= total)
        return;
    constexpr int kBand = 8;
    const int band = tile / (kBand * m_blocks), r = tile % (kBand * m_blocks);
    const int bw = min(kBand, n_blocks - band * kBand);   // column blocks of this band (the last one may be narrower)
    const int n_blk = band * kBand + r % bw, m_blk = r / bw;
    const int m0 = m_blk * S::kBM;
    const int ntb = n_blk * (WN * TN);
    // The n-tile of slot u of the block.  A block of fused Q | K | V channels is made of pairs of n-tiles half a head apart,
    // which the rotation turns into one another, whatever its width: slots 2 p and 2 p + 1 hold pair n_blk * kPairs + p.
    constexpr int kPairs = WN * TN / 2;
    const int hh = QKV ? out.dh >> 5 : 1;   // pairs in a head
    auto ntile = [&](int u) {
        if constexpr (!QKV)
            return ntb + u;
        const int pair = n_blk * kPairs + (u >> 1), head = pair / hh;
        return head * 2 * hh + (pair - head * hh) + (u & 1) * hh;
    };
    const int rows = min(M - m0, S::kBM);

    // Both operands are addressed through buffer resources: a 32-bit lane offset plus a scalar offset per tile.
    // Rows past M re-read row M - 1 and an n-tile past N / 16 the last one: their products are never stored, and no
    // copy is out of range (see above).  A wavefront whose share of a k-tile's copies is smaller repeats its last.
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16 *>(A + (size_t)m0 * K), 0, (unsigned)rows * (unsigned)K * 2u, 0x00020000);
    const __amdgpu_buffer_rsrc_t wrsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4 *>(Wp), 0, (unsigned)((size_t)K * N), 0x00020000);
    auto aunit = [&](int i) { return min(wave * S::kA + i, S::kAUnits - 1); };
    auto wunit = [&](int i) { return min(wave * S::kW + i, S::kWUnits - 1); };
    const int woff = lane * 16;
    unsigned wtile[S::kW];  // byte offset of the n-tile's first k-tile
#pragma unroll
    for (int i = 0; i < S::kW; ++i)
        wtile[i] = (unsigned)min(ntile(wunit(i)), ntiles - 1) * (unsigned)ktiles * 1024u;
    // Copy rg of the activations fills slots [64 rg, 64 rg + 64): block u = rg / 4, super-rows 4 (rg % 4) .. + 3.
    // Lane l writes slot s = l % 16 of super-row sj = 4 (rg % 4) + l / 16, which holds piece 2 pg + h of row sj of
    // m-tile 2u + e, where 4 (2e + h) + pg = s ^ sj.
    int aoff[S::kA];
#pragma unroll
    for (int i = 0; i < S::kA; ++i) {
        const int rg = aunit(i), u = rg >> 2, sj = 4 * (rg & 3) + (lane >> 4);
        const int p = (lane & 15) ^ sj, pg = p & 3, h = (p >> 2) & 1, e = p >> 3;
        aoff[i] = min((2 * u + e) * 16 + sj, rows - 1) * K * 2 + (2 * pg + h) * 16;
    }
    int rs[4];  // operand slot of this lane within a block, by 2e + h
#pragma unroll
    for (int c = 0; c < 4; ++c)
        rs[c] = wm * TM * 128 + j * 16 + ((4 * c + g) ^ j);
    const int wr0 = S::kAVec + wn * TN * 64 + lane;

    floatx4 acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int mt = 0; mt < TM; ++mt)
            acc[t][mt] = floatx4{0.f, 0.f, 0.f, 0.f};

    constexpr int L = S::kA + S::kW;   // copies of one k-tile per wavefront
    auto dma_tile = [&](int s, int kt) {
#pragma unroll
        for (int i = 0; i < S::kW; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrsrc, &lds[s][S::kAVec + wunit(i) * 64], 16, woff,
                                                     wtile[i] + (unsigned)(kbeg + kt) * 1024u, 0, 0);
#pragma unroll
        for (int i = 0; i < S::kA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, &lds[s][aunit(i) * 64], 16, aoff[i], (kbeg + kt) * 128, 0, 0);
    };
    auto read_op = [&](half8 (&op)[2], const u32x4 *cur, int mt) {
        op[0] = __builtin_bit_cast(half8, cur[(mt >> 1) * 256 + rs[2 * (mt & 1)]]);
        op[1] = __builtin_bit_cast(half8, cur[(mt >> 1) * 256 + rs[2 * (mt & 1) + 1]]);
    };

#pragma unroll
    for (int i = 0; i < D; ++i) {
        dma_tile(i, min(i, nk - 1));
        __builtin_amdgcn_sched_barrier(0);
    }
    half8 op[TM][2], w0, w1;   // operands of the current k-tile, weights of the current step
    u32x4 raw;                 // the packed weights of the step after
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D - 1) * L) : "memory");
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
        read_op(op[mt], lds[0], mt);
    {
        const u32x4 r0 = lds[0][wr0];
        if (TN > 1)
            raw = lds[0][wr0 + 64];
        w0 = widen8(r0.x, r0.y);
        w1 = widen8(r0.z, r0.w);
    }

    // One k-tile, in stage s of the ring: TN steps of one n-tile against all m-tiles.  kReq: k-tile `nx` is copied
    // into the stage once every wavefront has read it.
    constexpr int TB = TN >= 2 ? TN - 2 : 0;   // the step that starts with the hand-over
    auto tile_step = [&](auto s_c, auto req_c, int nx) {
        constexpr int s = decltype(s_c)::value, sn = (s + 1) % D;
        constexpr bool kReq = decltype(req_c)::value;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            half8 n0, n1;
            if (t == TB) {
                // All reads of this k-tile have been issued in earlier steps.  After the barrier they are complete for
                // every wavefront, and so is the copy of the next k-tile (younger: D - 2 k-tiles).
                // (A plain __syncthreads() would drain every outstanding copy here.)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kReq ? (D - 2) * L : 0) : "memory");
                if (kReq)
                    dma_tile(s, nx);
            }
            __builtin_amdgcn_sched_barrier(0);
            u32x4 raw2;
            if (TN >= 2) {
                raw2 = t + 2 < TN ? lds[s][wr0 + (t + 2) * 64] : lds[sn][wr0 + (t + 2 - TN) * 64];
                n0 = widen8(raw.x, raw.y);
                n1 = widen8(raw.z, raw.w);
            } else {
                raw2 = lds[sn][wr0];
                n0 = widen8(raw2.x, raw2.y);
                n1 = widen8(raw2.z, raw2.w);
            }
#pragma unroll
            for (int mt = 0; mt < TM; ++mt)
                acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, op[mt][0], acc[t][mt], 0, 0, 0);
#pragma unroll
            for (int mt = 0; mt < TM; ++mt) {
                acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, op[mt][1], acc[t][mt], 0, 0, 0);
                if (t == TN - 1)
                    read_op(op[mt], lds[sn], mt);
            }
            w0 = n0;
            w1 = n1;
            raw = raw2;
            // the order: a read of weights, then matrix and vector instructions in turn, in the last step with the
            // operand reads among them
            constexpr int kValu = 16 / (2 * TM) > 0 ? 16 / (2 * TM) : 1;
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int i = 0; i < 2 * TM; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (TN >= 2)
                    __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
                else if (i >= TM)   // one step per k-tile: its weights come behind the hand-over
                    __builtin_amdgcn_sched_group_barrier(0x002, 2 * kValu, 0);
                if (t == TN - 1 && i >= TM)
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kt = 0;
    for (; kt + D <= nk; kt += D) {
        // past the end the last k-tile is copied again: no branch, and the counts above stay exact
        auto next = [&](int s) { return min(kt + s + D, nk - 1); };
        tile_step(std::integral_constant<int, 0>{}, std::true_type{}, next(0));
        tile_step(std::integral_constant<int, 1>{}, std::true_type{}, next(1));
        if constexpr (D > 2)
            tile_step(std::integral_constant<int, 2 % D>{}, std::true_type{}, next(2));
        if constexpr (D > 3)
            tile_step(std::integral_constant<int, 3 % D>{}, std::true_type{}, next(3));
        if constexpr (D > 4)
            tile_step(std::integral_constant<int, 4 % D>{}, std::true_type{}, next(4));
    }
    // the up to D - 1 k-tiles that are left have been requested
    if (kt < nk)
        tile_step(std::integral_constant<int, 0>{}, std::false_type{}, 0);
    if constexpr (D > 2)
        if (kt + 1 < nk)
            tile_step(std::integral_constant<int, 1 % D>{}, std::false_type{}, 0);
    if constexpr (D > 3)
        if (kt + 2 < nk)
            tile_step(std::integral_constant<int, 2 % D>{}, std::false_type{}, 0);
    if constexpr (D > 4)
        if (kt + 3 < nk)
            tile_step(std::integral_constant<int, 3 % D>{}, std::false_type{}, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no copy may land in LDS after the workgroup has gone

    // acc[t][mt][r] of lane (g, j): row 16 * (wm * TM + mt) + j of the block, channel 4 * g + r of the n-tile of slot wn * TN + t
    if (!QKV && ksplit > 1) {
        const int mrow0 = m0 + wm * TM * 16 + j, nt0 = ntb + wn * TN;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            if (nt0 + t >= ntiles)
                continue;
#pragma unroll
            for (int mt = 0; mt < TM; ++mt) {
                const int m = mrow0 + 16 * mt;
                if (m < M)
                    *reinterpret_cast<floatx4 *>(partial + ((size_t)split * M + m) * N + (nt0 + t) * 16 + 4 * g) =
                        acc[t][mt];
            }
        }
        return;
    }
    // Stores.  The block goes through LDS as fp16 and leaves in 16-byte pieces of rows.  Straight from the accumulators it
    // left in 8 bytes a lane, 32 bytes of a row at a time, and the residual came in the same way (us, then / now: 2000 rows
    // 2048 <- 2048 with residual 25.2 / 21.8, 5120 <- 5120 93.9 / 88.3; 406 rows 4096 <- 4096 25.1 / 22.9; plain 12288 <- 4096 at
    // 406, 2048 and 8192 rows 50.2 / 47.7, 162 / 158, 617 / 604; SwiGLU, half the bytes, equal;
    // over 12 matrices 0.96 of the time from 400 rows on, 0.99 below).  A row's pieces are XORed with the row against
    // bank conflicts.
    constexpr int kPieces = S::kBN / 8, kThreads = 64 * S::kWaves;
    static_assert(S::kBM * kPieces <= D * (S::kAVec + S::kWVec), "the block must fit the stage ring");
    static_assert(kPieces % (TN % 2 == 0 ? 16 : 8) == 0, "the XOR stays in the row");
    u32x4 *tile_lds = &lds[0][0];
    auto piece_at = [&](int pieces, int row, int piece) { return row * pieces + (piece ^ (row & 7)); };
    // this lane's 4 channels of row 16 * (wm * TM + mt) + j, in the block's n-tile u
    auto stage = [&](int pieces, int mt, int u, half4 o) {
        const int at = piece_at(pieces, (wm * TM + mt) * 16 + j, 2 * u + (g >> 1));
        reinterpret_cast<u32x2 *>(tile_lds + at)[g & 1] = __builtin_bit_cast(u32x2, o);
    };
    half4 sc[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t)
        sc[t] = *reinterpret_cast<const half4 *>(scale + min(ntile(wn * TN + t), ntiles - 1) * 16 + 4 * g);
    __syncthreads();   // every wavefront has read its last operands, every copy has landed
    // pieces [0, n) of the block's rows: a thread takes n / kThreads of them, rows past M and columns past `cols` stay out
    const int cols = epi == kEpiSwiglu ? N / 2 : N, col0 = epi == kEpiSwiglu ? ntb * 8 : ntb * 16;
    auto leave = [&](auto pieces_c, auto &&piece) {
        constexpr int kRow = decltype(pieces_c)::value, kMine = S::kBM * kRow / kThreads;
        static_assert(S::kBM * kRow % kThreads == 0, "whole pieces");
#pragma unroll
        for (int i = 0; i < kMine; ++i) {
            const int task = tid + i * kThreads, row = task / kRow, col = col0 + task % kRow * 8;
            const half8 o = piece(i, __builtin_bit_cast(half8, tile_lds[piece_at(kRow, row, task % kRow)]));
            if (row < rows && col < cols)
                __builtin_memcpy(__builtin_assume_aligned(C + (size_t)(m0 + row) * cols + col, 8), &o, 16);
        }
    };
    if constexpr (!QKV && TN % 2 == 0) {
        if (epi == kEpiSwiglu) {
#pragma unroll
            for (int t = 0; t < TN; t += 2)
#pragma unroll
                for (int mt = 0; mt < TM; ++mt) {
                    // (the rounded quotient, as 32 rows and fewer have it; a product with v_rcp_f32's reciprocal, 2^-22 off,
                    // takes 77.4 us where this takes 81.0, 2000 rows, 11264 <- 2048)
                    half4 o;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float ga = acc[t][mt][r], ua = acc[t + 1][mt][r];
                        asm("" : "+v"(ga), "+v"(ua));   // (no product shared with the plain epilogue, which rounds it otherwise)
                        const float gate = (float)(_Float16)(ga * (float)sc[t][r]);
                        const float up = (float)(_Float16)(ua * (float)sc[t + 1][r]);
                        o[r] = (_Float16)(up * gate / (1.0f + __expf(-gate)));
                    }
                    stage(kPieces / 2, mt, (wn * TN + t) / 2, o);
                }
            __syncthreads();
            leave(std::integral_constant<int, kPieces / 2>{}, [](int, half8 o) { return o; });
            return;
        }
    }
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int mt = 0; mt < TM; ++mt) {
            half4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float f = acc[t][mt][r] * (float)sc[t][r];
                asm("" : "+v"(f));   // rounded to fp32 first in every block (the compiler merged a lone pair of the two steps)
                o[r] = (_Float16)f;
            }
            stage(kPieces, mt, wn * TN + t, o);
        }
    if constexpr (!QKV) {
        if (epi == kEpiResidual) {
            // all of the thread's residual pieces are on their way before the first store (loads wait for stores before them);
            // pieces outside read the nearest one inside
            half8 res[TM * TN / 2];
#pragma unroll
            for (int i = 0; i < TM * TN / 2; ++i) {
                const int task = tid + i * kThreads, row = task / kPieces, col = col0 + task % kPieces * 8;
                __builtin_memcpy(&res[i], __builtin_assume_aligned(residual + (size_t)(m0 + min(row, rows - 1)) * N +
                                                                       min(col, N - 8), 8), 16);
            }
            __syncthreads();
            leave(std::integral_constant<int, kPieces>{}, [&](int i, half8 o) { return o + res[i]; });
            return;
        }
    }
    __syncthreads();
    if constexpr (QKV) {
        // A lane takes 8 channels and their partners half a head on, turns them in fp32 and rounds again, to the bit as the
        // split kernel does.  (From the accumulators, with the angles of each lane's rows, this took 58 us instead of the
        // plain 51 for 2000 rows, 6144 <- 2048.)
        // piece q of a row: 8 channels of the first tile of pair q / 2
        constexpr int kTasks = S::kBM * kPairs * 2;
#pragma unroll 2
        for (int task = tid; task < kTasks; task += kThreads) {
            const int row = task / (kPairs * 2), q = task % (kPairs * 2), m = m0 + row;
            const int pair = n_blk * kPairs + (q >> 1), head = pair / hh, part = head / out.H, h = head - part * out.H;
            if (m >= M || part > 2)
                continue;
            const int b = m / out.S, pos = m - b * out.S, d = (pair - head * hh) * 16 + (q & 1) * 8, half = 16 * hh;
            half8 x = __builtin_bit_cast(half8, tile_lds[piece_at(kPieces, row, 4 * (q >> 1) + (q & 1))]);
            half8 y = __builtin_bit_cast(half8, tile_lds[piece_at(kPieces, row, 4 * (q >> 1) + 2 + (q & 1))]);
            if (out.rope != nullptr && part < 2) {
                const floatx4 *c = reinterpret_cast<const floatx4 *>(out.rope + (size_t)pos * out.dh + d);
                const floatx4 *sn = reinterpret_cast<const floatx4 *>(out.rope + (size_t)pos * out.dh + d + half);
                u32x4 px, py;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const floatx4 ce = c[e / 4], se = sn[e / 4];
                    const float a0 = (float)x[e], a1 = (float)x[e + 1], o0 = (float)y[e], o1 = (float)y[e + 1];
                    px[e / 2] = fma_f16x2(a0, ce[e % 4], -(o0 * se[e % 4]), a1, ce[e % 4 + 1], -(o1 * se[e % 4 + 1]));
                    py[e / 2] = fma_f16x2(o0, ce[e % 4], a0 * se[e % 4], o1, ce[e % 4 + 1], a1 * se[e % 4 + 1]);
                }
                x = __builtin_bit_cast(half8, px);
                y = __builtin_bit_cast(half8, py);
            }
            _Float16 *dst = (part == 0 ? out.q : part == 1 ? out.k : out.v) +
                            (((size_t)b * out.H + h) * (part == 0 ? out.S : out.T) + pos) * out.dh + d;
            *reinterpret_cast<half8 *>(dst) = x;
            *reinterpret_cast<half8 *>(dst + half) = y;
        }
    } else {
        leave(std::integral_constant<int, kPieces>{}, [](int, half8 o) { return o; });
    }
#endif
}

// Second pass of a split-k launch: sums the KS partial results of 4 adjacent channels of one row, applies the per-channel
// scale and the epilogue, rounds once (gate and up are rounded to fp16 before SwiGLU, as the single-pass kernel does).
// Bound by latency: everything a thread reads -- all shares, scales, residual -- is requested before the first use.  A
// loop over the shares waited for each before the next: 64 rows, 4096 <- 11008 in 14.9 us with it and 14.6 without, a
// step of four 4096-wide layers at 56 rows 630 and 619 us (with RMSnorm's gamma requested early as well).  KS = 0: any
// number of shares, `ksplit`, in such a loop (the tuning override may ask for one that the table never does).
template <int KS>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ partial,
                                                            const _Float16 *__restrict__ scale,
                                                            _Float16 *__restrict__ C,
                                                            const _Float16 *__restrict__ residual, int M, int N, int epi,
                                                            int ksplit)
{
    const int n_out = (epi == kEpiSwiglu) ? N / 2 : N;
    const int groups = n_out / 4;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= M * groups)
        return;
    const int m = idx / groups, o4 = (idx % groups) * 4;
    constexpr int kHeld = KS > 0 ? KS : 1;
    auto fetch4 = [&](floatx4 (&p)[kHeld], int n) {
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            p[k] = *reinterpret_cast<const floatx4 *>(partial + ((size_t)k * M + m) * N + n);
    };
    auto sum4 = [&](const floatx4 (&p)[kHeld], int n) {
        floatx4 s = p[0];
#pragma unroll
        for (int k = 1; k < kHeld; ++k)
            s += p[k];
        if constexpr (KS == 0)
            for (int k = 1; k < ksplit; ++k)
                s += *reinterpret_cast<const floatx4 *>(partial + ((size_t)k * M + m) * N + n);
        return s;
    };
    half4 o;
    if (epi == kEpiSwiglu) {
        const int ng = (o4 / 16) * 32 + o4 % 16, nu = ng + 16;  // gate tile 2u, up tile 2u+1
        floatx4 pg[kHeld], pu[kHeld];
        fetch4(pg, ng);
        fetch4(pu, nu);
        const half4 cg = *reinterpret_cast<const half4 *>(scale + ng), cu = *reinterpret_cast<const half4 *>(scale + nu);
        const floatx4 sg = sum4(pg, ng), su = sum4(pu, nu);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float gate = (float)(_Float16)(sg[r] * (float)cg[r]);
            const float up = (float)(_Float16)(su[r] * (float)cu[r]);
            o[r] = (_Float16)(up * gate / (1.0f + __expf(-gate)));
        }
    } else {
        floatx4 p[kHeld];
        fetch4(p, o4);
        const half4 sc = *reinterpret_cast<const half4 *>(scale + o4);
        half4 res = {0, 0, 0, 0};
        if (epi == kEpiResidual)
            res = *reinterpret_cast<const half4 *>(residual + (size_t)m * N + o4);
        const floatx4 sv = sum4(p, o4);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            o[r] = (_Float16)(sv[r] * (float)sc[r]);
        if (epi == kEpiResidual)
            o = o + res;
    }
    *reinterpret_cast<half4 *>(C + (size_t)m * n_out + o4) = o;
}

template <int TM, int TN, int WM, int WN, int D>
int launch_large_m(const GemmArgs &a, int ksplit)
{
    using S = TileShape<TM, TN, WM, WN, D>;
    const int m_blocks = (a.M + S::kBM - 1) / S::kBM, n_blocks = (a.N + S::kBN - 1) / S::kBN;
    const int grid = ((m_blocks * n_blocks + 7) / 8) * 8;
    float *partial = ksplit > 1 ? static_cast<float *>(a.ws) : nullptr;
    const auto kernel = a.epi == kEpiQkv ? w8a16_large_m_kernel<TM, TN, WM, WN, D, true> : w8a16_large_m_kernel<TM, TN, WM, WN, D, false>;
    hipLaunchKernelGGL(kernel, dim3(grid, ksplit), dim3(64 * S::kWaves), 0, a.st, a.A, a.Wp, a.scale, a.C, a.M, a.N, a.K,
                       m_blocks, n_blocks, a.residual, a.epi, ksplit, partial, a.qkv);
    EET_HIP_CHECK(hipGetLastError());
    if (ksplit > 1) {
        const int items = a.M * ((a.epi == kEpiSwiglu ? a.N / 2 : a.N) / 4);
        const auto reduce = ksplit == 2   ? splitk_reduce_kernel<2>
                            : ksplit == 3 ? splitk_reduce_kernel<3>
                            : ksplit == 4 ? splitk_reduce_kernel<4>
                            : ksplit == 6 ? splitk_reduce_kernel<6>
                            : ksplit == 8 ? splitk_reduce_kernel<8>
                                          : splitk_reduce_kernel<0>;
        hipLaunchKernelGGL(reduce, dim3((items + 255) / 256), dim3(256), 0, a.st, partial, a.scale, a.C, a.residual, a.M, a.N,
                           a.epi, ksplit);
        EET_HIP_CHECK(hipGetLastError());
    }
    return EET_OK;
}

// The block shapes and what they cost.  A launch with x workgroups per CU of the fullest XCD that walk nk k-tiles each
// takes about
//     base + (store [+ res]) * max(1, x) * (block area / 10^4) + nk * per_tile(x)   us
// where per_tile is linear between the values at 1/2, 1, just over 1, 2, just over 2, 3, just over 3, 4, 8, 24 and 64
// workgroups per CU (the jumps behind whole numbers are a CU that gets one workgroup more than the others).  The blocks
// go to the XCDs in eight equal ranges, so 84 blocks in three shares are 252 workgroups, but 33 on the 32 CUs of seven
// XCDs: counted over the whole chip such a launch looked 20 % cheaper than it is (406 rows, 3072 <- 8192: 43.8 us
// against 34.7 for what is taken now).  Fitted, shape by shape, to 14300 launches on MI355X: 20 weight matrices of
// decoders 1024 .. 5120 wide, 40 .. 8192 rows, one to eight shares of the k range; a fit is a fit: some of its
// constants (a store or residual of nothing, two workgroups cheaper than one and a bit) mean nothing by themselves.
// Fitted and checked with stores straight from the accumulators, before blocks left through LDS (649 problems outside the
// fit: those matrices at 25 row counts 33 .. 8192 and six matrices 1536 and 8192 wide: on average 1.5 % behind the fastest
// of the 20 shapes and their shares, at most 25 %, the same on the widths outside the fit).  With the epilogue as it is
// (229 problems, 17 matrices, 48 .. 8192 rows): 1.9 % and 16 %; other store terms gain 0.1 %.
struct TileCost {
    int tm, tn, wm, wn;
    float base, store, res, per_tile[11];
};
constexpr TileCost kTiles[] = {
    {2, 1, 1, 4, 2.917f, 1.247f, 0.000f, {0.161f, 0.166f, 0.191f, 0.247f, 0.315f, 0.335f, 0.426f, 0.477f, 0.892f, 2.520f, 6.530f}},
    {2, 2, 1, 4, 2.642f, 2.225f, 0.000f, {0.221f, 0.255f, 0.328f, 0.393f, 0.584f, 0.629f, 0.690f, 0.780f, 1.553f, 4.389f, 11.815f}},
    {4, 1, 1, 4, 2.166f, 2.141f, 0.568f, {0.200f, 0.222f, 0.275f, 0.364f, 0.518f, 0.565f, 0.615f, 0.716f, 1.379f, 3.961f, 11.391f}},
    {4, 2, 1, 4, 3.281f, 1.332f, 0.735f, {0.272f, 0.338f, 0.440f, 0.555f, 0.846f, 0.859f, 0.957f, 1.123f, 2.207f, 6.470f, 16.031f}},
    {4, 3, 1, 4, 5.194f, 0.355f, 1.088f, {0.352f, 0.405f, 0.589f, 0.747f, 0.994f, 1.149f, 1.234f, 1.570f, 3.029f, 9.078f, 22.839f}},
    {4, 4, 1, 4, 5.700f, 0.201f, 0.930f, {0.440f, 0.524f, 0.780f, 0.933f, 1.344f, 1.454f, 1.685f, 2.008f, 3.998f, 11.593f, 30.062f}},
    {6, 1, 1, 4, 2.159f, 1.850f, 1.611f, {0.232f, 0.279f, 0.358f, 0.469f, 0.652f, 0.723f, 0.782f, 0.959f, 1.841f, 5.355f, 14.470f}},
    {6, 2, 1, 4, 4.798f, 0.522f, 1.616f, {0.342f, 0.405f, 0.590f, 0.708f, 1.043f, 1.135f, 1.255f, 1.617f, 3.060f, 9.178f, 23.538f}},
    {6, 3, 1, 4, 6.617f, 0.000f, 1.187f, {0.470f, 0.543f, 0.787f, 0.988f, 1.367f, 1.546f, 1.623f, 2.113f, 4.265f, 12.731f, 26.329f}},
    {6, 4, 1, 4, 5.994f, 0.111f, 0.580f, {0.718f, 0.749f, 1.045f, 1.310f, 1.747f, 2.016f, 2.228f, 2.878f, 5.489f, 15.891f, 39.766f}},
    {8, 2, 1, 4, 5.896f, 0.166f, 1.236f, {0.442f, 0.494f, 0.746f, 0.904f, 1.319f, 1.455f, 1.657f, 1.987f, 3.930f, 11.468f, 29.993f}},
    {8, 3, 1, 4, 6.138f, 0.054f, 0.740f, {0.707f, 0.724f, 0.988f, 1.301f, 1.708f, 1.982f, 2.252f, 2.636f, 5.343f, 15.324f, 40.864f}},
    {8, 4, 1, 4, 6.961f, 0.008f, 1.063f, {0.786f, 0.835f, 1.333f, 1.620f, 2.470f, 2.513f, 2.955f, 3.415f, 6.896f, 19.815f, 51.087f}},
    {4, 2, 1, 8, 4.185f, 0.837f, 1.310f, {0.399f, 0.516f, 0.917f, 1.042f, 1.507f, 1.642f, 1.901f, 2.301f, 4.451f, 13.200f, 33.959f}},
    {4, 2, 2, 4, 5.578f, 0.425f, 1.405f, {0.373f, 0.494f, 0.871f, 1.017f, 1.499f, 1.627f, 1.852f, 2.296f, 4.527f, 13.521f, 35.022f}},
    {4, 5, 2, 4, 6.169f, 0.246f, 1.148f, {0.853f, 0.994f, 1.896f, 2.118f, 3.011f, 3.450f, 3.924f, 4.641f, 9.821f, 25.224f, 67.263f}},
    {6, 1, 1, 8, 4.801f, 0.530f, 1.081f, {0.320f, 0.406f, 0.623f, 0.745f, 1.022f, 1.192f, 1.353f, 1.654f, 3.212f, 9.524f, 24.507f}},
    {6, 2, 1, 8, 6.163f, 0.376f, 1.708f, {0.540f, 0.660f, 1.223f, 1.401f, 1.999f, 2.225f, 2.417f, 3.302f, 6.180f, 18.324f, 46.073f}},
    {8, 2, 1, 8, 6.156f, 0.302f, 1.639f, {0.662f, 0.806f, 1.571f, 1.734f, 2.698f, 2.744f, 3.195f, 3.889f, 7.725f, 22.208f, 51.472f}},
    {8, 4, 2, 4, 3.887f, 0.350f, 1.127f, {1.261f, 1.443f, 2.945f, 2.867f, 4.505f, 4.935f, 5.165f, 7.166f, 13.471f, 39.109f, 104.291f}}
};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

float per_tile_us(const TileCost &t, float x)
{
    constexpr float at[11] = {0.5f, 1.f, 1.001f, 2.f, 2.001f, 3.f, 3.001f, 4.f, 8.f, 24.f, 64.f};
    if (x <= at[0])
        return t.per_tile[0];
    for (int i = 1; i < 11; ++i)
        if (x <= at[i])
            return t.per_tile[i - 1] + (t.per_tile[i] - t.per_tile[i - 1]) * (x - at[i - 1]) / (at[i] - at[i - 1]);
    return t.per_tile[10] * x / at[10];
}

// a split launch pays a second kernel that reads what the first wrote
float split_reduce_us(int M, int N, int ks) { return 2.2f + (float)ks * M * N * 4.f / 3e6f; }

struct LargeMConfig {
    int tile = -1;    // index into kTiles
    int ksplit = 1;   // > 1: that many workgroups share a tile's k range (needs the fp32 workspace)
    float us = 1e30f;
};

// The best shape without a split and the best one with its k range split (us = 1e30: none is worth trying; a split is
// considered for launches of at most 200 blocks, i.e. where CUs would be idle, and leaves every share four k-tiles).
void pick_large_m(int M, int N, int K, int epi, LargeMConfig *whole, LargeMConfig *split)
{
    const int ktiles = K / 64;
    for (int i = 0; i < kNumTiles; ++i) {
        const TileCost &t = kTiles[i];
        if (epi == kEpiSwiglu && t.tn % 2 != 0)   // a wavefront holds whole (gate, up) pairs
            continue;
        const int bm = 16 * t.tm * t.wm, bn = 16 * t.tn * t.wn;
        const int blocks = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        const float area = (float)bm * bn * 1e-4f;
        auto cost = [&](int ks) {
            const float x = (blocks + 7) / 8 * ks / 32.f;   // the XCD with the most blocks decides
            const float store = ks > 1 ? 2.f * t.store : t.store + (epi == kEpiResidual ? t.res : 0.f);
            return t.base + store * (x > 1.f ? x : 1.f) * area + (float)ktiles / ks * per_tile_us(t, x);
        };
        if (const float us = cost(1); us < whole->us)
            *whole = LargeMConfig{i, 1, us};
        if (blocks <= 200)
            for (int ks : {2, 3, 4, 6, 8}) {
                if (ktiles / ks < 4 || blocks * ks > 560)
                    break;
                if (const float us = cost(ks) + split_reduce_us(M, N, ks); us < split->us)
                    *split = LargeMConfig{i, ks, us};
            }
    }
}

// 33 to 64 rows and no workspace for a split: with few channels the blocks leave most of the chip idle and each walks
// the whole k range alone, so its time is that of the k loop whatever M and N are.  The small-M kernel over 32-row
// slabs shares a block's k range among its wavefronts and has a block per few 16-channel tiles; its weights are read
// twice, from the Infinity Cache the second time, its second slab costs by its rows, and below 3072 k (2048 with SwiGLU)
// two short launches cost the host more than one.  Measured, us, slabs / blocks, at 33, 48 and 64 rows: 1024 <- 1024
// 6.2 / 5.4, 6.3 / 5.5, 6.1 / 5.5; 1024 <- 8192 14 / 23, 17 / 23, 21 / 23; 2048 <- 4096 10.1 / 13.0, 11.6 / 12.7,
// 13.4 / 12.7; 3072 <- 2048 9.0 / 8.2, 10.0 / 8.1, 9.7 / 8.1; 4096 <- 11008 24 / 31, 28 / 31, 32 / 31; 5120 <- 4096
// 13.7 / 13.6, 15.4 / 13.3, 16.6 / 13.8.  SwiGLU blocks hold whole (gate, up) pairs and are wider: 4096 <- 4096 13.0 /
// 17.4, 14.6 / 17.6, 16.3 / 17.7; 7168 <- 4096 15.6 / 17.7, 16.6 / 17.8, 18.4 / 18.5; 9216 <- 4096 22 / 18, 23 / 18, 25 / 19.
bool slabs_win(int M, int N, int K, int epi)
{
    if (M > 64 || K < 2048)
        return false;
    if (epi == kEpiSwiglu)
        return N <= 4096 || (N <= 8192 && M <= 48 && 8 * (long)K >= 3 * (long)N);
    return K >= 3072 && N <= 4096 && (M <= 48 || (N <= 2048 && K >= 6144));
}

// What the split of the fused Q | K | V rows costs as a kernel of its own: 5.0 us at 45 rows of 12288 channels, 6.5 at 406,
// 10.5 at 2000 rows of 6144, 69 at 8192 of 12288.
float qkv_split_us(int M, int N) { return 4.f + (float)M * N * 4.f / 6e6f; }

// What a call runs as (some block shape always does: the unsplit estimates are finite); tile < 0: 32-row slabs of the
// small-M kernel.
LargeMConfig plan_large_m(int M, int N, int K, int epi, size_t ws_bytes)
{
    // a split needs room for ksplit x M x N fp32; without it the best single-pass tile
    auto fits = [&](int ks) { return ks <= 1 || ws_bytes >= (size_t)ks * M * N * sizeof(float); };
    const eet::Tuning &tune = eet::tuning();
    LargeMConfig whole, split;
    pick_large_m(M, N, K, epi, &whole, &split);
    LargeMConfig c = split.us < whole.us && fits(split.ksplit) ? split : whole;
    if (tune.has_large_m) {   // "tm,tn[,ksplit[,wm,wn]]": runs when such a tile exists, else the table's choice stands
        for (int i = 0; i < kNumTiles; ++i) {
            const TileCost &t = kTiles[i];
            if (t.tm != tune.large_m_tm || t.tn != tune.large_m_tn || (epi == kEpiSwiglu && t.tn % 2 != 0) ||
                (tune.large_m_wm > 0 && (t.wm != tune.large_m_wm || t.wn != tune.large_m_wn)))
                continue;
            const int ks = tune.large_m_ksplit;
            return LargeMConfig{i, ks >= 1 && ks <= K / 64 && fits(ks) ? ks : 1, 0.f};
        }
    } else if (c.ksplit == 1 && slabs_win(M, N, K, epi)) {
        c = LargeMConfig{};
    }
    return c;
}

}  // namespace

// The workspace of a split that would win, or comes within 15 % of the unsplit launch (so that a caller who sizes its
// buffer once for a range of rows has the room where a split does win).
size_t eet::large_m_workspace(int M, int N, int K, int epi)
{
    LargeMConfig whole, split;
    pick_large_m(M, N, K, epi, &whole, &split);
    return split.us < 1.15f * whole.us ? (size_t)split.ksplit * M * N * sizeof(float) : 0;
}

extern "C" int eet_gemm_w8a16_large_m_shape(int M, int N, int K, int epilogue, size_t workspace_bytes, int *tm, int *tn,
                                            int *wm, int *wn, int *k_split)
{
    EET_REQUIRE(tm && tn && wm && wn && k_split, EET_ERR_INVALID_ARGUMENT, "eet_gemm_w8a16_large_m_shape: null pointer");
    EET_REQUIRE(M > 32 && N > 0 && K > 0 && K % 64 == 0 && N % 16 == 0 &&
                    (epilogue == kEpiNone || epilogue == kEpiResidual || (epilogue == kEpiSwiglu && N % 32 == 0)),
                EET_ERR_UNSUPPORTED_SHAPE,
                "eet_gemm_w8a16_large_m_shape: not a shape the large-M kernel takes (M=%d N=%d K=%d epilogue %d)", M, N, K,
                epilogue);
    const LargeMConfig c = plan_large_m(M, N, K, epilogue, workspace_bytes);
    const TileCost none{}, &t = c.tile < 0 ? none : kTiles[c.tile];
    *tm = t.tm, *tn = t.tn, *wm = t.wm, *wn = t.wn, *k_split = c.ksplit;
    return EET_OK;
}

int eet::run_large_m(const GemmArgs &a)
{
    // the kernel addresses A rows and the packed weights with 32-bit byte offsets
    if ((size_t)a.K * a.N >= (1ull << 31) || (size_t)a.K * 2 * 256 >= (1ull << 31))
        return eet::fail(EET_ERR_UNSUPPORTED_SHAPE, "eet_gemm_w8a16: K x N = %d x %d exceeds the 2 GiB weight limit",
                         a.K, a.N);
    const size_t ws_bytes = a.ws != nullptr && reinterpret_cast<uintptr_t>(a.ws) % 16 == 0 ? a.ws_bytes : 0;
    LargeMConfig c = plan_large_m(a.M, a.N, a.K, a.epi, ws_bytes);
    if (c.tile < 0)
        return a.epi == kEpiQkv ? kSplitApart : kTakesSlabs;
    if (a.epi == kEpiQkv && c.ksplit > 1) {
        // the epilogue takes whole sums: a split of the k range has to save more than the split kernel costs
        const LargeMConfig whole = plan_large_m(a.M, a.N, a.K, a.epi, 0);
        if (whole.tile < 0 || whole.ksplit > 1 || c.us + qkv_split_us(a.M, a.N) < whole.us)
            return kSplitApart;
        c = whole;
    }
    using Launcher = int (*)(const GemmArgs &, int);
    // in the order of kTiles; the last number is the depth of the stage ring, as deep as two workgroups of four
    // wavefronts (or one of eight) leave room for in the LDS
    constexpr Launcher launchers[] = {
        launch_large_m<2, 1, 1, 4, 5>,
        launch_large_m<2, 2, 1, 4, 5>,
        launch_large_m<4, 1, 1, 4, 5>,
        launch_large_m<4, 2, 1, 4, 5>,
        launch_large_m<4, 3, 1, 4, 4>,
        launch_large_m<4, 4, 1, 4, 3>,
        launch_large_m<6, 1, 1, 4, 4>,
        launch_large_m<6, 2, 1, 4, 4>,
        launch_large_m<6, 3, 1, 4, 3>,
        launch_large_m<6, 4, 1, 4, 2>,
        launch_large_m<8, 2, 1, 4, 3>,
        launch_large_m<8, 3, 1, 4, 2>,
        launch_large_m<8, 4, 1, 4, 2>,
        launch_large_m<4, 2, 1, 8, 4>,
        launch_large_m<4, 2, 2, 4, 4>,
        launch_large_m<4, 5, 2, 4, 4>,
        launch_large_m<6, 1, 1, 8, 4>,
        launch_large_m<6, 2, 1, 8, 4>,
        launch_large_m<8, 2, 1, 8, 4>,
        launch_large_m<8, 4, 2, 4, 3>
    };
    static_assert(sizeof(launchers) / sizeof(launchers[0]) == kNumTiles, "one launcher per block shape");
    return launchers[c.tile](a, c.ksplit);
}
