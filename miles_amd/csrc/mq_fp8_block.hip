// FP8 e4m3 block-scale quantizers and the block dequantizer for gfx950.
//
//   mode 0  "block_fp8"          scale = amax/448 (true division), q = e4m3(clamp(w/scale)); an all-zero
//                                tile has scale 0 and every byte 0xFF   (reference: tools/convert_hf_to_fp8.py:39-70)
//   mode 1  "fp8_blockwise_cast" absmax = max(amax,1e-10), x_s = absmax/448, q = e4m3(clamp(x * (1/x_s)))
//                                                                       (reference: miles/kernels/quant/fp8_blockwise.py:43-58)
//   mode 2  "per_block_cast_to_fp8" (power-of-two scales) absmax = max(amax,1e-4), sf = 2^ceil(log2(absmax/448)),
//                                q = e4m3(x * (1/sf)).  SGLang's function (third party, not in the reference tree; called at
//                                .../processors/quantizer_fp8.py:139-147); restated from its published source
//   dequant y = bf16(float(q) * s[i/B][j/B])                            (reference: tools/fp8_cast_bf16.py:15-40)
//
// Fast path (bf16 or fp16, 128x128 tiles, 16-byte aligned rows): one 512-lane workgroup (eight wavefronts) owns one tile.
// Lane t loads four 16-byte row segments (rows t/16 + 32 i, columns 8 (t%16) ..+8) so that sixteen lanes read one
// contiguous 256-byte tile row; the 32 values stay in registers, the tile amax is reduced with DPP inside each
// wavefront and through eight LDS words across the wavefronts, and the tile is quantized from registers:
// HBM traffic is one read of the input and one write of the codes and scale.
#include <mutex>

#include "mq_api_internal.hpp"
#include "mq_common.hpp"
#include "mq_group.hpp"

namespace mq {

constexpr int kTile = 128;
#ifndef MQ_TILE_THREADS
#define MQ_TILE_THREADS 512
#endif
constexpr int kTileThreads = MQ_TILE_THREADS;            // 8 wavefronts per 128x128 tile
constexpr int kRowsPerThread = 2048 / kTileThreads;     // 16-byte row segments per lane
constexpr int kRowStep = kTileThreads / 16;             // tile rows covered per pass of the workgroup
constexpr int kTileWaves = kTileThreads / kWave;

// 2^ceil(log2 v) for a normal positive v (the floor of 1e-4 / 448 keeps it normal): exponent, plus one when the
// mantissa is not zero.  For bf16 / fp16 inputs this is what pow(2, ceil(log2(v))) evaluates to in floating point
// as well: v is either an exact power of two or far from one.
__device__ __forceinline__ float ceil_pow2_scale(float v) {
    const uint32_t u = f2u(v);
    return u2f(((u >> 23) + ((u & 0x7FFFFFu) != 0)) << 23);
}

// Everything that is the same for the whole workgroup stays on the scalar unit (with the job lookup and the tile
// addressing in vector instructions the kernel issued 460 of them per wavefront; it issues about 200 now and the
// vector unit is busy a third of the time, the memory system being what bounds it): the job lookup, the tile's row and column (a
// multiply-high division with constants from the host), the 64-bit base addresses of the tile in the input and in the
// output.  A lane adds 32-bit offsets to those bases.  Interior tiles take a path with no bounds tests at all; edge
// tiles load from clamped (always valid) addresses and zero what lies outside, so that in both cases the four loads of
// a lane are issued back to back.
// which tensor and which of its tiles a workgroup works on: searched in the running counts of a kernel-argument table, or
// read off the two-dimensional grid of a device table (the workgroup then leaves if its tensor has fewer tiles)
struct TilePick {
    int32_t ji;         // index into tab.job
    int32_t tile;       // -1: nothing to do
};
__device__ __forceinline__ TilePick pick_tile(const TileTable& tab) {
    const int32_t item = xcd_contiguous_item(tab.total);
    if (item < 0) return TilePick{0, -1};
    const JobRef ref = find_job(tab, item);
    return TilePick{ref.ji, item - ref.start};
}
__device__ __forceinline__ TilePick pick_tile(const TileRef& tab) {
    const TileJob& job = tab.job[blockIdx.y];
    const int32_t tiles = ((job.M + kTile - 1) / kTile) * ((job.K + kTile - 1) / kTile);
    return TilePick{(int32_t)blockIdx.y, xcd_contiguous_item(tiles)};
}
// Tiles of a launch below which a lane issues its four loads at once.  Syncs, us, one then three / at once: 840 tiles 10.9 / 10.5,
// 2400 22.0 / 21.8, 2800 26.2 / 25.9, 4500 38.6 / 38.4, 7500 61.2 / 61.3, 18500 143.1 / 144.4.
constexpr uint32_t kShortLaunch = 4096;
template <int MODE, class Table, int F16>
__global__ __launch_bounds__(kTileThreads) void fp8_block128_kernel(const Table tab) {
    constexpr uint32_t kInfBits = F16 ? 0x7C00u : 0x7F80u;      // pattern of +inf; anything above is a NaN
    __shared__ uint32_t wave_amax[kTileWaves];
    const TilePick pick = pick_tile(tab);
    if (pick.tile < 0) return;
    const TileJob& job = tab.job[pick.ji];
    const uint32_t tile = (uint32_t)pick.tile;
    const uint32_t M = (uint32_t)job.M, K = (uint32_t)job.K, ldw = (uint32_t)job.ldw;
    const uint32_t tiles_k = (K + kTile - 1) / kTile;
    uint32_t ti = tile, tj = 0;
    if (tiles_k > 1) {
        ti = tile_div(tile, job.magic_k, job.shifts & 0xFFu);
        tj = tile - ti * tiles_k;
    }
    // row-blocked input: the tile's rows sit in block ti / tiles_per_block, at the same offset inside it
    const uint16_t* __restrict__ wt = (const uint16_t*)load_global_ptr(&job.w);
    uint32_t wti = ti;
    if (job.tiles_per_block > 0) {
        const uint32_t tpb = (uint32_t)job.tiles_per_block;
        const uint32_t blk = tpb > 1 ? tile_div(ti, job.magic_b, job.shifts >> 8) : ti;
        wt += (int64_t)blk * job.block_stride;
        wti = ti - blk * tpb;
    }
    wt += (int64_t)wti * kTile * ldw + (int64_t)tj * kTile;
    uint8_t* __restrict__ qt = (uint8_t*)load_global_ptr(&job.q) + (int64_t)ti * kTile * K + (int64_t)tj * kTile;
    float* __restrict__ tile_scales = load_global_ptr(&job.scale);
    const uint32_t rows_left = M - ti * kTile, cols_left = K - tj * kTile;     // both at least 1
    const bool full = rows_left >= (uint32_t)kTile && cols_left >= (uint32_t)kTile;

    const uint32_t t = threadIdx.x, r0 = t >> 4, c0 = (t & 15u) * 8u;
    const bool col_ok = full || c0 < cols_left;  // K % 8 == 0: an 8-wide segment is entirely inside or outside
    u32x4 v[kRowsPerThread];
    const bool short_launch = gridDim.x * gridDim.y < kShortLaunch;
    if (full) {
        const uint32_t off = (r0 * ldw + c0) * 2u;
#pragma unroll
        for (int i = 0; i < kRowsPerThread; i++) {
            v[i] = ld16((const char*)wt + (off + (uint32_t)i * (2u * kRowStep) * ldw));
            // The first quarter of the tile is waited for before the other three are requested.  With all four loads
            // of every lane in flight at once the sync ran 0.5 - 1.2 % slower (alternating runs on one GPU): the
            // memory queues are full either way, and the narrower front of requests keeps more of them on open pages.
            // A short launch has a memory latency less without the wait (kShortLaunch).
            if (i == 0 && kRowsPerThread > 2 && !short_launch) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    } else {
        const uint32_t c = col_ok ? c0 : 0u;
#pragma unroll
        for (int i = 0; i < kRowsPerThread; i++) {
            const uint32_t r = r0 + kRowStep * i;
            const uint32_t rr = r < rows_left ? r : rows_left - 1u;
            const u32x4 x = ld16((const char*)wt + (rr * ldw + c) * 2u);
            v[i] = (col_ok && r < rows_left) ? x : u32x4{0u, 0u, 0u, 0u};
        }
    }
    const uint32_t qoff = r0 * K + c0;
    auto row_ok = [&](int i) { return full || (col_ok && r0 + kRowStep * i < rows_left); };

    uint32_t m2 = 0;
#pragma unroll
    for (int i = 0; i < kRowsPerThread; i++) {
        m2 = max2_u16(m2, abs2(v[i].x));
        m2 = max2_u16(m2, abs2(v[i].y));
        m2 = max2_u16(m2, abs2(v[i].z));
        m2 = max2_u16(m2, abs2(v[i].w));
    }
    uint32_t m = wave_max(hmax_u16(m2));
    if ((t & (kWave - 1)) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    m = 0;
#pragma unroll
    for (int k = 0; k < kTileWaves; k++) m = umax(m, wave_amax[k]);
    if (MODE != 0 && m >= kInfBits) {
        // An infinity or a NaN in the tile (rare, and uniform over the workgroup).  Mode 1: Triton's max, maximum and
        // clamp return the operand that is not NaN, so the tile maximum skips NaN and a NaN product clamps to -448.
        // Mode 2: torch's amax hands a NaN on, 2^ceil(log2(.)) of inf / NaN is inf / NaN, and nothing clamps.
        float sx;
        if (MODE == 1) {
            uint32_t mf = 0;
#pragma unroll
            for (int i = 0; i < kRowsPerThread; i++) {
                const uint32_t u[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t lo = u[k] & 0x7FFFu, hi = (u[k] >> 16) & 0x7FFFu;
                    mf = umax(mf, umax(lo > kInfBits ? 0u : lo, hi > kInfBits ? 0u : hi));
                }
            }
            mf = wave_max(mf);
            __syncthreads();                    // every wavefront has read the first set of maxima
            if ((t & (kWave - 1)) == 0) wave_amax[t >> 6] = mf;
            __syncthreads();
            mf = 0;
#pragma unroll
            for (int k = 0; k < kTileWaves; k++) mf = umax(mf, wave_amax[k]);
            const float finite_max = elem_lo<F16>(mf);
            sx = (finite_max > 1e-10f ? finite_max : 1e-10f) / kFp8Max;
        } else {
            sx = u2f(m > kInfBits ? 0x7FC00000u : 0x7F800000u);
        }
        const float yx = 1.0f / sx;
        if (t == 0) tile_scales[tile] = sx;
#pragma unroll 1
        for (int i = 0; i < kRowsPerThread; i++) {
            const float f[8] = {elem_lo<F16>(v[i].x), elem_hi<F16>(v[i].x), elem_lo<F16>(v[i].y), elem_hi<F16>(v[i].y),
                                elem_lo<F16>(v[i].z), elem_hi<F16>(v[i].z), elem_lo<F16>(v[i].w), elem_hi<F16>(v[i].w)};
            uint32_t c[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float p = f[j] * yx;
                if (MODE == 1) p = __builtin_fminf(__builtin_fmaxf(p, -kFp8Max), kFp8Max);
                c[j] = sw_e4m3fn(p);
            }
            if (row_ok(i))
                st8(qt + (qoff + (uint32_t)i * kRowStep * K),
                    u32x2{c[0] | (c[1] << 8) | (c[2] << 16) | (c[3] << 24), c[4] | (c[5] << 8) | (c[6] << 16) | (c[7] << 24)});
        }
        return;
    }
    const float amax = elem_lo<F16>(m);

    float s;
    if (MODE == 0) s = amax / kFp8Max;
    else if (MODE == 1) s = (amax > 1e-10f ? amax : 1e-10f) / kFp8Max;
    else s = ceil_pow2_scale((amax > 1e-4f ? amax : 1e-4f) / kFp8Max);
    const float y = 1.0f / s;
    if (t == 0) tile_scales[tile] = s;

    if (MODE == 0 && !(amax > 0.0f) && amax == amax) {
        // all-zero tile: 0/0 on every element; the reference's CPU result is the negative NaN code
#pragma unroll
        for (int i = 0; i < kRowsPerThread; i++)
            if (row_ok(i)) st8(qt + (qoff + (uint32_t)i * kRowStep * K), u32x2{0xFFFFFFFFu, 0xFFFFFFFFu});
        return;
    }
    const bool fast_div = (MODE != 0) || shared_div_ok(s);

#pragma unroll
    for (int i = 0; i < kRowsPerThread; i++) {
        float f[8] = {elem_lo<F16>(v[i].x), elem_hi<F16>(v[i].x), elem_lo<F16>(v[i].y), elem_hi<F16>(v[i].y),
                      elem_lo<F16>(v[i].z), elem_hi<F16>(v[i].z), elem_lo<F16>(v[i].w), elem_hi<F16>(v[i].w)};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // |w/s| <= 448 (1 + 2^-22): no clamp is needed, the convert rounds anything up to 464 to 448
            if (MODE != 0) f[j] = f[j] * y;
            else f[j] = fast_div ? div_by_shared(f[j], s, y) : f[j] / s;
        }
        u32x2 o;
        o.x = hw_e4m3x4(f[0], f[1], f[2], f[3]);
        o.y = hw_e4m3x4(f[4], f[5], f[6], f[7]);
        if (row_ok(i)) st8(qt + (qoff + (uint32_t)i * kRowStep * K), o);
    }
}

// 128x128 tiles of a matrix with unit column stride and nothing else: any row stride, any column count, rows at any element
// boundary, fp32 as well as 16-bit.  The tile split is the fast kernel's (lane t: rows t/16 + 32 i, eight columns from
// 8 (t%16)); loads and stores are the same 16 and 8 bytes, only unaligned.  fp32: rows t/32 + 16 i, four columns from
// 4 (t%32), so that a load instruction takes whole lines there as well (eight columns from two loads, each of half of every
// line: two [4096, 8192] tensors 63.7 us, 55.0 this way; with non-temporal stores of the four bytes 57.5).  Past the
// matrix's edge nothing is masked: the last rows are read again, and a segment that would leave the row is moved back to end
// with it, so that the maximum sees only the tile's own elements (a tile at least a segment wide) and a byte that two lanes
// own is written twice with one value.  Bound by the memory system, which takes unaligned rows at 4.9 TB/s (24 [4097, 4099] bf16 tensors, 3.3 with
// non-temporal loads and 2.9 with non-temporal stores too) and aligned fp32 rows (LINES, non-temporal loads) at 6.1.  Twelve
// [1545, 2563] bf16 tensors as one list: 779 us in the two-pass kernel below, one launch each; 72 us here, host included.
// `aligned`: tensors that the fast kernel would take; a NaN's code and scale have that kernel's sign and payload.
template <int MODE, int DT, bool LINES>
__global__ __launch_bounds__(kTileThreads) void fp8_block128_any_kernel(const TileTable tab, const bool aligned) {
    constexpr uint32_t kInfBits = DT == MQ_F32 ? 0x7F800000u : DT == MQ_F16 ? 0x7C00u : 0x7F80u;
    constexpr uint32_t kSize = DT == MQ_F32 ? 4u : 2u;
    constexpr int kF16 = DT == MQ_F16;
    // a lane's segment is one 16-byte load: eight columns, or four fp32 ones
    constexpr uint32_t kCols = DT == MQ_F32 ? 4u : 8u, kRowLanes = kTile / kCols, kStep = kTileThreads / kRowLanes;
    constexpr int kRows = kTile / kStep;
    __shared__ uint32_t wave_amax[kTileWaves];
    const int32_t x = blockIdx.x % kXcds, k = blockIdx.x / kXcds, run = k >> tab.chunk_shift;
    const int32_t item = ((run * kXcds + x) << tab.chunk_shift) + (k - (run << tab.chunk_shift));
    if (item >= tab.total) return;
    const JobRef ref = find_job(tab, item);
    const TileJob& job = tab.job[ref.ji];
    const uint32_t tile = (uint32_t)(item - ref.start);
    const uint32_t M = (uint32_t)job.M, K = (uint32_t)job.K, ldw = (uint32_t)job.ldw;
    const uint32_t tiles_k = (K + kTile - 1) / kTile;
    uint32_t ti = tile, tj = 0;
    if (tiles_k > 1) {
        ti = tile_div(tile, job.magic_k, job.shifts & 0xFFu);
        tj = tile - ti * tiles_k;
    }
    const char* __restrict__ wt = (const char*)load_global_ptr(&job.w) + ((int64_t)ti * kTile * ldw + (int64_t)tj * kTile) * kSize;
    uint8_t* __restrict__ qt = (uint8_t*)load_global_ptr(&job.q) + (int64_t)ti * kTile * K + (int64_t)tj * kTile;
    float* __restrict__ tile_scales = load_global_ptr(&job.scale);
    const uint32_t rows_left = M - ti * kTile, cols_left = K - tj * kTile;     // both at least 1

    const uint32_t t = threadIdx.x, r0 = t / kRowLanes, c0 = (t % kRowLanes) * kCols;
    const bool narrow = cols_left < kCols;                                     // uniform over the workgroup
    const uint32_t c = narrow ? 0u : c0 + kCols <= cols_left ? c0 : cols_left - kCols;
    u32x4 v[kRows];
    if (!narrow) {
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            const uint32_t r = r0 + kStep * i, rr = r < rows_left ? r : rows_left - 1u;
            const char* at = wt + (rr * ldw + c) * kSize;
            v[i] = LINES ? ld16(at) : ld16_at2(at);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            const uint32_t r = r0 + kStep * i, rr = r < rows_left ? r : rows_left - 1u;
            uint32_t e[8];
#pragma unroll
            for (uint32_t j = 0; j < kCols; j++) {
                const char* at = wt + (rr * ldw + (j < cols_left ? j : cols_left - 1u)) * kSize;
                e[j] = DT == MQ_F32 ? *(const uint32_t*)at : *(const uint16_t*)at;
            }
            if (DT == MQ_F32) v[i] = u32x4{e[0], e[1], e[2], e[3]};
            else v[i] = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
        }
    }
    // the kCols elements of row segment i
    auto element = [&](int i, int j) -> float {
        if (DT == MQ_F32) return u2f(v[i][j & 3]);
        const uint32_t pair = v[i][(j >> 1) & 3];
        return (j & 1) ? elem_hi<kF16>(pair) : elem_lo<kF16>(pair);
    };
    auto workgroup_max = [&](uint32_t m) {
        m = wave_max(m);
        if ((t & (kWave - 1)) == 0) wave_amax[t >> 6] = m;
        __syncthreads();
        m = 0;
#pragma unroll
        for (int k = 0; k < kTileWaves; k++) m = umax(m, wave_amax[k]);
        return m;
    };
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < kRows; i++) {
        u32x4 x = v[i];
        // (a copy: the magnitudes of all 32 elements would otherwise be kept for MODE 1's second look at them, 82 registers
        // instead of 50 and two workgroups per compute unit instead of four: 24 [200000, 32] tensors 272 us instead of 169)
        if (MODE == 1 && DT == MQ_F32) asm("" : "+v"(x));
        if (DT == MQ_F32)
            m = umax(umax(umax(m, x.x & 0x7FFFFFFFu), umax(x.y & 0x7FFFFFFFu, x.z & 0x7FFFFFFFu)), x.w & 0x7FFFFFFFu);
        else
            m = max2_u16(max2_u16(m, max2_u16(abs2(x.x), abs2(x.y))), max2_u16(abs2(x.z), abs2(x.w)));
    }
    m = workgroup_max(DT == MQ_F32 ? m : hmax_u16(m));
    const bool special = m >= kInfBits;      // an infinity or a NaN in the tile, as in the fast kernel
    if (MODE == 1 && special) {
        uint32_t finite = 0;
#pragma unroll
        for (int i = 0; i < kRows; i++)
#pragma unroll
            for (uint32_t j = 0; j < kCols; j++) {
                const uint32_t a = f2u(element(i, j)) & 0x7FFFFFFFu;
                finite = umax(finite, a > 0x7F800000u ? 0u : a);
            }
        __syncthreads();                     // every wavefront has read the first set of maxima
        m = workgroup_max(finite);
    }
    const float amax = DT == MQ_F32 || (MODE == 1 && special) ? u2f(m) : elem_lo<kF16>(m);
    float s;
    if (MODE == 0) s = amax / kFp8Max;
    else if (MODE == 1) s = (amax > 1e-10f ? amax : 1e-10f) / kFp8Max;
    else s = special ? (aligned && m > kInfBits ? u2f(0x7FC00000u) : amax) : ceil_pow2_scale((amax > 1e-4f ? amax : 1e-4f) / kFp8Max);
    const float y = 1.0f / s;
    if (t == 0) tile_scales[tile] = s;
    const bool zero_tile = MODE == 0 && !(amax > 0.0f) && amax == amax;       // 0 / 0: the negative NaN code
    // software arithmetic where the hardware conversion or the shared-divisor sequence do not hold: infinities, NaN,
    // scales at the ends of the fp32 range
    const bool plain = !special && (MODE != 0 || shared_div_ok(s));
#pragma unroll
    for (int i = 0; i < kRows; i++) {
        uint32_t o[kCols / 4];
        if (zero_tile) {
#pragma unroll
            for (uint32_t j = 0; j < kCols; j += 4) o[j / 4] = 0xFFFFFFFFu;
        } else if (plain) {
            float f[kCols];
#pragma unroll
            for (uint32_t j = 0; j < kCols; j++) {
                const float x = element(i, j);
                f[j] = MODE != 0 ? x * y : DT == MQ_F32 ? div24_by_shared(x, s, y) : div_by_shared(x, s, y);
            }
#pragma unroll
            for (uint32_t j = 0; j < kCols; j += 4)       // at most 448 (1 + 2^-22): rounds to 448 by itself
                o[j / 4] = hw_e4m3x4(f[j], f[j + 1], f[j + 2], f[j + 3]);
        } else if (MODE == 0 && DT != MQ_F32 && aligned) {
#pragma unroll
            for (uint32_t j = 0; j < kCols; j += 4)
                o[j / 4] = hw_e4m3x4(element(i, j) / s, element(i, j + 1) / s, element(i, j + 2) / s, element(i, j + 3) / s);
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kCols; j++) {
                const float x = element(i, j);
                float p = MODE != 0 ? x * y : x / s;
                if (MODE == 0) p = clamp_keep_nan(p, -kFp8Max, kFp8Max);                            // torch.clamp
                else if (MODE == 1) p = __builtin_fminf(__builtin_fmaxf(p, -kFp8Max), kFp8Max);     // tl.clamp: NaN -> -448
                const uint32_t code = sw_e4m3fn(p) << (8 * (j & 3));
                o[j / 4] = (j & 3) == 0 ? code : o[j / 4] | code;
            }
        }
        const uint32_t r = r0 + kStep * i;
        if (r >= rows_left || c0 >= cols_left) continue;
        uint8_t* at = qt + (r * K + c);
        if (!narrow) {
            if (kCols == 8) st8_at1(at, u32x2{o[0], o[kCols / 4 - 1]});
            else st4_at1(at, o[0]);
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kCols - 1; j++)
                if (j < cols_left) at[j] = (uint8_t)(o[j / 4] >> (8 * (j & 3)));
        }
    }
}

constexpr int kGenThreads = 256;
// Any dtype, any strides, any block size: one workgroup per tile, two passes over the tile (the second
// one is served by the caches).  Correctness path for what the tile kernels do not take: other block sizes, column
// strides, rows of 2^24 elements and more.
template <int MODE>
__global__ __launch_bounds__(kGenThreads) void fp8_block_generic_kernel(const void* __restrict__ w, int dtype,
                                                                         int64_t sxm, int64_t sxn,
                                                                         uint8_t* __restrict__ q, int64_t ldq,
                                                                         float* __restrict__ scale, int64_t M,
                                                                         int64_t K, int bm, int bk, int tiles_k) {
    __shared__ uint32_t wave_amax[kGenThreads / kWave];
    const int t = threadIdx.x;
    const int64_t tile = blockIdx.x;
    const int64_t ti = tile / tiles_k, tj = tile - ti * tiles_k;
    const int64_t r0 = ti * bm, c0 = tj * bk;
    const int n = bm * bk;
    uint32_t m = 0;
    for (int idx = t; idx < n; idx += kGenThreads) {
        const int64_t r = r0 + idx / bk, c = c0 + idx % bk;
        if (r < M && c < K) {
            const uint32_t a = f2u(load_f32(w, r * sxm + c * sxn, dtype)) & 0x7FFFFFFFu;
            m = umax(m, (MODE == 1 && a > 0x7F800000u) ? 0u : a);      // Triton's max skips NaN, torch's amax hands it on
        }
    }
    m = wave_max(m);
    if ((t & (kWave - 1)) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    m = umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3]));
    const float amax = u2f(m);
    float s, y;
    if (MODE == 0) {
        s = amax / kFp8Max;
        y = 0.0f;
    } else if (MODE == 1) {
        const float absmax = amax > 1e-10f ? amax : 1e-10f;
        s = absmax / kFp8Max;
        y = 1.0f / s;
    } else {
        s = m >= 0x7F800000u ? amax : ceil_pow2_scale((amax > 1e-4f ? amax : 1e-4f) / kFp8Max);   // inf / NaN stay
        y = 1.0f / s;
    }
    if (t == 0) scale[tile] = s;
    const bool zero_tile = MODE == 0 && !(amax > 0.0f) && amax == amax;
    for (int idx = t; idx < n; idx += kGenThreads) {
        const int64_t r = r0 + idx / bk, c = c0 + idx % bk;
        if (r < M && c < K) {
            uint32_t code;
            if (zero_tile) code = 0xFFu;
            else {
                const float x = load_f32(w, r * sxm + c * sxn, dtype);
                float v = MODE != 0 ? x * y : x / s;
                if (MODE == 0) v = clamp_keep_nan(v, -kFp8Max, kFp8Max);                              // torch.clamp
                else if (MODE == 1) v = __builtin_fminf(__builtin_fmaxf(v, -kFp8Max), kFp8Max);        // tl.clamp: NaN -> -448
                code = sw_e4m3fn(v);
            }
            q[r * ldq + c] = (uint8_t)code;
        }
    }
}

// ---- per-tensor / per-channel (reference: tools/convert_hf_to_fp8.py:73-86,
//      quantizer_fp8.py:153-158) ---------------------------------------------------------------
// pass 1: amax per row (per_channel) or per tensor (atomic max on the float bit pattern)
__global__ __launch_bounds__(256) void fp8_row_amax_kernel(const void* __restrict__ w, int dtype, int64_t ldw,
                                                           int64_t K, uint32_t* __restrict__ amax_bits,
                                                           int per_channel) {
    __shared__ uint32_t wave_amax[4];
    const int t = threadIdx.x;
    const int64_t r = blockIdx.x;
    uint32_t m = 0;
    for (int64_t c = t; c < K; c += 256) m = umax(m, f2u(load_f32(w, r * ldw + c, dtype)) & 0x7FFFFFFFu);
    m = wave_max(m);
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    if (t == 0) {
        m = umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3]));
        if (per_channel) amax_bits[r] = m;
        else atomicMax(amax_bits, m);
    }
}
// pass 2: scale = max(amax, floor)/448 ; q = e4m3(clamp(w/scale)).  With one scale for the whole
// tensor the quotient is first rounded to the weight's dtype (torch keeps `weight / zero_dim_scale`
// in the weight's dtype).
__global__ __launch_bounds__(256) void fp8_row_quant_kernel(const void* __restrict__ w, int dtype, int64_t ldw,
                                                            int64_t K, const uint32_t* __restrict__ amax_bits,
                                                            float floor_v, int per_channel,
                                                            uint8_t* __restrict__ q, float* __restrict__ scale) {
    const int t = threadIdx.x;
    const int64_t r = blockIdx.x;
    float amax = u2f(per_channel ? amax_bits[r] : amax_bits[0]);
    if (amax < floor_v) amax = floor_v;
    const float s = amax / kFp8Max;
    if (t == 0 && (per_channel || r == 0)) scale[per_channel ? r : 0] = s;
    for (int64_t c = t; c < K; c += 256) {
        float v = load_f32(w, r * ldw + c, dtype) / s;
        if (!per_channel) v = round_to_dtype(v, dtype);
        v = clamp_keep_nan(v, -kFp8Max, kFp8Max);
        q[r * K + c] = (uint8_t)sw_e4m3fn(v);
    }
}
// ---- rows, and whole tensors, of 16-byte units -------------------------------------------------------------------
// What the two passes above do, from 16-byte loads (E elements: eight of a 16-bit dtype, four of fp32), for up to 64 tensors
// a launch.  LINES: aligned units, streamed with non-temporal accesses.  Otherwise any element boundary: the
// last unit of a row, or of the tensor, is moved back to end with it, so that it codes a few elements a second time, to the
// same bytes.  HBM-bound.  The quotient x / s is the exact one (shared-divisor sequence, which keeps the sign of a -0
// numerator; the division itself when s leaves the guarded range); fp32 quotients come correctly rounded from
// div24_by_shared where that matters to an e4m3 code.
// Four tensors in one list against a launch (per channel) or three (per tensor) each, us of the kernels: per channel [4096,
// 8192] bf16 72 -> 61 (6.6 TB/s), fp32 129 -> 108 (6.2), [4095, 8191] bf16 90 -> 74, [1024, 2048] bf16 16.8 -> 6.0; per tensor
// [4096, 8192] fp32 218 -> 179, [4095, 8191] bf16 138 -> 104, [1024, 2048] fp32 39 -> 16.
template <int DT> constexpr int kUnitElems = DT == MQ_F32 ? 4 : 8;
template <int DT, bool LINES, bool KEEP = false>
__device__ __forceinline__ u32x4 ld_unit(const void* p, int64_t elem) {
    const char* at = (const char*)p + elem * (DT == MQ_F32 ? 4 : 2);
    return !LINES ? ld16_at2(at) : KEEP ? ld16_keep(at) : ld16(at);
}
// the largest magnitude of a unit: an fp32 pattern, or packed 16-bit patterns
template <int DT>
__device__ __forceinline__ uint32_t unit_max(uint32_t m, const u32x4 v) {
    if (DT == MQ_F32)
        return umax(m, umax(umax(v.x & 0x7FFFFFFFu, v.y & 0x7FFFFFFFu), umax(v.z & 0x7FFFFFFFu, v.w & 0x7FFFFFFFu)));
    return max2_u16(m, max2_u16(max2_u16(abs2(v.x), abs2(v.y)), max2_u16(abs2(v.z), abs2(v.w))));
}
// what a lane collected with unit_max, as an fp32 pattern
template <int DT>
__device__ __forceinline__ uint32_t unit_max_f32(uint32_t m) {
    return DT == MQ_F32 ? m : f2u(DT == MQ_F16 ? elem_lo<1>(hmax_u16(m)) : elem_lo<0>(hmax_u16(m)));
}
// codes of one unit; ROUNDED: the quotient is rounded to the dtype first (one scale for the whole tensor).  `plain`: the
// scale is in the range of the division sequence (shared_div_ok), so no element is infinite or NaN and no quotient exceeds
// 448 by more than its rounding.  A zero, subnormal (a quotient by its few bits may be far above 448), huge or non-finite
// scale takes divisions, the clamp and the software conversion.
template <int DT, bool ROUNDED, bool LINES>
__device__ __forceinline__ void scaled_unit(const u32x4 v, float s, float y, bool plain, uint8_t* __restrict__ q) {
    constexpr int E = kUnitElems<DT>;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float f[E];
#pragma unroll
    for (int j = 0; j < E; j++) {
        if (DT == MQ_F32) f[j] = u2f(w[j]);
        else if (DT == MQ_F16) f[j] = (j & 1) ? elem_hi<1>(w[j / 2]) : elem_lo<1>(w[j / 2]);
        else f[j] = (j & 1) ? elem_hi<0>(w[j / 2]) : elem_lo<0>(w[j / 2]);
    }
#pragma unroll
    for (int j = 0; j < E; j++)
        f[j] = !plain ? f[j] / s : DT == MQ_F32 ? div24_by_shared(f[j], s, y) : div_by_shared(f[j], s, y);
    if (ROUNDED && DT != MQ_F32) {
#pragma unroll
        for (int j = 0; j < E; j += 2) {
            if (DT == MQ_BF16 && plain) {
                const uint32_t p = hw_bf16x2(f[j], f[j + 1]);
                f[j] = bf16_lo(p);
                f[j + 1] = bf16_hi(p);
            } else {
                f[j] = round_to_dtype(f[j], DT);
                f[j + 1] = round_to_dtype(f[j + 1], DT);
            }
        }
    }
    u32x2 o = {0u, 0u};
    if (plain) {
        o.x = hw_e4m3x4(f[0], f[1], f[2], f[3]);
        if (E == 8) o.y = hw_e4m3x4(f[E - 4], f[E - 3], f[E - 2], f[E - 1]);
    } else {
#pragma unroll
        for (int j = 0; j < E; j++) {
            const uint32_t c = sw_e4m3fn(clamp_keep_nan(f[j], -kFp8Max, kFp8Max)) << (8 * (j & 3));
            if (j < 4) o.x |= c;
            else o.y |= c;
        }
    }
    if (LINES && E == 8) st8(q, u32x2{o.x, o.y});
    else if (LINES) st4(q, o.x);
    else if (E == 8) st8_at1(q, u32x2{o.x, o.y});
    else st4_at1(q, o.x);
}
struct ChannelJob {
    const void* w;
    uint8_t* q;
    float* scale;
    int64_t ldw;
    int32_t K, M;
    float floor_v;
    int32_t pad;
};
struct ChannelTable {
    int32_t n, chunk, max_blocks, pad;      // grid: max_blocks workgroups (a multiple of 8 * chunk) x n tensors
    ChannelJob job[kMaxGroup];
};
// per channel: a row lives in the registers of ROWLANES lanes (up to UNITS units each), so it is read once: amax across the
// lanes, one scale, codes.  ROWLANES = 64: four rows per workgroup, no LDS; 256: one row.  An XCD takes runs of consecutive
// rows, as the flat kernels take runs of consecutive blocks.
template <int ROWLANES, int DT, int UNITS, bool LINES>
__global__ __launch_bounds__(256) void fp8_channel_kernel(const ChannelTable tab) {
    __shared__ uint32_t wave_amax[4];
    constexpr int kRows = 256 / ROWLANES, E = kUnitElems<DT>;
    const ChannelJob& job = tab.job[blockIdx.y];
    const void* __restrict__ w = load_global_ptr(&job.w);
    uint8_t* __restrict__ q = load_global_ptr(&job.q);
    const int t = threadIdx.x, lane = t % ROWLANES, K = job.K;
    const int64_t block = xcd_chunked_block(tab.chunk), row = block * kRows + t / ROWLANES;
    if (block * kRows >= job.M) return;
    const bool row_ok = row < job.M;
    const int64_t src = (row_ok ? row : job.M - 1) * job.ldw;
    const int units = (K + E - 1) / E, last = K - E;
    u32x4 v[UNITS];
    uint32_t m = 0;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const int unit = lane + u * ROWLANES, at = unit * E < last ? unit * E : last;      // (lanes past the end read the last unit)
        v[u] = u * ROWLANES < units ? ld_unit<DT, LINES>(w, src + at) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < UNITS; u++) m = unit_max<DT>(m, v[u]);
    m = wave_max(unit_max_f32<DT>(m));
    if (ROWLANES == 256) {
        if ((t & 63) == 0) wave_amax[t >> 6] = m;
        __syncthreads();
        m = umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3]));
    }
    float amax = u2f(m);
    if (amax < job.floor_v) amax = job.floor_v;
    const float s = amax / kFp8Max, y = 1.0f / s;
    const bool plain = shared_div_ok(s);
    if (!row_ok) return;
    if (lane == 0) load_global_ptr(&job.scale)[row] = s;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const int unit = lane + u * ROWLANES, at = unit * E < last ? unit * E : last;
        if (unit < units) scaled_unit<DT, false, LINES>(v[u], s, y, plain, q + row * K + at);
    }
}
struct ScaledJob {
    const void* w;
    uint8_t* q;
    float* scale;
    uint32_t* maxima;       // of the amax pass, ScaledTable::words of them
    int64_t n;              // elements
    float floor_v;
    int32_t pad;
};
struct ScaledTable {
    int32_t n, chunk, max_blocks;
    int32_t words;          // partial maxima of a tensor: a power of two, at most kScaledWords
    int32_t amax_blocks;    // workgroups of the amax pass for each tensor
    int32_t pad;
    ScaledJob job[kMaxGroup];
};
// per tensor: an amax pass over n contiguous elements, and a flat quantize pass that folds the partial maxima by itself, under
// its loads.  The maxima are read by every workgroup of the second pass, so they are few: a workgroup of the amax pass is 1024
// lanes, 64 of them cover a tensor where eight share a launch, and a wavefront folds 64 words with one load.  (256 words, read
// by each wavefront: four [4096, 8192] fp32 111 us in the second pass instead of 101.)  As jobs a workgroup of the amax
// pass has a word of its own; the direct calls have fewer words than workgroups, cleared beforehand, and take the maximum
// atomically, at some 8 ns each.
constexpr int kScaledLoads = 4, kScaledUnits = 4, kScaledShortUnits = 2, kAmaxThreads = 1024, kScaledWords = 256, kDirectWords = 64, kDirectBlocks = 256;
// KEEP of the four loads of a trip are left in the memory-side cache for the quantize pass (kept_quarters; unaligned loads
// carry no hint and stay there anyway).
// A lane of the quantize pass takes four units, which is what gains by that cache (two: four [4096, 8192] bf16 62.5 us against
// 56.4, without the cache 63.5 and 63.9); of a list under 8 MiB, two, which leaves it twice the workgroups (two [512, 1024]
// 3.5 us, 4.4 with four).  Both passes together, us, before and after: four [4096, 8192] bf16 105 -> 100, fp32 179 -> 171,
// two [4095, 8191] 55.4 -> 53.2, eight [2198, 1333] 25.6 -> 22.9.
constexpr int64_t kScaledLongList = (8ll << 20) / 16;       // units of a list
template <int DT, bool LINES, int KEEP>
__global__ __launch_bounds__(kAmaxThreads) void fp8_scaled_amax_kernel(const ScaledTable tab) {
    __shared__ uint32_t wave_amax[kAmaxThreads / kWave];
    constexpr int E = kUnitElems<DT>;
    const ScaledJob& job = tab.job[blockIdx.y];
    const void* __restrict__ w = load_global_ptr(&job.w);
    const int t = threadIdx.x;
    const int64_t n = job.n, units = (n + E - 1) / E, last = LINES ? n / E * E - E : n - E;      // of the units that lanes past the end read again
    uint32_t m = 0;
    for (int64_t base = (int64_t)blockIdx.x * (kAmaxThreads * kScaledLoads); base < units; base += (int64_t)gridDim.x * (kAmaxThreads * kScaledLoads)) {
        u32x4 v[kScaledLoads];
        // (a loop for each kind: loads that one loop chooses between lose the hint)
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            const int64_t at = (base + i * kAmaxThreads + t) * E;
            v[i] = ld_unit<DT, LINES, true>(w, at < last ? at : last);
        }
#pragma unroll
        for (int i = KEEP; i < kScaledLoads; i++) {
            const int64_t at = (base + i * kAmaxThreads + t) * E;
            v[i] = ld_unit<DT, LINES>(w, at < last ? at : last);
        }
#pragma unroll
        for (int i = 0; i < kScaledLoads; i++) m = unit_max<DT>(m, v[i]);
    }
    if (LINES && last + E < n && blockIdx.x == 0 && t == 0) m = unit_max<DT>(m, ld_unit<DT, false>(w, n - E));
    m = wave_max(unit_max_f32<DT>(m));
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    if (t != 0) return;
    m = 0;
#pragma unroll
    for (int k = 0; k < kAmaxThreads / kWave; k++) m = umax(m, wave_amax[k]);
    uint32_t* __restrict__ word = load_global_ptr(&job.maxima) + (blockIdx.x & (uint32_t)(tab.words - 1));
    if (tab.amax_blocks > tab.words) atomicMax(word, m);
    else *word = m;
}
template <int DT, bool LINES, int UNITS>
__global__ __launch_bounds__(256) void fp8_scaled_quant_kernel(const ScaledTable tab) {
    __shared__ uint32_t wave_amax[4];
    constexpr int E = kUnitElems<DT>;
    const ScaledJob& job = tab.job[blockIdx.y];
    const void* __restrict__ w = load_global_ptr(&job.w);
    const uint32_t* __restrict__ maxima = load_global_ptr(&job.maxima);
    uint8_t* __restrict__ q = load_global_ptr(&job.q);
    const int64_t n = job.n, first = xcd_chunked_block(tab.chunk) * (256 * UNITS), base = first + threadIdx.x;
    if (first * E >= n) return;
    const int64_t last = LINES ? n / E * E - E : n - E;
    u32x4 v[UNITS];
#pragma unroll
    for (int i = 0; i < UNITS; i++) {
        const int64_t at = (base + i * 256) * E;
        v[i] = ld_unit<DT, LINES>(w, at < last ? at : last);
    }
    static_assert(kScaledWords <= 256, "a word per lane");
    uint32_t m = wave_max(maxima[threadIdx.x & (uint32_t)(tab.words - 1)]);
    if (tab.words > kWave) {
        if ((threadIdx.x & 63) == 0) wave_amax[threadIdx.x >> 6] = m;
        __syncthreads();
        m = umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3]));
    }
    float amax = u2f(m);
    if (amax < job.floor_v) amax = job.floor_v;
    const float s = amax / kFp8Max, y = 1.0f / s;
    const bool plain = shared_div_ok(s);
    if (base == 0) *load_global_ptr(&job.scale) = s;
#pragma unroll
    for (int i = 0; i < UNITS; i++) {
        const int64_t at = (base + i * 256) * E;
        if (!LINES && at < n) scaled_unit<DT, true, false>(v[i], s, y, plain, q + (at < last ? at : last));
        else if (LINES && at <= last) scaled_unit<DT, true, true>(v[i], s, y, plain, q + at);
        else if (LINES && at < n) scaled_unit<DT, true, false>(ld_unit<DT, false>(w, n - E), s, y, plain, q + (n - E));      // the tail
    }
}

__global__ void fill_u32_kernel(uint32_t* p, uint32_t v, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ---- dequant ----------------------------------------------------------------------------------
// Fast path: N % 8 == 0, block a power of two >= 8, aligned pointers.  The tensor is a flat run of 8-code
// units; each lane turns kDqUnroll units (8-byte loads, kDqThreads units apart) into bf16 (16-byte stores), so a
// wavefront writes 1 KiB of consecutive output per store instruction.  Row and column of a unit come from a multiply-high
// division by the row length (exact for every 32-bit unit index), not from an integer divide.
constexpr int kDqThreads = 256;
// (units per lane, alternating runs, one / two / four: 6.53-6.57 / 6.47-6.50 / 6.23-6.27 TB/s on 96 DeepSeek-V3 expert
// matrices, 6.21-6.23 / 6.17-6.22 / 6.11-6.14 on eight [16384, 7168] tensors)
#ifndef MQ_DQ_UNROLL
#define MQ_DQ_UNROLL 1
#endif
constexpr int kDqUnroll = MQ_DQ_UNROLL;
struct DequantJob {
    const uint8_t* x;
    const float* s;
    uint16_t* y;
    uint32_t units;          // M * N / 8
    uint32_t units_per_row;  // N / 8
    uint32_t magic, shift;   // floor(n / units_per_row) == (t + ((n - t) >> 1)) >> shift, t = mulhi(magic, n)
    int32_t block_shift;     // log2(block)
    int32_t tiles_n;
    int32_t N;               // columns (the form for any alignment)
};
struct DequantTable {
    int32_t n;
    int32_t max_blocks;
    int32_t chunk;           // blocks per XCD chunk (xcd_chunked_block); max_blocks is a multiple of 8 * chunk
    int32_t pad;
    DequantJob job[kMaxGroup];
};

__global__ __launch_bounds__(kDqThreads) void fp8_dequant_kernel(const DequantTable tab) {
    const DequantJob& job = tab.job[blockIdx.y];
    const int64_t base64 = xcd_chunked_block(tab.chunk) * (kDqThreads * kDqUnroll);
    if (base64 >= job.units) return;
    const uint32_t base = (uint32_t)base64;
    u32x2 in[kDqUnroll];
    float scale[kDqUnroll];
    // every load is issued before the first use: a lane past the end reads the workgroup's first unit again (always
    // there) and stores nothing
#pragma unroll
    for (int i = 0; i < kDqUnroll; i++) {
        const uint32_t unit = base + i * kDqThreads + threadIdx.x;
        const uint32_t uc = unit < job.units ? unit : base;
        // an ordinary (cached) load: with the non-temporal hint the 8-byte code loads of this kernel, which writes
        // twice what it reads, ran 2 % slower (6.36 against 6.50 TB/s on 36 tensors of [4096, 2560]); the 4- and
        // 16-byte code loads of the other unpacking kernels measured the other way round and keep the hint
        in[i] = *reinterpret_cast<const u32x2*>(job.x + (int64_t)uc * 8);
        const uint32_t th = __umulhi(job.magic, uc);
        const uint32_t r = (th + ((uc - th) >> 1)) >> job.shift;
        const uint32_t c = (uc - r * job.units_per_row) * 8u;
        scale[i] = job.s[(int64_t)(r >> job.block_shift) * job.tiles_n + (c >> job.block_shift)];
    }
    __builtin_amdgcn_sched_barrier(0);      // (and the scheduler keeps the first unit's arithmetic below the last load)
#pragma unroll
    for (int i = 0; i < kDqUnroll; i++) {
        const uint32_t unit = base + i * kDqThreads + threadIdx.x;
        if (unit >= job.units) continue;
        const float sc = scale[i];
        const uint32_t wd[2] = {in[i].x, in[i].y};
        uint32_t o[4];
        // a NaN code (0x7F / 0xFF) or a non-finite scale must give the canonical bf16 NaN 0x7FC0
        bool special = (f2u(sc) & 0x7F800000u) == 0x7F800000u;
#pragma unroll
        for (int k = 0; k < 2; k++) special |= (((wd[k] & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u) != 0u;
        if (!special) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const f32x2 a = hw_e4m3x2_decode<false>(wd[k]);
                const f32x2 b = hw_e4m3x2_decode<true>(wd[k]);
                o[2 * k] = hw_bf16x2(a.x * sc, a.y * sc);
                o[2 * k + 1] = hw_bf16x2(b.x * sc, b.y * sc);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                uint32_t h[4];
#pragma unroll
                for (int b = 0; b < 4; b++) h[b] = sw_bf16(sw_e4m3fn_decode((wd[k] >> (8 * b)) & 0xFFu) * sc);
                o[2 * k] = h[0] | (h[1] << 16);
                o[2 * k + 1] = h[2] | (h[3] << 16);
            }
        }
        st16(job.y + (int64_t)unit * 8, u32x4{o[0], o[1], o[2], o[3]});
    }
}

// Rows of any length >= 8 and any alignment: units_per_row = ceil(N / 8), and the last unit of a row is moved back to end with
// the row, decoding a few codes a second time.  Such a unit may reach into two tiles, hence two scales.  Bound by HBM and, a
// little, by the lines that neighbouring rows' units share.
// Eight [2049, 4099] matrices as one job list: 40 us with the submission, 5.0 TB/s, what [2048, 4096] ones take (200 us in the
// element-wise kernel, a launch each).
__global__ __launch_bounds__(kDqThreads) void fp8_dequant_any_kernel(const DequantTable tab) {
    const DequantJob& job = tab.job[blockIdx.y];
    const int64_t base64 = xcd_chunked_block(tab.chunk) * kDqThreads;
    if (base64 >= job.units) return;
    const uint32_t unit = (uint32_t)base64 + threadIdx.x;
    const uint32_t uc = unit < job.units ? unit : (uint32_t)base64;
    const uint32_t th = __umulhi(job.magic, uc);
    const uint32_t r = (th + ((uc - th) >> 1)) >> job.shift;
    const uint32_t at = (uc - r * job.units_per_row) * 8u, last = (uint32_t)job.N - 8u;
    const uint32_t c = at < last ? at : last;
    const int64_t off = (int64_t)r * job.N + c;
    const u32x2 in = ld8_at1(job.x + off);
    const float* __restrict__ s = job.s + (int64_t)(r >> job.block_shift) * job.tiles_n;
    const uint32_t tile = c >> job.block_shift;
    const float s0 = s[tile], s1 = s[(c + 7u) >> job.block_shift];
    const uint32_t split = ((tile + 1u) << job.block_shift) - c;      // elements of the first tile
    if (unit >= job.units) return;
    const uint32_t wd[2] = {in.x, in.y};
    bool special = (f2u(s0) & 0x7F800000u) == 0x7F800000u || (f2u(s1) & 0x7F800000u) == 0x7F800000u;
#pragma unroll
    for (int k = 0; k < 2; k++) special |= (((wd[k] & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u) != 0u;
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const float sc[4] = {4u * k < split ? s0 : s1, 4u * k + 1u < split ? s0 : s1, 4u * k + 2u < split ? s0 : s1, 4u * k + 3u < split ? s0 : s1};
        if (!special) {
            const f32x2 a = hw_e4m3x2_decode<false>(wd[k]), b = hw_e4m3x2_decode<true>(wd[k]);
            o[2 * k] = hw_bf16x2(a.x * sc[0], a.y * sc[1]);
            o[2 * k + 1] = hw_bf16x2(b.x * sc[2], b.y * sc[3]);
        } else {
            uint32_t h[4];
#pragma unroll
            for (int b = 0; b < 4; b++) h[b] = sw_bf16(sw_e4m3fn_decode((wd[k] >> (8 * b)) & 0xFFu) * sc[b]);
            o[2 * k] = h[0] | (h[1] << 16);
            o[2 * k + 1] = h[2] | (h[3] << 16);
        }
    }
    st16_at2(job.y + off, u32x4{o[0], o[1], o[2], o[3]});
}

__global__ __launch_bounds__(256) void fp8_dequant_generic_kernel(const uint8_t* __restrict__ x,
                                                                  const float* __restrict__ s,
                                                                  uint16_t* __restrict__ y, int64_t M, int64_t N,
                                                                  int block, int tiles_n) {
    const int64_t total = M * N;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t r = i / N, c = i - r * N;
        y[i] = (uint16_t)sw_bf16(sw_e4m3fn_decode(x[i]) * s[(r / block) * tiles_n + c / block]);
    }
}

}  // namespace mq

using namespace mq;

bool mq_fp8_tile_fast_ok(const void* w, int dtype, int64_t sxm, int64_t sxn, const void* q, int64_t M, int64_t K,
                         int bm, int bk) {
    // rows and columns below 2^24: a lane addresses its tile with 32-bit byte offsets from the tile's base
    return (dtype == MQ_BF16 || dtype == MQ_F16) && bm == kTile && bk == kTile && sxn == 1 && (K % 8) == 0 && (sxm % 8) == 0 &&
           ((uintptr_t)w % 16) == 0 && ((uintptr_t)q % 8) == 0 && M <= 0x7FFFFFFF && K < (1 << 24) && sxm > 0 &&
           sxm < (1 << 24);
}

// the same tiles without the 16-byte alignment, and of fp32 matrices (fp8_block128_any_kernel)
bool mq_fp8_tile_any_ok(const void* w, int dtype, int64_t sxm, int64_t sxn, int64_t M, int64_t K, int bm, int bk) {
    // 127 rows of 2^24 two-byte (2^23 four-byte) elements are what a 32-bit byte offset covers
    return dtype >= MQ_BF16 && dtype <= MQ_F32 && bm == kTile && bk == kTile && sxn == 1 && M <= 0x7FFFFFFF && K < (1 << 24) &&
           sxm > 0 && sxm < (dtype == MQ_F32 ? 1 << 23 : 1 << 24) && ((uintptr_t)w % (dtype == MQ_F32 ? 4 : 2)) == 0;
}

// fills the division constants of a descriptor whose w, q, scale, ldw, M, K and row blocks are set; returns its tile count
int64_t mq_fp8_tile_job_finish(TileJob& j) {
    const uint32_t tiles_k = (uint32_t)((j.K + kTile - 1) / kTile);
    uint32_t shift_k = 0, shift_b = 0;
    if (tiles_k > 1) tile_div_magic(tiles_k, j.magic_k, shift_k);
    if (j.tiles_per_block > 1) tile_div_magic((uint32_t)j.tiles_per_block, j.magic_b, shift_b);
    j.shifts = shift_k | (shift_b << 8);
    return (int64_t)((j.M + kTile - 1) / kTile) * tiles_k;
}

template <class Table>
static void tile_launch(int mode, bool f16, dim3 grid, hipStream_t st, const Table& tab) {
    const dim3 blk(kTileThreads);
    if (f16) {
        if (mode == 0) hipLaunchKernelGGL((fp8_block128_kernel<0, Table, 1>), grid, blk, 0, st, tab);
        else if (mode == 1) hipLaunchKernelGGL((fp8_block128_kernel<1, Table, 1>), grid, blk, 0, st, tab);
        else hipLaunchKernelGGL((fp8_block128_kernel<2, Table, 1>), grid, blk, 0, st, tab);
    } else {
        if (mode == 0) hipLaunchKernelGGL((fp8_block128_kernel<0, Table, 0>), grid, blk, 0, st, tab);
        else if (mode == 1) hipLaunchKernelGGL((fp8_block128_kernel<1, Table, 0>), grid, blk, 0, st, tab);
        else hipLaunchKernelGGL((fp8_block128_kernel<2, Table, 0>), grid, blk, 0, st, tab);
    }
}

// Dynamic LDS that leaves a compute unit (160 KB) two workgroups, or three.  Their registers are enough for four, which fill
// the memory system best unless a launch reads more lines at a time than it keeps open; see mq_fp8_tile_launch_group.
constexpr unsigned kTwoPerCu = 56u << 10, kThreePerCu = 44u << 10;
template <int DT, bool LINES>
static void tile_any_launch(int mode, dim3 grid, unsigned lds, bool aligned, hipStream_t st, const TileTable& tab) {
    const dim3 blk(kTileThreads);
    if (mode == 0) hipLaunchKernelGGL((fp8_block128_any_kernel<0, DT, LINES>), grid, blk, lds, st, tab, aligned);
    else if (mode == 1) hipLaunchKernelGGL((fp8_block128_any_kernel<1, DT, LINES>), grid, blk, lds, st, tab, aligned);
    else hipLaunchKernelGGL((fp8_block128_any_kernel<2, DT, LINES>), grid, blk, lds, st, tab, aligned);
}

// n finished descriptors in device memory, all of one 16-bit dtype; max_tiles: the largest tensor's tile count
int mq_fp8_tile_launch_table(int mode, int dtype, const TileJob* device_jobs, int n, int64_t max_tiles, hipStream_t st) {
    if (n == 0 || max_tiles == 0) return MQ_OK;
    const int64_t gx = xcd_grid(max_tiles);
    if (gx >= 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "too many tiles");
    tile_launch(mode, dtype == MQ_F16, dim3((unsigned)gx, (unsigned)n), st, TileRef{device_jobs});
    return mq_check_launch("fp8 block quant");
}

bool mq_fp8_tile_rows_share_lines(const void* w, int64_t ldw) { return (uintptr_t)w % 128 != 0 || ldw % 64 != 0; }
// The most tiles of a launch for which the any-alignment kernel, with its temporal loads and stores, ends sooner whatever the
// rows.  Inputs from HBM, us of a launch among others, fast kernel / that one (runs of one side differ by 0.05): block_fp8 32 tiles
// 5.02 / 4.59, 64 5.13 / 4.67, 80 5.16 / 4.73, 96 5.22 / 5.10, 112 5.28 / 5.28, 128 5.31 / 5.67, 256 5.84 / 6.88; blockwise cast 64
// 4.66 / 4.44, 80 4.71 / 4.49, 96 4.71 / 4.89, 128 4.83 / 5.50, 256 5.36 / 6.79.  (In a captured graph, where launches follow one another
// sooner, the fast one is ahead by 0.3 throughout: 64 tiles 4.47 / 4.74; alone 7.5 / 7.4.)
constexpr int64_t kAnyTiles = 80;
// Where most tiles are of tensors whose rows begin inside a 128-byte line, two tiles share the line at their border: the fast
// kernel's non-temporal loads fetch it, and its partial stores write it, once for each.  The temporal accesses of the other kernel
// pay as soon as every compute unit has several tiles.  Inputs from HBM, us, fast / any (runs of one side differ by 0.1): rows of
// 1032 elements 288 tiles 6.54 / 8.22, 576 9.95 / 10.8, 864 13.3 / 13.3, 1152 16.0 / 15.3, 1728 23.0 / 19.7, 6528 of 2056 97 / 60; of 8200 520
// 9.4 / 9.9, 1040 15.0 / 15.0, 1560 20.9 / 19.6, 4160 54 / 45, 16640 244 / 159.  Rows of whole half lines have one border in two
// on a line, and gain later: of 2592 1008 13.0 / 14.0, 1344 17.1 / 17.6 (blockwise cast 16.5 / 17.3), 1491 18.1 / 18.2, 2016 23.2 / 22.5,
// 4032 44.4 / 39.1; of 2080 1207 15.2 / 15.8, 1496 18.0 / 18.1, 1802 20.9 / 20.7.  (Inputs that are still in the memory-side cache gain at
// any number of tiles: 288 of 1032 5.9 / 5.2, 1152 13.9 / 11.4.)
constexpr int64_t kSharedTiles = 1152, kHalfLineTiles = 1536;

// tab.job[i] filled by the caller (w, q, scale, ldw, M, K, row blocks), all of one dtype; fills the division constants
// and `end`, launches.  `aligned`: every tensor passed mq_fp8_tile_fast_ok, otherwise mq_fp8_tile_any_ok.
// Aligned tensors take the any-alignment kernel as well in short launches and where tiles share lines (kAnyTiles, kSharedTiles); with rows
// of whole lines 2 x [8192, 8192] 64.9 / 74.4, 12 x [1545, 2624] the fast one 28.2.
int mq_fp8_tile_launch_group(int mode, int dtype, bool aligned, TileTable& tab, hipStream_t st) {
    int64_t tiles = 0, shared = 0, halves = 0;     // tiles, those of tensors whose rows share lines, and share them at half a line
    bool blocked = false;
    for (int i = 0; i < tab.n; i++) {
        TileJob& j = tab.job[i];
        const int64_t own = mq_fp8_tile_job_finish(j);
        tiles += own;
        if (tiles >= 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "too many tiles");
        tab.end[i] = (int32_t)tiles;
        blocked |= j.tiles_per_block != 0;
        if (!mq_fp8_tile_rows_share_lines(j.w, j.ldw)) continue;
        shared += own;
        if ((uintptr_t)j.w % 64 == 0 && j.ldw % 32 == 0) halves += own;
    }
    if (tiles == 0) return MQ_OK;
    seal_table(tab);
    const bool sharing = shared * 2 > tiles && tiles >= (halves * 2 > shared ? kHalfLineTiles : kSharedTiles);
    if (aligned && (blocked || (!sharing && tiles > kAnyTiles))) {      // (row blocks are the fast kernel's)
        tile_launch(mode, dtype == MQ_F16, dim3((unsigned)xcd_grid(tiles)), st, tab);
        return mq_check_launch("fp8 block quant");
    }
    bool lines = dtype == MQ_F32;      // whole 128-byte lines per tile row (every segment inside its row as well: K % 8 == 0)
    int64_t elems = 0, narrowest = INT64_MAX;
    bool slim = false;                 // few columns, the last few of them with tiles of their own
    for (int i = 0; i < tab.n; i++) {
        const TileJob& j = tab.job[i];
        lines &= ((uintptr_t)j.w % 128) == 0 && j.ldw % 32 == 0 && j.K % 8 == 0;
        elems += (int64_t)j.M * j.K;
        narrowest = j.K < narrowest ? j.K : narrowest;
        slim |= j.K < 4 * kTile && (j.K - 1) % kTile < 32;
    }
    // Neighbouring tiles of unaligned rows share lines, so the longer an XCD's runs of tiles are the better, as long as
    // every XCD has several: 24 [4097, 4099] bf16 tensors 4.48 / 4.73 / 4.77 / 4.93 TB/s with runs of 8 / 16 / 32 / 64.
    while (tab.chunk_shift < 6 && (tiles >> (tab.chunk_shift + 1)) >= 64) tab.chunk_shift++;
    const int64_t gx = xcd_grid_chunked(tiles, 1ll << tab.chunk_shift);
    if (gx >= 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "too many tiles");
    const dim3 grid((unsigned)gx);
    // The blockwise cast of long fp32 lists takes two or three workgroups per compute unit instead of four, whose tiles outgrow
    // an XCD's L2 before the neighbours have read the lines they share (us, four / three / two):
    //   unaligned rows of more than a tile, from 160 MiB on two: [4095, 8191] two 71 / 68 / 66, eight 286 / 259 / 240; [4097, 2051]
    //     eight 69 / 67 / 66, 32 of them 268 / 250 / 240; 268 MB of 195 columns 88 / 78 / 73, of 451 79 / 74 / 72, of 705 78 / 70 /
    //     67, 184 MB of 195 columns 60.2 / 53.7 / 51.1, of 1031 48.7 / 47.7 / 46.6 (but 268 MB of 250 columns 68 / 66 / 69, of 509
    //     66 / 65 / 68); three where they are slim: 268 MB of 129 columns 79 / 73 / 85, of 145 87 / 77 / 86, of 259 70 / 69 / 72;
    //   from 96 MiB on three: 134 MB of 145 columns 45 / 41 / 45, of 195 44 / 40 / 40, of 257 37.5 / 37.0 / 37.9, of 1163 37.5 / 36.2 /
    //     36.7, [4095, 8191] 34.7 / 34.2 / 35.9; up to two tiles wide from 48 MiB on: 67 MB of 145 columns 24.6 / 23.5 / 24.8, of 195
    //     24.1 / 23.2 / 22.6, but of 270 21.0 / 21.7 / 21.8, of 771 21.2 / 21.8 / 21.8;
    //   up to a tile wide always four: [65537, 67] 15 of them 59 / 60 / 69;
    //   whole lines, from 16384 tiles and 32768 columns on, two: [1024, 32768] four 120 / 119 / 119, eight 242 / 242 / 229; but
    //     [4096, 8192] eight 220 / 221 / 225, [16384, 128] 64 of them 116 / 118 / 119.
    unsigned lds = 0;
    if (mode == 1 && dtype == MQ_F32) {
        const int64_t mib = (elems * 4) >> 20;
        if (lines) lds = tiles >= 16384 && narrowest >= 32768 ? kTwoPerCu : 0u;
        else if (narrowest > kTile) lds = mib >= 160 && !slim ? kTwoPerCu : mib >= (narrowest <= 2 * kTile ? 48 : 96) ? kThreePerCu : 0u;
    }
    if (dtype == MQ_BF16) tile_any_launch<MQ_BF16, false>(mode, grid, lds, aligned, st, tab);
    else if (dtype == MQ_F16) tile_any_launch<MQ_F16, false>(mode, grid, lds, aligned, st, tab);
    else if (lines) tile_any_launch<MQ_F32, true>(mode, grid, lds, aligned, st, tab);
    else tile_any_launch<MQ_F32, false>(mode, grid, lds, aligned, st, tab);
    return mq_check_launch("fp8 block quant");
}

static int fp8_block_launch(int mode, const void* w, int dtype, int64_t sxm, int64_t sxn, void* q, float* scale,
                            int64_t M, int64_t K, int bm, int bk, hipStream_t stream) {
    if ((!w || !q || !scale) && M != 0 && K != 0) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (M < 0 || K < 0 || bm <= 0 || bk <= 0) return mq_fail(MQ_ERR_ARG, "bad shape or block size");
    if (dtype < MQ_BF16 || dtype > MQ_F32) return mq_fail(MQ_ERR_ARG, "unsupported dtype");
    if (M == 0 || K == 0) return MQ_OK;
    const bool aligned = mq_fp8_tile_fast_ok(w, dtype, sxm, sxn, q, M, K, bm, bk);
    if (aligned || mq_fp8_tile_any_ok(w, dtype, sxm, sxn, M, K, bm, bk)) {
        TileTable tab{};
        tab.n = 1;
        tab.job[0] = TileJob{w, q, scale, (int32_t)sxm, (int32_t)M, (int32_t)K, 0, 0, 0, 0, 0};
        return mq_fp8_tile_launch_group(mode, dtype, aligned, tab, stream);
    }
    const int64_t tiles_m = (M + bm - 1) / bm, tiles_k = (K + bk - 1) / bk;
    const int64_t tiles = tiles_m * tiles_k;
    if (tiles > 0x7FFFFFFF || tiles_k > 0x7FFFFFFF) return mq_fail(MQ_ERR_ARG, "too many tiles");
    if ((int64_t)bm * bk > (1 << 24)) return mq_fail(MQ_ERR_ARG, "block too large");
    dim3 grid((unsigned)tiles), blk(kGenThreads);
    if (mode == 0)
        hipLaunchKernelGGL(fp8_block_generic_kernel<0>, grid, blk, 0, stream, w, dtype, sxm, sxn, (uint8_t*)q, K, scale,
                           M, K, bm, bk, (int)tiles_k);
    else if (mode == 1)
        hipLaunchKernelGGL(fp8_block_generic_kernel<1>, grid, blk, 0, stream, w, dtype, sxm, sxn, (uint8_t*)q, K, scale,
                           M, K, bm, bk, (int)tiles_k);
    else
        hipLaunchKernelGGL(fp8_block_generic_kernel<2>, grid, blk, 0, stream, w, dtype, sxm, sxn, (uint8_t*)q, K, scale,
                           M, K, bm, bk, (int)tiles_k);
    return mq_check_launch("fp8 block quant");
}

extern "C" int mq_fp8_block_quant(const void* w, int dtype, int64_t ldw, void* q, float* scale, int64_t M, int64_t K,
                                  int block_m, int block_k, void* stream) {
    return fp8_block_launch(0, w, dtype, ldw, 1, q, scale, M, K, block_m, block_k, (hipStream_t)stream);
}

extern "C" int mq_fp8_blockwise_cast(const void* x, int dtype, int64_t stride_m, int64_t stride_n, void* y, float* s,
                                     int64_t M, int64_t N, int block_m, int block_n, void* stream) {
    return fp8_block_launch(1, x, dtype, stride_m, stride_n, y, s, M, N, block_m, block_n, (hipStream_t)stream);
}

extern "C" int mq_fp8_block_quant_pow2(const void* w, int dtype, int64_t ldw, void* q, float* scale, int64_t M, int64_t K,
                                       void* stream) {
    return fp8_block_launch(2, w, dtype, ldw, 1, q, scale, M, K, kTile, kTile, (hipStream_t)stream);
}

// How the rows of a tensor are held (fp8_channel_kernel): lanes per row and units per lane, and whether the rows are whole
// aligned units.  A wavefront per row while that leaves a lane no more than four units; sixteen units a lane are 64
// registers.  0: rows of less than a unit or of more than 4096, which take the element-wise kernels.
enum ChannelForm { kChannelNone = 0, kChannel64x4 = 1, kChannel64x8, kChannel256x4, kChannel256x8, kChannel256x16, kChannelLines = 8 };
int mq_fp8_channel_form(const void* w, int dtype, int64_t ldw, const void* q, int64_t M, int64_t K) {
    if (dtype < MQ_BF16 || dtype > MQ_F32 || M <= 0 || M > 0x7FFFFFFF) return kChannelNone;
    const int64_t E = dtype == MQ_F32 ? 4 : 8, units = (K + E - 1) / E;
    if (K < E || units > 256 * 16 || (uintptr_t)w % (dtype == MQ_F32 ? 4 : 2) != 0) return kChannelNone;
    const int64_t blocks = units <= 256 ? (M + 3) / 4 : M;
    if (blocks > 0x7FFFF000ll) return kChannelNone;          // (the grid is padded by up to 511 workgroups)
    const bool lines = K % E == 0 && ldw % E == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)q % E == 0;
    return (units <= 256 ? kChannel64x4 : units <= 1024 ? kChannel256x4 : units <= 2048 ? kChannel256x8 : kChannel256x16) | (lines ? kChannelLines : 0);
}
int64_t mq_fp8_channel_blocks(int form, int64_t M) { return (form & ~kChannelLines) <= kChannel64x8 ? (M + 3) / 4 : M; }
template <int DT, bool LINES>
static void channel_launch(int form, const ChannelTable& tab, hipStream_t st) {
    const dim3 grid((unsigned)tab.max_blocks, (unsigned)tab.n), blk(256);
    switch (form) {
        case kChannel64x4: hipLaunchKernelGGL((fp8_channel_kernel<64, DT, 4, LINES>), grid, blk, 0, st, tab); break;
        case kChannel64x8: hipLaunchKernelGGL((fp8_channel_kernel<64, DT, 8, LINES>), grid, blk, 0, st, tab); break;
        case kChannel256x4: hipLaunchKernelGGL((fp8_channel_kernel<256, DT, 4, LINES>), grid, blk, 0, st, tab); break;
        case kChannel256x8: hipLaunchKernelGGL((fp8_channel_kernel<256, DT, 8, LINES>), grid, blk, 0, st, tab); break;
        default: hipLaunchKernelGGL((fp8_channel_kernel<256, DT, 16, LINES>), grid, blk, 0, st, tab); break;
    }
}
// The form of a whole list (neither with kChannelLines), rows of at most `units`; inputs from HBM, us, runs of one side differ by
// 0.05 to 0.2.  Of 257 to 384 units half of the lanes of a 256-lane row and more have nothing in their second unit: a wavefront per
// row from 8192 rows on, which are one round of its workgroups (256 lanes / 64; 8192 rows of 2056 bf16 12.6 / 12.0, of 3072 15.4 / 14.9;
// 18540 of 2056 25.6 / 24.2, of 2560 27.6 / 25.1, of 2563 31.2 / 29.8, of 2880 29.6 / 28.8, of 3072 30.4 / 30.1, of 3200 31.6 / 31.3, but of 3584 33.4 /
// 34.9; of 1028 fp32 22.7 / 20.1; 6180 of 2880 12.0 / 12.6, 1545 of 2560 4.7 / 5.2).  A second round with hardly anything in it costs the wider rows
// of 16-bit elements what that gives: 8300 rows of 2880 14.9 / 15.3, of 3072 15.5 / 15.6, 8600 15.8 / 15.7 (of 2560 14.1 / 13.4; of 1440 fp32
// 12.8 / 12.5).
// Few rows leave a wavefront alone with its row: 256 lanes from 129 units on up to 2048 rows (device time, 64 lanes / 256; 64 rows
// of 1040 2.9 / 2.3, of 2048 3.6 / 2.6; 512 3.4 / 2.8 and 4.1 / 2.9, 1024 3.6 / 3.3 and 4.4 / 3.5, 2048 4.1 / 4.1 and 4.9 / 4.3, 2052 4.2 / 4.4 and 4.9 / 5.0).
static int channel_list_form(int form, int dtype, int64_t units, int64_t rows) {
    constexpr int64_t kRound = 8192, kThin = kRound + kRound / 32;
    const int64_t widest = dtype != MQ_F32 && rows > kRound && rows <= kThin ? 320 : 384;
    if (form == kChannel64x4 && units > 128 && rows <= 2048) return kChannel256x4;
    if (form == kChannel256x4 && units <= widest && rows >= kRound) return kChannel64x8;
    return form;
}
// n <= kMaxGroup tensors of one dtype and one form
int mq_fp8_channel_launch_group(int dtype, int form, const MqScaledArgs* a, int n, hipStream_t st) {
    ChannelTable tab{};
    tab.n = n;
    const bool lines = (form & kChannelLines) != 0;
    int64_t mx = 0, rows = 0, cols = 0;
    for (int i = 0; i < n; i++) {
        rows += a[i].M;
        cols = a[i].K > cols ? a[i].K : cols;
    }
    const int64_t E = dtype == MQ_F32 ? 4 : 8;
    form = channel_list_form(form & ~kChannelLines, dtype, (cols + E - 1) / E, rows);
    for (int i = 0; i < n; i++) {
        tab.job[i] = ChannelJob{a[i].w, (uint8_t*)a[i].q, a[i].scale, a[i].ldw, (int32_t)a[i].K, (int32_t)a[i].M, a[i].floor_v, 0};
        const int64_t blocks = mq_fp8_channel_blocks(form, a[i].M);
        mx = blocks > mx ? blocks : mx;
    }
    tab.chunk = (int32_t)flat_chunk(mx);
    tab.max_blocks = (int32_t)flat_padded(mx, tab.chunk);
    if (dtype == MQ_F32) lines ? channel_launch<MQ_F32, true>(form, tab, st) : channel_launch<MQ_F32, false>(form, tab, st);
    else if (dtype == MQ_F16) lines ? channel_launch<MQ_F16, true>(form, tab, st) : channel_launch<MQ_F16, false>(form, tab, st);
    else lines ? channel_launch<MQ_BF16, true>(form, tab, st) : channel_launch<MQ_BF16, false>(form, tab, st);
    return mq_check_launch("fp8 per-channel quant");
}

// one scale for a contiguous tensor: 1 from aligned addresses (only a tail of less than a unit is not), 2 from any others; 0:
// not for these kernels
int mq_fp8_scaled_form(const void* w, int dtype, int64_t ldw, const void* q, int64_t M, int64_t K) {
    if (dtype < MQ_BF16 || dtype > MQ_F32 || M <= 0 || M > 0x7FFFFFFF || (ldw != K && M != 1)) return 0;
    const int64_t E = dtype == MQ_F32 ? 4 : 8, n = M * K;
    if (n < E || (n + E - 1) / E >= (1ll << 38) || (uintptr_t)w % (dtype == MQ_F32 ? 4 : 2) != 0) return 0;
    return (uintptr_t)w % 16 == 0 && (uintptr_t)q % E == 0 ? 1 : 2;
}
template <int DT, bool LINES>
static void scaled_launch(const ScaledTable& tab, int keep, bool whole, hipStream_t st) {
    const dim3 amax((unsigned)tab.amax_blocks, (unsigned)tab.n), quant((unsigned)tab.max_blocks, (unsigned)tab.n);
    if (!LINES || keep == 4) hipLaunchKernelGGL((fp8_scaled_amax_kernel<DT, LINES, 4>), amax, dim3(kAmaxThreads), 0, st, tab);
    else if (keep == 2) hipLaunchKernelGGL((fp8_scaled_amax_kernel<DT, LINES, LINES ? 2 : 4>), amax, dim3(kAmaxThreads), 0, st, tab);
    else hipLaunchKernelGGL((fp8_scaled_amax_kernel<DT, LINES, LINES ? 0 : 4>), amax, dim3(kAmaxThreads), 0, st, tab);
    if (whole) hipLaunchKernelGGL((fp8_scaled_quant_kernel<DT, LINES, kScaledUnits>), quant, dim3(256), 0, st, tab);
    else hipLaunchKernelGGL((fp8_scaled_quant_kernel<DT, LINES, kScaledShortUnits>), quant, dim3(256), 0, st, tab);
}
// n <= kMaxGroup tensors of one dtype and one form, each with `words` words for its partial maxima (a power of two; fewer than
// kScaledWords: cleared first)
int mq_fp8_scaled_launch_group(int dtype, int form, const MqScaledArgs* a, int n, int words, hipStream_t st) {
    ScaledTable tab{};
    tab.n = n;
    const int64_t E = dtype == MQ_F32 ? 4 : 8;
    int64_t units = 0, all = 0;
    for (int i = 0; i < n; i++) {
        const int64_t numel = a[i].M * a[i].K, u = (numel + E - 1) / E;
        all += u;
        tab.job[i] = ScaledJob{a[i].w, (uint8_t*)a[i].q, a[i].scale, a[i].maxima, numel, a[i].floor_v, 0};
        units = u > units ? u : units;
    }
    const int64_t trips = (units + kAmaxThreads * kScaledLoads - 1) / (kAmaxThreads * kScaledLoads);
    if (words >= kScaledWords) {
        // what the chip holds (two workgroups per CU) from all tensors together, but not fewer than 64 for each, and no more
        // than it has trips
        int blocks = kScaledWords;
        while (blocks > 1 && ((blocks > 64 && blocks * n > 512) || blocks / 2 >= trips)) blocks /= 2;
        tab.words = tab.amax_blocks = blocks;
    } else {
        tab.words = words;
        tab.amax_blocks = (int32_t)(trips < kDirectBlocks ? trips : kDirectBlocks);
        for (int i = 0; i < n; i++) hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, a[i].maxima, 0u, words);
    }
    const bool whole = all >= kScaledLongList;
    const int64_t block = 256 * (whole ? kScaledUnits : kScaledShortUnits), blocks = (units + block - 1) / block, chunk = flat_chunk(blocks);
    if (flat_padded(blocks, chunk) >= 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "tensor too large");
    tab.chunk = (int32_t)chunk;
    tab.max_blocks = (int32_t)flat_padded(blocks, chunk);
    const bool lines = form == 1;
    const int keep = kept_quarters(all * 16);
    if (dtype == MQ_F32) lines ? scaled_launch<MQ_F32, true>(tab, keep, whole, st) : scaled_launch<MQ_F32, false>(tab, keep, whole, st);
    else if (dtype == MQ_F16) lines ? scaled_launch<MQ_F16, true>(tab, keep, whole, st) : scaled_launch<MQ_F16, false>(tab, keep, whole, st);
    else lines ? scaled_launch<MQ_BF16, true>(tab, keep, whole, st) : scaled_launch<MQ_BF16, false>(tab, keep, whole, st);
    return mq_check_launch("fp8 scaled quant");
}

static int fp8_scaled_quant(const void* w, int dtype, int64_t ldw, void* q, float* scale, void* amax_ws, int64_t M,
                            int64_t K, int per_channel, float floor_in_dtype, void* stream) {
    if ((!w || !q) && M != 0 && K != 0) return mq_fail(MQ_ERR_ARG, "null pointer");
    if ((!scale || !amax_ws) && (M != 0 || !per_channel)) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (dtype < MQ_BF16 || dtype > MQ_F32 || M < 0 || K < 0) return mq_fail(MQ_ERR_ARG, "bad argument");
    if (M == 0 || K == 0) return MQ_OK;
    if (M > 0x7FFFFFFF) return mq_fail(MQ_ERR_ARG, "too many rows");
    hipStream_t st = (hipStream_t)stream;
    const MqScaledArgs one{w, q, scale, (uint32_t*)amax_ws, ldw, M, K, floor_in_dtype};
    if (per_channel) {
        const int form = mq_fp8_channel_form(w, dtype, ldw, q, M, K);
        if (form) return mq_fp8_channel_launch_group(dtype, form, &one, 1, st);
    } else {
        // (the workspace holds a word per row, that of the static form 64 for a tensor)
        const int form = mq_fp8_scaled_form(w, dtype, ldw, q, M, K);
        if (form) return mq_fp8_scaled_launch_group(dtype, form, &one, 1, M >= kDirectWords ? kDirectWords : 1, st);
    }
    // rows of more than 4096 units or of less than one, strided tensors with one scale
    if (!per_channel) hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, (uint32_t*)amax_ws, 0u, 1);
    hipLaunchKernelGGL(fp8_row_amax_kernel, dim3((unsigned)M), dim3(256), 0, st, w, dtype, ldw, K,
                       (uint32_t*)amax_ws, per_channel);
    hipLaunchKernelGGL(fp8_row_quant_kernel, dim3((unsigned)M), dim3(256), 0, st, w, dtype, ldw, K,
                       (const uint32_t*)amax_ws, floor_in_dtype, per_channel, (uint8_t*)q, scale);
    return mq_check_launch("fp8 scaled quant");
}

extern "C" int mq_fp8_scaled_quant(const void* w, int dtype, int64_t ldw, void* q, float* scale, void* amax_ws,
                                   int64_t M, int64_t K, int per_channel, float floor_in_dtype, void* stream) {
    return fp8_scaled_quant(w, dtype, ldw, q, scale, amax_ws, M, K, per_channel, floor_in_dtype, stream);
}

// ---- the same quantizer for callers that cannot allocate ------------------------------------------------------
// The amax workspace (one word per tensor, or one per row with per-channel scales) lives in a file-scope device
// array instead of coming from the caller.  `scratch` names the array in host code only as a symbol: its address in
// device memory differs per GPU and is looked up once per device with hipGetSymbolAddress; kernels and fills get
// that address, never the symbol.
static __device__ __align__(256) uint32_t scratch[MQ_FP8_STATIC_MAX_ROWS];
static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_lock;
static uint32_t* g_scratch_ptr[kMaxDevices];      // device address of `scratch` on each GPU, 0 until first use there
static int64_t g_scratch_next[kMaxDevices];       // first word of the array that the next call on that GPU takes

// `words` words of `scratch` on the current device for one call, or null with the error text set.  Calls take
// consecutive pieces of the array (whole 256-byte lines), starting over at its beginning when a piece no longer fits:
// two calls that are in flight together -- on two streams, from two host threads -- only share words when the pieces
// handed out between them add up to more than the array.
static uint32_t* scratch_on_current_device(int64_t words) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        mq_fail(MQ_ERR_HIP, "mq_fp8_scaled_quant_static: no current device (or a device index above 63)");
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            mq_fail(MQ_ERR_HIP, "mq_fp8_scaled_quant_static: hipGetSymbolAddress failed for the amax workspace");
            return nullptr;
        }
        g_scratch_ptr[dev] = (uint32_t*)p;
    }
    const int64_t piece = (words + 63) / 64 * 64;
    if (g_scratch_next[dev] + piece > MQ_FP8_STATIC_MAX_ROWS) g_scratch_next[dev] = 0;
    uint32_t* at = g_scratch_ptr[dev] + g_scratch_next[dev];
    g_scratch_next[dev] += piece;
    return at;
}

extern "C" int mq_fp8_scaled_quant_static(const void* w, int dtype, int64_t ldw, void* q, float* scale, int64_t M,
                                          int64_t K, int per_channel, float floor_in_dtype, void* stream) {
    if (per_channel && M > MQ_FP8_STATIC_MAX_ROWS)
        return mq_fail(MQ_ERR_ARG, "mq_fp8_scaled_quant_static: per-channel scales take at most MQ_FP8_STATIC_MAX_ROWS "
                                   "(262144) rows; use mq_fp8_scaled_quant with a workspace of its own");
    uint32_t* ws = scratch_on_current_device(per_channel && M > 0 ? M : 1);
    if (!ws) return MQ_ERR_HIP;
    return fp8_scaled_quant(w, dtype, ldw, q, scale, ws, M, K, per_channel, floor_in_dtype, stream);
}

bool mq_fp8_dequant_fast_ok(const void* x, const void* y, int64_t M, int64_t N, int block) {
    const bool pow2 = block >= 8 && (block & (block - 1)) == 0;
    return (N % 8) == 0 && N >= 16 && pow2 && ((uintptr_t)x % 8) == 0 && ((uintptr_t)y % 16) == 0 &&
           M * (N / 8) < 0xFFFFFFF0ll;
}

// the same without the alignment: rows of nine codes and more (two units)
bool mq_fp8_dequant_any_ok(const void* y, int64_t M, int64_t N, int block) {
    const bool pow2 = block >= 8 && (block & (block - 1)) == 0;
    return N >= 9 && N < (1ll << 31) && pow2 && ((uintptr_t)y % 2) == 0 && M * ((N + 7) / 8) < 0xFFFFFFF0ll;
}

// `aligned`: every tensor passed mq_fp8_dequant_fast_ok, otherwise mq_fp8_dequant_any_ok
int mq_fp8_dequant_launch_group(const MqDequantArgs* a, int n, bool aligned, hipStream_t st) {
    DequantTable tab{};
    tab.n = n;
    int64_t mx = 0;
    for (int i = 0; i < n; i++) {
        DequantJob& j = tab.job[i];
        j.x = (const uint8_t*)a[i].x;
        j.s = a[i].s;
        j.y = (uint16_t*)a[i].y;
        const uint32_t d = (uint32_t)((a[i].N + 7) / 8);   // >= 2
        j.units = (uint32_t)(a[i].M * d);
        j.N = (int32_t)a[i].N;
        j.units_per_row = d;
        uint32_t l = 0;
        while ((1ull << l) < d) l++;                 // ceil(log2 d) >= 1
        j.magic = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
        j.shift = l - 1;
        int bs = 0;
        while ((1 << bs) < a[i].block) bs++;
        j.block_shift = bs;
        j.tiles_n = (int32_t)((a[i].N + a[i].block - 1) / a[i].block);
        const int per_block = aligned ? kDqThreads * kDqUnroll : kDqThreads;
        const int64_t b = ((int64_t)j.units + per_block - 1) / per_block;
        if (b > mx) mx = b;
    }
    if (mx == 0) return MQ_OK;
    const int64_t chunk = flat_chunk(mx);
    mx = flat_padded(mx, chunk);
    tab.chunk = (int32_t)chunk;
    tab.max_blocks = (int32_t)mx;
    if (aligned) hipLaunchKernelGGL(fp8_dequant_kernel, dim3((unsigned)mx, (unsigned)n), dim3(kDqThreads), 0, st, tab);
    else hipLaunchKernelGGL(fp8_dequant_any_kernel, dim3((unsigned)mx, (unsigned)n), dim3(kDqThreads), 0, st, tab);
    return mq_check_launch("fp8 block dequant");
}

// One lane per output word.  ROW_MAJOR = false: DeepGEMM's layout [batch][ceil(kb/4)][align(mn,4)], consecutive lanes
// take consecutive rows; true: the same words as a contiguous [batch][mn][ceil(kb/4)] array (what `.contiguous()` makes
// of the transposed view, e.g. inside a flattened transport payload).
template <bool ROW_MAJOR>
__global__ __launch_bounds__(256) void ue8m0_pack_scales_kernel(const float* __restrict__ sf, uint32_t* __restrict__ out,
                                                                int64_t total, int64_t mn, int64_t amn, int64_t kb,
                                                                int64_t kw, int64_t tile_rows) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        int64_t r, j, b;
        if (ROW_MAJOR) {
            j = i % kw;
            r = (i / kw) % mn;
            b = i / (kw * mn);
        } else {
            r = i % amn;
            j = (i / amn) % kw;
            b = i / (amn * kw);
        }
        uint32_t word = 0;
        if (r < mn) {
            const float* row = sf + (b * tile_rows + r / 128) * kb;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * j + e < kb) word |= ((__float_as_uint(row[4 * j + e]) >> 23) & 0xFFu) << (8 * e);
        }
        out[i] = word;
    }
}

extern "C" int mq_ue8m0_pack_scales(const float* sf, int32_t* out, int64_t batch, int64_t mn, int64_t kb,
                                    int64_t tile_rows, int row_major, void* stream) {
    if ((!sf || !out) && batch != 0 && mn != 0 && kb != 0) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (batch < 0 || mn < 0 || kb < 0 || tile_rows < (mn + 127) / 128) return mq_fail(MQ_ERR_ARG, "bad shape");
    const int64_t amn = (mn + 3) / 4 * 4, kw = (kb + 3) / 4, total = batch * kw * (row_major ? mn : amn);
    if (total == 0) return MQ_OK;
    int64_t blocks = (total + 255) / 256;
    if (blocks > mq_grid_cap()) blocks = mq_grid_cap();
    const dim3 grid((unsigned)blocks), blk(256);
    if (row_major)
        hipLaunchKernelGGL(ue8m0_pack_scales_kernel<true>, grid, blk, 0, (hipStream_t)stream, sf, (uint32_t*)out, total, mn, amn, kb, kw, tile_rows);
    else
        hipLaunchKernelGGL(ue8m0_pack_scales_kernel<false>, grid, blk, 0, (hipStream_t)stream, sf, (uint32_t*)out, total, mn, amn, kb, kw, tile_rows);
    return mq_check_launch("ue8m0 scale pack");
}

extern "C" int mq_fp8_block_dequant(const void* x, const float* s, void* y, int64_t M, int64_t N, int block,
                                    void* stream) {
    if ((!x || !s || !y) && M != 0 && N != 0) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (M < 0 || N < 0 || block <= 0) return mq_fail(MQ_ERR_ARG, "bad shape or block size");
    if (M == 0 || N == 0) return MQ_OK;
    const int64_t tiles_n = (N + block - 1) / block;
    if (tiles_n > 0x7FFFFFFF) return mq_fail(MQ_ERR_ARG, "too many tiles");
    hipStream_t st = (hipStream_t)stream;
    const bool aligned = mq_fp8_dequant_fast_ok(x, y, M, N, block);
    if (aligned || mq_fp8_dequant_any_ok(y, M, N, block)) {
        MqDequantArgs a{x, s, y, M, N, block};
        return mq_fp8_dequant_launch_group(&a, 1, aligned, st);
    }
    int64_t blocks = (M * N + 255) / 256;
    if (blocks > mq_grid_cap()) blocks = mq_grid_cap();
    hipLaunchKernelGGL(fp8_dequant_generic_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (const uint8_t*)x, s,
                       (uint16_t*)y, M, N, block, (int)tiles_n);
    return mq_check_launch("fp8 block dequant");
}
